// What gemm.hip and gemm_flex.hip share: a 16-bit product and the way it is carried out.
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>
#include <cstdint>

#include "kernels/gemm_flex_plan.h"

namespace paras {
namespace flex {

struct Problem {
    const std::uint16_t* a;
    const std::uint16_t* b;
    const std::uint16_t* add;
    std::uint16_t* c;
    long M, N, K;
    long lda, ldb, ldc, ld_add;
    long sa, sb, sc, sadd, batch;
    float alpha, beta;
    bool a_rows, b_rows;        // the operand is contiguous along its rows, not along the contraction (a_rows only with b_rows)
    bool bf16;
};
bool takes(const Problem& q);                       // sizes and alignments the kernel can read
Plan plan(const Problem& q, bool may_split);
inline size_t workspace(const Problem& q, const Plan& p) {
    return p.splits > 1 ? static_cast<size_t>(p.splits) * q.batch * q.M * q.N * sizeof(float) : 0;
}
int launch(const Problem& q, const Plan& plan, void* workspace, hipStream_t s);

}  // namespace flex
}  // namespace paras
