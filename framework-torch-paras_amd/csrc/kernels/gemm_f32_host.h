// What gemm.hip and gemm_f32.hip share: an fp32 product and the way it is carried out.
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>

namespace paras {
namespace f32 {

struct Problem {
    const float* a;
    const float* b;
    const float* add;
    float* c;
    long M, N, K;
    long lda, ldb, ldc, ld_add;
    long sa, sb, sc, sadd, batch;
    float alpha, beta;
    bool a_rows, b_rows;        // the operand is contiguous along its rows, not along the contraction (a_rows only with b_rows)
    int  causal_kind;           // see Params in gemm_f32.hip
    long causal_first;
};
struct Plan {
    int  tile = 0, splits = 1;
    long k_per_split = 0;
};

bool takes(const Problem& q);
Plan plan(const Problem& q, bool may_split);
size_t workspace(const Problem& q, const Plan& pl);
int launch(const Problem& q, const Plan& pl, void* ws, hipStream_t s);

}  // namespace f32
}  // namespace paras
