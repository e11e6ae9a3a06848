// Host side of the 16-bit product with operands either way round (kernel: gemm_flex_kernel.h): the
// choice of tile and of the number of parts the contraction is split into, the kernel that adds the
// parts, and the launch.
#include <hip/hip_runtime.h>

#include "core/device_context.h"
#include "core/status.h"
#include "kernels/gemm_flex_host.h"
#include "kernels/gemm_flex_kernel.h"
#include "paras_hip.h"

namespace paras {
namespace flex {
namespace {

// Adds the parts in order and applies the epilogue; V columns per thread.
struct FinishParams {
    const float* partial;
    const std::uint16_t* add;
    std::uint16_t* c;
    long M, N, sc, sadd, ldc, ld_add;
    int  splits;
    float alpha, beta;
};
template <typename T, int V>
__global__ __launch_bounds__(256) void gemm_flex_finish_kernel(const FinishParams p) {
    using El = Elem<T>;
    typedef float vec __attribute__((ext_vector_type(V)));
    const long mn = p.M * p.N, i = (static_cast<long>(blockIdx.x) * 256 + threadIdx.x) * V;
    if (i >= mn) return;
    const long batch = blockIdx.y;
    const float* src = p.partial + batch * p.splits * mn + i;
    vec t = *reinterpret_cast<const vec*>(src);
    int sp = 1;
    for (; sp + 3 < p.splits; sp += 4) {          // four parts in flight, added in order
        vec v[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) v[u] = *reinterpret_cast<const vec*>(src + (sp + u) * mn);
#pragma unroll
        for (int u = 0; u < 4; ++u) t += v[u];
    }
    for (; sp < p.splits; ++sp) t += *reinterpret_cast<const vec*>(src + sp * mn);
    const unsigned row = static_cast<unsigned>(i / p.N), col = static_cast<unsigned>(i - static_cast<long>(row) * p.N);
    std::uint16_t o[V];
#pragma unroll
    for (int r = 0; r < V; ++r) {
        float v = p.alpha * t[r];
        if (p.add) v = fmaf(p.beta, El::to_f32((p.add + batch * p.sadd)[row * p.ld_add + col + r]), v);
        o[r] = El::from_f32(v);
    }
    std::uint16_t* dst = p.c + batch * p.sc + static_cast<long>(row) * p.ldc + col;
    if constexpr (V == 4) {
        u32x2 w2;
        w2[0] = o[0] | (static_cast<std::uint32_t>(o[1]) << 16);
        w2[1] = o[2] | (static_cast<std::uint32_t>(o[3]) << 16);
        *reinterpret_cast<u32x2*>(dst) = w2;
    } else {
        *dst = o[0];
    }
}

static_assert(kTiles[kTile128x128].m == 128 && kTiles[kTile128x128].n == 128 && kTiles[kTile128x128].stages == 2, "the tile that paras_gemm_nt_ws splits");
static_assert(kPlanStep == kBK, "gemm_flex_plan.h");

}  // namespace

bool takes(const Problem& q) {
    auto aligned = [](const void* p, long ld, long stride) {
        return (reinterpret_cast<uintptr_t>(p) & 15) == 0 && ld % 8 == 0 && stride % 8 == 0 && ld <= kMaxLd;
    };
    if (q.a_rows && !q.b_rows) return false;
    if (!aligned(q.a, q.lda, q.sa) || !aligned(q.b, q.ldb, q.sb)) return false;
    // (a chunk of 8 contraction steps is in or out as a whole)
    if (q.K <= 0 || q.K >= (1L << 30) || (!(q.a_rows && q.b_rows) && q.K % 8 != 0)) return false;
    const long tiles = ((q.M + 31) / 32) * ((q.N + 63) / 64);          // (below 2^25: M and N fit as well)
    return q.batch <= 65535 && tiles * q.batch < (1L << 25);
}

Plan plan(const Problem& q, bool may_split) { return plan_of(q.M, q.N, q.K, q.batch, q.a_rows, q.b_rows, may_split); }

int launch(const Problem& q, const Plan& plan, void* workspace, hipStream_t s) {
    auto narrow = [](long v) { return static_cast<int>(v); };       // (takes())
    Params p{};
    p.a = q.a; p.b = q.b; p.add = q.add;
    p.out = plan.splits > 1 ? workspace : q.c;
    p.M = narrow(q.M); p.N = narrow(q.N); p.K = narrow(q.K);
    p.lda = static_cast<std::uint32_t>(q.lda); p.ldb = narrow(q.ldb); p.ldc = q.ldc; p.ld_add = q.ld_add;
    p.sa = q.sa; p.sb = q.sb; p.sc = q.sc; p.sadd = q.sadd;
    p.alpha = q.alpha; p.beta = q.beta;
    const Tile t = kTiles[plan.tile];
    p.splits = static_cast<std::uint32_t>(plan.splits);
    p.k_per_split = narrow(plan.k_per_split);
    const long wgs = (q.M + t.m - 1) / t.m * ((q.N + t.n - 1) / t.n) * plan.splits * q.batch;
    const unsigned grid = static_cast<unsigned>(wgs);
    if (q.a_rows)      launch_rr(q.bf16, plan.tile, p, grid, s);
    else if (q.b_rows) launch_kr(q.bf16, plan.tile, p, grid, s);
    else               launch_kk(q.bf16, plan.tile, p, grid, s);
    PARAS_HIP_TRY(hipGetLastError());
    if (plan.splits > 1) {
        const bool vec = q.N % 4 == 0 && q.ldc % 4 == 0 && q.sc % 4 == 0 && (reinterpret_cast<uintptr_t>(q.c) & 7) == 0;
        const long n = (q.M * q.N + (vec ? 1023 : 255)) / (vec ? 1024 : 256);
        const FinishParams f{static_cast<const float*>(workspace), q.add, q.c, q.M, q.N, q.sc, q.sadd, q.ldc, q.ld_add, plan.splits, q.alpha, q.beta};
        const dim3 g(static_cast<unsigned>(n), static_cast<unsigned>(q.batch));
        if (q.bf16) { if (vec) hipLaunchKernelGGL((gemm_flex_finish_kernel<bf16_t, 4>), g, dim3(256), 0, s, f);
                      else     hipLaunchKernelGGL((gemm_flex_finish_kernel<bf16_t, 1>), g, dim3(256), 0, s, f); }
        else        { if (vec) hipLaunchKernelGGL((gemm_flex_finish_kernel<f16_t, 4>), g, dim3(256), 0, s, f);
                      else     hipLaunchKernelGGL((gemm_flex_finish_kernel<f16_t, 1>), g, dim3(256), 0, s, f); }
        PARAS_HIP_TRY(hipGetLastError());
    }
    return PARAS_OK;
}

}  // namespace flex
}  // namespace paras
