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
template <typename T, int V>
__global__ __launch_bounds__(256) void gemm_flex_finish_kernel(const Params p) {
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

// Per tile shape: rows, columns, workgroups a CU holds at once, and in us the time of one tile of 64
// contraction steps on a CU that is full (`step`) and at least, on a CU with a single workgroup (`lat`: a
// barrier and the way from L2).
struct Tile { int m, n, per_cu; double step, lat; };
constexpr Tile kTiles[] = {{256, 256, 1, 1.39, 0.66}, {192, 256, 1, 1.09, 0.26}, {128, 256, 1, 0.93, 0.17}, {128, 128, 2, 0.86, 0.58},
                           {64, 128, 3, 0.94, 0.39}, {64, 64, 4, 0.84, 0.20}, {32, 128, 3, 0.84, 0.26}};
constexpr int kTileCount = 7;
constexpr int kCus = 256;

}  // namespace

bool takes(const Problem& q) {
    auto aligned = [](const void* p, long ld, long stride) {
        return (reinterpret_cast<uintptr_t>(p) & 15) == 0 && ld % 8 == 0 && stride % 8 == 0 && ld <= kMaxLd;
    };
    if (q.a_rows && !q.b_rows) return false;
    if (!aligned(q.a, q.lda, q.sa) || !aligned(q.b, q.ldb, q.sb)) return false;
    // (a chunk of 8 contraction steps is in or out as a whole)
    if (q.K <= 0 || q.K >= (1L << 30) || (!(q.a_rows && q.b_rows) && q.K % 8 != 0)) return false;
    const long tiles = ((q.M + 31) / 32) * ((q.N + 63) / 64);
    return q.batch <= 65535 && tiles * q.batch < (1L << 25);
}

// The least estimated time over tile shapes and numbers of parts.  Rounds of workgroups times the time of
// their share of the contraction and of their stores, plus the second kernel where the contraction is in
// parts.  The constants were fitted to 6900 timings (1 to 16384 rows, 512 to 14336 columns, contractions of 8
// to 14336, all three layouts): over those the choice is 1.9 % slower than the best one in the mean and 10 % at the
// 95th percentile.  What the rule trades: a 256 x 256 tile reads half as much per flop as a 128 x 128 one
// (16384 x 4096 x 4096 395 against 459 us), but with 192 of them for 256 CUs a quarter of the chip idles
// (3000 x 4096 x 4096 98 us, with 256 tiles of 192 x 256 83 us); with few tiles the contraction is cut up
// instead (8 x 14336 x 4096 41 us whole, 25 us in four parts).
Plan plan(const Problem& q, bool may_split) {
    Plan best;
    double best_us = 1e30;
    const long k_tiles = (q.K + kBK - 1) / kBK;
    const double mn = static_cast<double>(q.M) * q.N * q.batch;
    for (int t = 0; t < kTileCount; ++t) {
        const Tile& tl = kTiles[t];
        if (t < 3 && q.K <= 512) continue;           // mostly stores: small tiles overlap them with other tiles' work
        const long mt = (q.M + tl.m - 1) / tl.m, nt = (q.N + tl.n - 1) / tl.n, tiles = mt * nt * q.batch;
        // the share of its panels that a workgroup is the first to ask for comes from further away than L2
        const double first = (static_cast<double>(tl.n) / mt + static_cast<double>(tl.m) / nt) / (tl.m + tl.n);
        const double lat = tl.lat + 0.54 * first, stores = tl.m * tl.n / 65536.0 * 4.7;
        for (int s = 1; s <= (may_split ? 32 : 1); s = s < 4 ? s + 1 : s + s / 2) {
            if (s > 1 && (s * 2 > k_tiles || tiles * s > 1600)) break;
            const long per = (k_tiles + s - 1) / s, parts = (k_tiles + per - 1) / per, paired = per + (per & 1);
            const long wgs = tiles * parts, slots = static_cast<long>(kCus) * tl.per_cu, full = wgs / slots;
            const long rest = (wgs - full * slots + kCus - 1) / kCus;
            auto round = [&](double n) {
                const double c = tl.step * n / tl.per_cu;
                return paired * (c > lat ? c : lat) + 2.3 + stores * n;
            };
            double us = full * round(tl.per_cu) + (rest > 0 ? round(static_cast<double>(rest)) : 0.0);
            if (parts > 1) us += 3.0 + mn * (8.0 * parts + 2.0) / 6.9e6;
            if (us < best_us) {
                best_us = us;
                best.tile = t;
                best.splits = static_cast<int>(parts);
                best.k_per_split = per * kBK;
            }
        }
    }
    return best;
}

int launch(const Problem& q, const Plan& plan, void* workspace, hipStream_t s) {
    Params p{};
    p.a = q.a; p.b = q.b; p.add = q.add; p.c = q.c;
    p.M = q.M; p.N = q.N; p.K = q.K;
    p.lda = q.lda; p.ldb = q.ldb; p.ldc = q.ldc; p.ld_add = q.ld_add;
    p.sa = q.sa; p.sb = q.sb; p.sc = q.sc; p.sadd = q.sadd;
    p.alpha = q.alpha; p.beta = q.beta;
    const Tile t = kTiles[plan.tile];
    p.m_tiles = static_cast<int>((q.M + t.m - 1) / t.m);
    p.n_tiles = static_cast<int>((q.N + t.n - 1) / t.n);
    p.splits = plan.splits;
    p.k_per_split = plan.k_per_split;
    p.partial = static_cast<float*>(workspace);
    const long wgs = static_cast<long>(p.m_tiles) * p.n_tiles * plan.splits * q.batch;
    const unsigned grid = static_cast<unsigned>(wgs);
    if (q.a_rows)      launch_rr(q.bf16, plan.tile, p, grid, s);
    else if (q.b_rows) launch_kr(q.bf16, plan.tile, p, grid, s);
    else               launch_kk(q.bf16, plan.tile, p, grid, s);
    PARAS_HIP_TRY(hipGetLastError());
    if (plan.splits > 1) {
        const bool vec = q.N % 4 == 0 && q.ldc % 4 == 0 && q.sc % 4 == 0 && (reinterpret_cast<uintptr_t>(q.c) & 7) == 0;
        const long n = (q.M * q.N + (vec ? 1023 : 255)) / (vec ? 1024 : 256);
        const dim3 g(static_cast<unsigned>(n), static_cast<unsigned>(q.batch));
        if (q.bf16) { if (vec) hipLaunchKernelGGL((gemm_flex_finish_kernel<bf16_t, 4>), g, dim3(256), 0, s, p);
                      else     hipLaunchKernelGGL((gemm_flex_finish_kernel<bf16_t, 1>), g, dim3(256), 0, s, p); }
        else        { if (vec) hipLaunchKernelGGL((gemm_flex_finish_kernel<f16_t, 4>), g, dim3(256), 0, s, p);
                      else     hipLaunchKernelGGL((gemm_flex_finish_kernel<f16_t, 1>), g, dim3(256), 0, s, p); }
        PARAS_HIP_TRY(hipGetLastError());
    }
    return PARAS_OK;
}

}  // namespace flex
}  // namespace paras
