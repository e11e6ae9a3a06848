// The kernel of the 16-bit products in gemm_flex.hip (mainloop: gemm_flex.h), apart so that the
// translation units that instantiate it compile side by side.
#pragma once

#include "kernels/gemm_flex.h"

namespace paras {
namespace flex {

// (112 bytes: a launch whose arguments take more than that costs the host 0.7 us more, 3.4 for 2.7.)
struct Params {
    const std::uint16_t* a;
    const std::uint16_t* b;
    const std::uint16_t* add;   // may be null
    void* out;                  // splits == 1: the result; otherwise fp32 [batch][split][M][N]
    long sa, sb, sc, sadd;      // batch strides (elements)
    long ldc, ld_add;
    int  M, N, K;
    int  ldb;
    std::uint32_t lda : 23;     // (up to kMaxLd, as ldb)
    std::uint32_t splits : 9;   // parts of the contraction, one workgroup each per tile (up to 384)
    int  k_per_split;           // contraction steps per part (a multiple of 64)
    float alpha, beta;
};
static_assert(kMaxLd < (1L << 23), "Params::lda");
static_assert(sizeof(Params) <= 112, "see above");

// Workgroup w runs on XCD w % 8, each with an L2 of its own: every XCD takes a contiguous run of the
// work list, and the list walks the tiles in bands of kBand row tiles, so that the 32 workgroups an XCD
// runs together are about 4 row panels x 8 column panels.  Parts of the contraction and batch entries
// are the outer dimensions of the list.
constexpr int kXcds = 8, kBand = 4;
// (The quotients come from vector arithmetic: each is moved to a scalar register, or everything that depends on
// them -- buffer descriptors, loop bounds -- would be held per lane.)
struct Work { int batch, split, mt, nt; };
__device__ __forceinline__ unsigned scalar(unsigned v) { return static_cast<unsigned>(__builtin_amdgcn_readfirstlane(static_cast<int>(v))); }
__device__ __forceinline__ Work work_of(unsigned m_tiles, unsigned n_tiles, unsigned splits, unsigned wg, unsigned total) {
    const unsigned q = total / kXcds, r = total % kXcds, x = wg % kXcds;
    const unsigned lin = x * q + (x < r ? x : r) + wg / kXcds;
    const unsigned tiles = m_tiles * n_tiles;
    const unsigned outer = scalar(lin / tiles);
    const unsigned t = lin - outer * tiles;
    const unsigned per_band = kBand * n_tiles;
    const unsigned band = scalar(t / per_band), in = t - band * per_band;
    const unsigned left = m_tiles - band * kBand, rows = left < kBand ? left : kBand;
    const unsigned nt = scalar(in / rows), batch = scalar(outer / splits);
    return {static_cast<int>(batch), static_cast<int>(outer - batch * splits),
            static_cast<int>(band * kBand + (in - nt * rows)), static_cast<int>(nt)};
}

template <typename T, int MI, int NJ, int ST, bool AR, bool BR>
__global__ __launch_bounds__(kThreads, (MI * NJ >= 32 || ST * (MI + NJ) > 20 ? 1 : 2)) void gemm_flex_kernel(const Params p) {
    using El = Elem<T>;
    using OA = Operand<MI, AR>;
    using OB = Operand<NJ, BR>;
    __shared__ __attribute__((aligned(1024))) std::uint16_t a0[OA::kElems];
    __shared__ __attribute__((aligned(1024))) std::uint16_t a1[OA::kElems];
    __shared__ __attribute__((aligned(1024))) std::uint16_t a2[OA::kElems];     // (stages past ST are never named, and take no memory)
    __shared__ __attribute__((aligned(1024))) std::uint16_t a3[OA::kElems];
    __shared__ __attribute__((aligned(1024))) std::uint16_t b0[OB::kElems];
    __shared__ __attribute__((aligned(1024))) std::uint16_t b1[OB::kElems];
    __shared__ __attribute__((aligned(1024))) std::uint16_t b2[OB::kElems];
    __shared__ __attribute__((aligned(1024))) std::uint16_t b3[OB::kElems];
    asm volatile("" ::"s"(p.ldc), "s"(p.ld_add));          // (fetched with the rest: left to itself the compiler does it in front of the stores)
    const Work w = work_of((static_cast<unsigned>(p.M) + 32 * MI - 1) / (32 * MI), (static_cast<unsigned>(p.N) + 32 * NJ - 1) / (32 * NJ),
                           p.splits, blockIdx.x, gridDim.x);
    const long row0 = static_cast<long>(w.mt) * (32 * MI), col0 = static_cast<long>(w.nt) * (32 * NJ);
    const long k_first = static_cast<long>(w.split) * p.k_per_split;
    const long k_count = p.K - k_first < p.k_per_split ? p.K - k_first : p.k_per_split;
    const int wave = wave_id();
    OA oa;
    OB ob;
    oa.init(p.a + w.batch * p.sa, p.lda, p.M, row0, k_first, k_count, wave >> 1);
    ob.init(p.b + w.batch * p.sb, p.ldb, p.N, col0, k_first, k_count, wave & 1);
    float4v acc[MI][NJ];
    if constexpr (ST == 2)      mainloop<T, MI, NJ, 2>(oa, ob, static_cast<int>(k_count), {a0, a1}, {b0, b1}, acc);
    else if constexpr (ST == 3) mainloop<T, MI, NJ, 3>(oa, ob, static_cast<int>(k_count), {a0, a1, a2}, {b0, b1, b2}, acc);
    else                        mainloop<T, MI, NJ, 4>(oa, ob, static_cast<int>(k_count), {a0, a1, a2, a3}, {b0, b1, b2, b3}, acc);

    const int lane = threadIdx.x & 63;
    const int l16 = lane & 15, kq = lane >> 4;
    const long wrow = row0 + (wave >> 1) * 16 * MI + l16, wcol = col0 + (wave & 1) * 16 * NJ + 4 * kq;
    if (p.splits > 1) {
        float* dst = static_cast<float*>(p.out) + static_cast<long>(w.batch * static_cast<int>(p.splits) + w.split) * (static_cast<long>(p.M) * p.N);
        const bool vec = p.N % 4 == 0;
#pragma unroll
        for (int i = 0; i < MI; ++i) {
            const long row = wrow + i * 16;
            if (row >= p.M) continue;
#pragma unroll
            for (int j = 0; j < NJ; ++j) {
                const long col = wcol + j * 16;
                if (vec) {
                    if (col < p.N) *reinterpret_cast<float4v*>(dst + row * p.N + col) = acc[i][j];
                } else {
#pragma unroll
                    for (int r = 0; r < 4; ++r)
                        if (col + r < p.N) dst[row * p.N + col + r] = acc[i][j][r];
                }
            }
        }
        return;
    }
    std::uint16_t* C = static_cast<std::uint16_t*>(p.out) + w.batch * p.sc;
    const std::uint16_t* ADD = p.add ? p.add + w.batch * p.sadd : nullptr;
    // plain product into rows of 8-byte aligned pieces: the conversion instruction, four columns per store; a
    // row block in which a NaN turns up takes the software narrowing (which writes NaNs as the host's types do)
    const bool plain = p.alpha == 1.0f && ADD == nullptr && p.ldc % 4 == 0 && p.sc % 4 == 0 && (reinterpret_cast<uintptr_t>(p.out) & 7) == 0;
#pragma unroll
    for (int i = 0; i < MI; ++i) {
        const long row = wrow + i * 16;
        bool nan_here = false;
        if (plain) {
            float probe = 0.0f;
#pragma unroll
            for (int j = 0; j < NJ; ++j)
#pragma unroll
                for (int r = 0; r < 4; ++r) probe += acc[i][j][r];
            nan_here = __builtin_amdgcn_ballot_w64(probe != probe) != 0;      // (an infinity minus an infinity counts as well)
        }
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
            const long col = wcol + j * 16;
            if (row >= p.M || col >= p.N) continue;
            if (plain && col + 3 < p.N) {
                std::uint16_t o[4];
                if (__builtin_expect(nan_here, 0)) {
#pragma unroll
                    for (int r = 0; r < 4; ++r) o[r] = El::from_f32(acc[i][j][r]);
                } else {
#pragma unroll
                    for (int r = 0; r < 4; ++r) o[r] = El::from_f32_finite(acc[i][j][r]);
                }
                u32x2 w2;
                w2[0] = o[0] | (static_cast<std::uint32_t>(o[1]) << 16);
                w2[1] = o[2] | (static_cast<std::uint32_t>(o[3]) << 16);
                *reinterpret_cast<u32x2*>(C + row * p.ldc + col) = w2;
            } else {
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    if (col + r >= p.N) continue;
                    float v = p.alpha * acc[i][j][r];
                    if (ADD) v = fmaf(p.beta, El::to_f32(ADD[row * p.ld_add + col + r]), v);
                    C[row * p.ldc + col + r] = El::from_f32(v);
                }
            }
        }
    }
}

// Tile forms; kTiles in gemm_flex.hip describes them in the same order.
template <typename T, bool AR, bool BR>
void launch_tile(int tile, const Params& p, unsigned grid, hipStream_t s) {
    const dim3 g(grid), t(kThreads);
    if constexpr (!AR && !BR) {          // (the permuted units of a tile that lies along its rows need widths of 64 or 128)
        switch (tile) {
            case 12: hipLaunchKernelGGL((gemm_flex_kernel<T, 8, 7, 2, AR, BR>), g, t, 0, s, p); return;
            case 13: hipLaunchKernelGGL((gemm_flex_kernel<T, 7, 7, 2, AR, BR>), g, t, 0, s, p); return;
            case 14: hipLaunchKernelGGL((gemm_flex_kernel<T, 6, 7, 2, AR, BR>), g, t, 0, s, p); return;
        }
    }
    switch (tile) {
        case 0: hipLaunchKernelGGL((gemm_flex_kernel<T, 8, 8, 2, AR, BR>), g, t, 0, s, p); break;
        case 1: hipLaunchKernelGGL((gemm_flex_kernel<T, 6, 8, 2, AR, BR>), g, t, 0, s, p); break;
        case 2: hipLaunchKernelGGL((gemm_flex_kernel<T, 6, 6, 3, AR, BR>), g, t, 0, s, p); break;
        case 3: hipLaunchKernelGGL((gemm_flex_kernel<T, 6, 4, 3, AR, BR>), g, t, 0, s, p); break;
        case 4: hipLaunchKernelGGL((gemm_flex_kernel<T, 4, 4, 2, AR, BR>), g, t, 0, s, p); break;
        case 5: hipLaunchKernelGGL((gemm_flex_kernel<T, 4, 4, 3, AR, BR>), g, t, 0, s, p); break;
        case 6: hipLaunchKernelGGL((gemm_flex_kernel<T, 2, 4, 2, AR, BR>), g, t, 0, s, p); break;
        case 7: hipLaunchKernelGGL((gemm_flex_kernel<T, 2, 4, 4, AR, BR>), g, t, 0, s, p); break;
        case 8: hipLaunchKernelGGL((gemm_flex_kernel<T, 2, 2, 2, AR, BR>), g, t, 0, s, p); break;
        case 9: hipLaunchKernelGGL((gemm_flex_kernel<T, 2, 2, 3, AR, BR>), g, t, 0, s, p); break;
        case 10: hipLaunchKernelGGL((gemm_flex_kernel<T, 2, 2, 4, AR, BR>), g, t, 0, s, p); break;
        default: hipLaunchKernelGGL((gemm_flex_kernel<T, 1, 4, 4, AR, BR>), g, t, 0, s, p); break;
    }
}

// One explicit instantiation per translation unit (gemm_flex_{kk,kr,rr}.hip): which operands lie along the rows.
void launch_kk(bool bf16, int tile, const Params& p, unsigned grid, hipStream_t s);   // x W^T
void launch_kr(bool bf16, int tile, const Params& p, unsigned grid, hipStream_t s);   // dy W
void launch_rr(bool bf16, int tile, const Params& p, unsigned grid, hipStream_t s);   // dy^T x

}  // namespace flex
}  // namespace paras
