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
#pragma unroll
            for (int j = 0; j < NJ; ++j) {
                const long col = wcol + j * 16;
                const float4v v = in_turn<2>(acc[i][j]);
                if (row >= p.M) continue;
                if (vec) {
                    if (col < p.N) *reinterpret_cast<float4v*>(dst + row * p.N + col) = v;
                } else {
#pragma unroll
                    for (int r = 0; r < 4; ++r)
                        if (col + r < p.N) dst[row * p.N + col + r] = v[r];
                }
            }
        }
        return;
    }
    // Whole rows from LDS.  Stored from the accumulators, 8 bytes a lane with a test per store (and two bytes with an addend), a tile of 256 x 256
    // took 8 us for its stores, a burst from all CUs at once.  Forward and both gradients, that and this: bf16 3000 x 4096 x 4096 268 and 253 us,
    // 8192 x 2048 x 2048 with a bias 268 and 213, fp16 4555 x 9152 x 64 89.5 and 79.8.
    lds_u16* const out = wave == 0 ? (lds_u16*)a0 : wave == 1 ? (lds_u16*)a1 : wave == 2 ? (lds_u16*)b0 : (lds_u16*)b1;
    static_assert(16 * MI * 16 * NJ <= OA::kElems && 16 * MI * 16 * NJ <= OB::kElems, "a wave's rows in a stage");
    __syncthreads();                                        // (no wave's requests are on their way to the stages)
    float probe = 0.0f;                                     // (an infinity minus an infinity counts as a NaN as well)
    if (p.alpha == 1.0f && p.add == nullptr) {
#pragma unroll
        for (int i = 0; i < MI; ++i)
#pragma unroll
            for (int j = 0; j < NJ; ++j) {
                const float4v v = in_turn<0>(acc[i][j]);
                probe += (v[0] + v[1]) + (v[2] + v[3]);
                RowsOut<NJ>::lay(out, i * 16 + l16, j, kq, pack4<T>(v));
            }
    } else {
        // (rows and columns that do not exist take an addend that does: their results are not stored)
        const std::uint16_t* add = p.add ? p.add + w.batch * p.sadd : nullptr;
        const bool four = p.N % 4 == 0 && ((p.ld_add | p.sadd) & 3) == 0 && (reinterpret_cast<uintptr_t>(p.add) & 7) == 0;
#pragma unroll
        for (int i = 0; i < MI; ++i) {
            const long row = wrow + i * 16 < p.M ? wrow + i * 16 : p.M - 1;
            const std::uint16_t* from = add + row * p.ld_add;
#pragma unroll
            for (int j = 0; j < NJ; ++j) {
                const long col = wcol + j * 16;
                float4v v = in_turn<1>(acc[i][j]);
#pragma unroll
                for (int r = 0; r < 4; ++r) v[r] *= p.alpha;
                if (add) {
                    float4v b;
                    if (four) {
                        const u32x2 t = *reinterpret_cast<const u32x2*>(from + (col < p.N ? col : p.N - 4));
#pragma unroll
                        for (int r = 0; r < 4; ++r) b[r] = El::to_f32(static_cast<std::uint16_t>(t[r >> 1] >> (16 * (r & 1))));
                    } else {
#pragma unroll
                        for (int r = 0; r < 4; ++r) b[r] = El::to_f32(from[col + r < p.N ? col + r : p.N - 1]);
                    }
#pragma unroll
                    for (int r = 0; r < 4; ++r) v[r] = fmaf(p.beta, b[r], v[r]);
                }
                probe += (v[0] + v[1]) + (v[2] + v[3]);
                RowsOut<NJ>::lay(out, i * 16 + l16, j, kq, pack4<T>(v));
            }
        }
    }
    const bool nan_here = __builtin_amdgcn_ballot_w64(probe != probe) != 0;
    const bool wide = ((p.ldc | p.sc) & 7) == 0 && (reinterpret_cast<uintptr_t>(p.out) & 15) == 0;
    const long r0 = wrow - l16, c0 = wcol - 4 * kq;
    store_rows<T, MI, NJ>(out, static_cast<std::uint16_t*>(p.out) + w.batch * p.sc + r0 * p.ldc + c0, p.ldc, p.M - r0, p.N - c0, wide, nan_here);
}

// Tile forms; kTiles in gemm_flex.hip describes them in the same order.
template <typename T, bool AR, bool BR>
void launch_tile(int tile, const Params& p, unsigned grid, hipStream_t s) {
    const dim3 g(grid), t(kThreads);
    if constexpr (!AR) {                 // (a tile that lies along its rows permutes 32-byte units in groups of four: its width is 32 or a multiple of 64)
        switch (tile) {
            case 13: hipLaunchKernelGGL((gemm_flex_kernel<T, 3, 4, 4, AR, BR>), g, t, 0, s, p); return;
            case 14: hipLaunchKernelGGL((gemm_flex_kernel<T, 3, 4, 2, AR, BR>), g, t, 0, s, p); return;
            case 15: hipLaunchKernelGGL((gemm_flex_kernel<T, 3, 2, 4, AR, BR>), g, t, 0, s, p); return;
            case 16: hipLaunchKernelGGL((gemm_flex_kernel<T, 5, 4, 2, AR, BR>), g, t, 0, s, p); return;
        }
        if constexpr (!BR) {
            switch (tile) {
                case 17: hipLaunchKernelGGL((gemm_flex_kernel<T, 8, 7, 2, AR, BR>), g, t, 0, s, p); return;
                case 18: hipLaunchKernelGGL((gemm_flex_kernel<T, 6, 7, 2, AR, BR>), g, t, 0, s, p); return;
            }
        }
    }
    switch (tile) {
        case 0: hipLaunchKernelGGL((gemm_flex_kernel<T, 8, 8, 2, AR, BR>), g, t, 0, s, p); break;
        case 1: hipLaunchKernelGGL((gemm_flex_kernel<T, 6, 8, 2, AR, BR>), g, t, 0, s, p); break;
        case 2: hipLaunchKernelGGL((gemm_flex_kernel<T, 6, 6, 3, AR, BR>), g, t, 0, s, p); break;
        case 3: hipLaunchKernelGGL((gemm_flex_kernel<T, 6, 4, 4, AR, BR>), g, t, 0, s, p); break;
        case 4: hipLaunchKernelGGL((gemm_flex_kernel<T, 4, 4, 2, AR, BR>), g, t, 0, s, p); break;
        case 5: hipLaunchKernelGGL((gemm_flex_kernel<T, 4, 4, 4, AR, BR>), g, t, 0, s, p); break;
        case 6: hipLaunchKernelGGL((gemm_flex_kernel<T, 2, 4, 2, AR, BR>), g, t, 0, s, p); break;
        case 7: hipLaunchKernelGGL((gemm_flex_kernel<T, 2, 4, 4, AR, BR>), g, t, 0, s, p); break;
        case 8: hipLaunchKernelGGL((gemm_flex_kernel<T, 2, 2, 3, AR, BR>), g, t, 0, s, p); break;
        case 9: hipLaunchKernelGGL((gemm_flex_kernel<T, 2, 2, 4, AR, BR>), g, t, 0, s, p); break;
        case 10: hipLaunchKernelGGL((gemm_flex_kernel<T, 4, 2, 3, AR, BR>), g, t, 0, s, p); break;
        case 11: hipLaunchKernelGGL((gemm_flex_kernel<T, 1, 2, 4, AR, BR>), g, t, 0, s, p); break;
        default: hipLaunchKernelGGL((gemm_flex_kernel<T, 6, 4, 2, AR, BR>), g, t, 0, s, p); break;
    }
}

// One explicit instantiation per translation unit (gemm_flex_{kk,kr,rr}.hip): which operands lie along the rows.
void launch_kk(bool bf16, int tile, const Params& p, unsigned grid, hipStream_t s);   // x W^T
void launch_kr(bool bf16, int tile, const Params& p, unsigned grid, hipStream_t s);   // dy W
void launch_rr(bool bf16, int tile, const Params& p, unsigned grid, hipStream_t s);   // dy^T x

}  // namespace flex
}  // namespace paras
