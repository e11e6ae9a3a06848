// Dense (optionally batched) products for gfx950, fp32 accumulation and one rounding:
//
//   C[b] = T( alpha * A[b] B[b]^T + beta * addend[b] )      A [M, K], B [N, K], C [M, N]
//
// The reference bounces mm / bmm / addmm / linear to ATen on the host
// (csrc/ops/vision_ops.cpp:248-309,388-423: copy to CPU, at::mm / at::bmm /
// at::addmm / at::linear with fp32 accumulation and one rounding, copy back).
// This file holds the choice of kernel, the kernels for few rows (which stream the
// weights of a decode-time projection) and the general kernel for what no other takes; the
// tile kernels are gemm_flex.hip (16-bit) and gemm_f32.hip, and take operands that are contiguous along
// the contraction ("NT": x W^T of nn.Linear, q k^T) or along their rows (its gradients).
// `addend` is a matrix with row stride ld_add; ld_add = 0 broadcasts one row
// (a bias) over all rows.
#include <hip/hip_runtime.h>
#include <type_traits>

#include "core/device_context.h"
#include "core/device_math.h"
#include "core/status.h"
#include "kernels/gemm_f32_host.h"
#include "kernels/gemm_flex_host.h"
#include "kernels/gemm_tile.h"
#include "kernels/stream_rows.h"
#include "paras_hip.h"

namespace paras {
namespace {

using namespace gemm;

struct DenseParams {
    const std::uint16_t* a;
    const std::uint16_t* b;
    const std::uint16_t* add;   // may be null
    std::uint16_t* c;
    long M, N, K;
    long lda, ldb, ldc, ld_add;
    long sa, sb, sc, sadd;      // batch strides (elements)
    float alpha, beta;
    double alpha64, beta64;     // the same, for fp64 tensors
    int  swapped;               // few-row kernels only: a and b have changed places (few output COLUMNS, many rows), so a
                                // result (row of a, row of b) belongs at c[row of b][row of a], and the addend likewise
};

// ---- up to 32 rows (from 17 on over contractions of less than 6144 or more than 4096 weight rows: few_rows_up_to): the decode-time projections, bound by streaming the weights once.  A workgroup owns 16 NBG
// weight rows and its eight waves split the contraction (stream_rows.h); 8 XQ activation rows at most.
using stream::Mma16;

// What the streaming kernel needs of DenseParams, in 112 bytes: a launch whose arguments take more costs the host 0.7 us more, 3.4 for 2.7.
struct FewParams {
    const std::uint16_t* a;
    const std::uint16_t* b;
    const std::uint16_t* add;
    std::uint16_t* c;
    long sa, sb, sc, sadd, ldc, ld_add;
    std::uint16_t M, swapped;       // (up to 32 rows)
    int  N, K;
    int  lda, ldb;                  // (flex::takes(), as N and K)
    int  rows_each;
    float alpha, beta;
};
static_assert(sizeof(FewParams) <= 112, "see above");

template <typename T, typename P>
__device__ __forceinline__ void few_rows_store(const P& p, std::uint16_t* C, const std::uint16_t* ADD, bool vec_ok, long row, long col, long cols, float4_t t) {
    using El = Elem<T>;
    if (row >= p.M) return;
    if (p.swapped) {        // `row` is a column of the caller's result and `col + r` a row of it
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            if (col + r >= cols) continue;
            float v = p.alpha * t[r];
            if (ADD) v = fmaf(p.beta, El::to_f32(ADD[(col + r) * p.ld_add + row]), v);
            C[(col + r) * p.ldc + row] = El::from_f32(v);
        }
        return;
    }
    std::uint16_t o16[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        float v = p.alpha * t[r];
        if (ADD && col + r < cols) v = fmaf(p.beta, El::to_f32(ADD[row * p.ld_add + col + r]), v);
        o16[r] = El::from_f32(v);
    }
    if (vec_ok && col + 3 < cols) {
        u32x2 w2;
        w2[0] = o16[0] | (static_cast<std::uint32_t>(o16[1]) << 16);
        w2[1] = o16[2] | (static_cast<std::uint32_t>(o16[3]) << 16);
        *reinterpret_cast<u32x2*>(C + row * p.ldc + col) = w2;
    } else {
#pragma unroll
        for (int r = 0; r < 4; ++r)
            if (col + r < cols) C[row * p.ldc + col + r] = o16[r];
    }
}
template <typename P>
__device__ __forceinline__ bool few_rows_vec(const P& p) {
    return (p.ldc % 4 == 0) && (p.sc % 4 == 0) && ((reinterpret_cast<uintptr_t>(p.c) & 7) == 0);
}

template <typename T, int NBG, int XQ>
__global__ __launch_bounds__(stream::kThreads, 4) void stream_gemm_nt_kernel(const FewParams p) {
    using S = stream::Shape<1, NBG, XQ>;
    constexpr int MB = S::kXBlocks;
    __shared__ __attribute__((aligned(1024))) std::uint16_t lds[S::kLdsElems];
    // (One fetch for all of them: left to itself the compiler fetches what places the result in front of the stores, 0.2 us of a product.)
    asm volatile("" ::"s"(p.M), "s"(p.swapped), "s"(p.N), "s"(p.K), "s"(p.lda), "s"(p.ldb), "s"(p.rows_each), "s"(p.alpha), "s"(p.beta), "s"(p.ldc), "s"(p.c));
    const long bidx = blockIdx.y;
    const std::uint16_t* A = p.a + bidx * p.sa;
    const int lane = threadIdx.x & 63;
    const long n0 = static_cast<long>(blockIdx.x) * p.rows_each, rows = p.N - n0 < p.rows_each ? p.N - n0 : p.rows_each;
    const std::uint16_t* const w[1] = {p.b + bidx * p.sb + n0 * p.ldb};
    std::uint32_t x_off[XQ];
#pragma unroll
    for (int q = 0; q < XQ; ++q) {
        long xrow = q * 8 + (lane >> 3);
        if (xrow >= p.M) xrow = p.M - 1;                    // clamped rows are computed but never stored
        x_off[q] = static_cast<std::uint32_t>(xrow * p.lda * 2);
    }
    constexpr int step = 16 * NBG;
    const int count = static_cast<int>((rows + step - 1) / step);
    stream::products<T, 1, NBG, XQ, true>(w, p.ldb, rows, step, count, p.K, A, (static_cast<long>(p.M - 1) * p.lda + p.K) * 2, x_off, lds,
                                    [&](int j, const float4_t (&acc)[NBG][MB]) __attribute__((always_inline)) {
        stream::share<NBG, MB>(lds, acc);
        const int blk = stream::wave_id();                  // wave w finishes result block w
        if (blk < NBG * MB) {
            const float4_t t = stream::sum_of<NBG, MB>(lds, blk / MB, blk % MB);
            if (XQ > 1 || (lane & 15) < 8)
                few_rows_store<T>(p, p.c + bidx * p.sc, p.add ? p.add + bidx * p.sadd : nullptr, few_rows_vec(p), (blk % MB) * 16 + (lane & 15),
                                  n0 + j * step + (blk / MB) * 16 + 4 * (lane >> 4), n0 + rows, t);
        }
        lds_barrier();                                      // the LDS is free for the next block
    });
}

// ---- 33 to 128 rows, as few_rows_up_to says: the same split, but with this many activation rows per weight row a trip
// through LDS for each would cost more than it saves, so every wave feeds its MFMAs straight from memory (weights
// as the row operand, with plain loads: non-temporal ones measured 5-18 % slower, each 128-byte line being touched by two
// instructions; the activation rows from L2), and the eight partial results meet in LDS in wave order.  Lane l of
// a 16x16 result holds activation row l%16 and weight rows 4*(l/16) .. +3.
constexpr int kSkinnyWaves = 8;
constexpr int kSkinnyMaxM = 128;
constexpr int kFewRowsM = 32;            // the staged tiles take over from here, and from 17 rows on over long contractions (few_rows_up_to)

template <typename T, int MB, int NB>   // MB = 16-row blocks of activations, NB = 16-row blocks of weights per workgroup
__global__ __launch_bounds__(kSkinnyWaves * 64) void skinny_gemm_nt_kernel(const DenseParams p) {
    using El = Elem<T>;
    __shared__ float4_t part[kSkinnyWaves][NB * MB][64];
    const long bidx = blockIdx.y;
    const std::uint16_t* A = p.a + bidx * p.sa;
    const std::uint16_t* B = p.b + bidx * p.sb;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int r16 = lane & 15, kg = lane >> 4;
    const long n0 = static_cast<long>(blockIdx.x) * (16 * NB);
    const std::uint16_t* wp[NB];
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
        long wrow = n0 + nb * 16 + r16;
        if (wrow >= p.N) wrow = p.N - 1;                    // clamped rows are computed but never stored
        wp[nb] = B + wrow * p.ldb + kg * 16;
    }
    const std::uint16_t* xp[MB];
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) {
        long xrow = mb * 16 + r16;
        if (xrow >= p.M) xrow = p.M - 1;
        xp[mb] = A + xrow * p.lda + kg * 16;
    }
    float4_t acc[NB][MB];
#pragma unroll
    for (int nb = 0; nb < NB; ++nb)
#pragma unroll
        for (int mb = 0; mb < MB; ++mb) acc[nb][mb] = float4_t{0.f, 0.f, 0.f, 0.f};
    // The contraction is walked in pieces of 64 (two MFMAs): lane group kg supplies elements
    // 16 kg .. 16 kg + 7 of a piece to the first MFMA and the next eight to the second -- any
    // assignment works as long as both operands use the same one -- so that the four groups
    // together read whole 128-byte lines of a row.  A batch is kPieces pieces: every load of the
    // batch is requested before its first MFMA, so a wave pays the memory latency once per batch.
    const long pieces = p.K / 64;
    constexpr int kPieces = MB <= 4 ? 2 : 1;
    // this wave's pieces are wave, wave + W, ...; each workgroup starts at a different one of them and
    // wraps around, so that the workgroups do not all read the same part of every weight row at once
    const long mine = pieces > wave ? (pieces - wave + kSkinnyWaves - 1) / kSkinnyWaves : 0;
    const long first = mine > 0 ? (static_cast<long>(blockIdx.x) * 3) % mine : 0;
    auto piece_at = [&](long t) {
        long r = t + first;
        if (r >= mine) r -= mine;
        return (wave + r * kSkinnyWaves) * 64;
    };
    long t = 0;
    for (; t + kPieces <= mine; t += kPieces) {
        u32x4 wv[kPieces][2][NB], xv[kPieces][2][MB];
#pragma unroll
        for (int u = 0; u < kPieces; ++u)
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const long k = piece_at(t + u) + h * 8;
#pragma unroll
                for (int nb = 0; nb < NB; ++nb) wv[u][h][nb] = load16(wp[nb] + k);
#pragma unroll
                for (int mb = 0; mb < MB; ++mb) xv[u][h][mb] = load16(xp[mb] + k);
            }
#pragma unroll
        for (int u = 0; u < kPieces; ++u)
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int mb = 0; mb < MB; ++mb)
#pragma unroll
                    for (int nb = 0; nb < NB; ++nb) acc[nb][mb] = Mma16<T>::run(wv[u][h][nb], xv[u][h][mb], acc[nb][mb]);
    }
    for (; t < mine; ++t) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const long k = piece_at(t) + h * 8;
            u32x4 wv[NB];
#pragma unroll
            for (int nb = 0; nb < NB; ++nb) wv[nb] = load16(wp[nb] + k);
#pragma unroll
            for (int mb = 0; mb < MB; ++mb) {
                const u32x4 xv = load16(xp[mb] + k);
#pragma unroll
                for (int nb = 0; nb < NB; ++nb) acc[nb][mb] = Mma16<T>::run(wv[nb], xv, acc[nb][mb]);
            }
        }
    }
#pragma unroll
    for (int nb = 0; nb < NB; ++nb)
#pragma unroll
        for (int mb = 0; mb < MB; ++mb) part[wave][nb * MB + mb][lane] = acc[nb][mb];
    __syncthreads();
    // wave w finishes result blocks w, w + 8, ...
    std::uint16_t* C = p.c + bidx * p.sc;
    const std::uint16_t* ADD = p.add ? p.add + bidx * p.sadd : nullptr;
    const bool vec_ok = few_rows_vec(p);
    for (int blk = wave; blk < NB * MB; blk += kSkinnyWaves) {
        float4_t t = part[0][blk][lane];
#pragma unroll
        for (int w = 1; w < kSkinnyWaves; ++w) {
            const float4_t o = part[w][blk][lane];
#pragma unroll
            for (int r = 0; r < 4; ++r) t[r] += o[r];
        }
        few_rows_store<T>(p, C, ADD, vec_ok, (blk % MB) * 16 + r16, n0 + (blk / MB) * 16 + 4 * kg, p.N, t);
    }
}

// Up to 32 rows: the weight rows are dealt out evenly, one workgroup per CU or two where a CU's share is more than 32 of them,
// in blocks of 16 rows, or of 32 from a share of 17 on (the activations are read once per block).  The last block of a workgroup is cut
// short where its share ends: rows past it are requested with an empty extent.  Whole blocks of 16 for everyone left 64 of 256
// CUs with one block where the others had two (8 x 14336 x 4096 27.0 us, 28 rows each 21.8; 16 x 7168 x 2048 9.3 -> 7.8),
// and shares below eight rows ask for less than a request holds (8 x 4096 x 4096 16 / 8 / 4 rows each: 9.6 / 11.0 / 17.3 us; 1024
// rows 6.1 / 5.9 / 5.9).
// More rows than 32: two blocks of weight rows per workgroup when that still leaves a workgroup for every CU: every
// activation fragment then feeds two MFMAs, which halves the reads of the activations from L2.
template <typename T>
void launch_skinny(const DenseParams& p, long batch, hipStream_t s) {
    const dim3 block(kSkinnyWaves * 64);
    const int mb = static_cast<int>((p.M + 15) / 16);
    if (mb <= 2) {
        constexpr long kCus = 256;
        auto share = [&](long workgroups) { return ((p.N * batch + workgroups - 1) / workgroups + 3) / 4 * 4; };
        const bool two = share(kCus) > 16;
        const long even = share(kCus) > 32 ? share(2 * kCus) : (share(kCus) > 8 ? share(kCus) : 8), rows_each = even < p.N ? even : p.N;
        const dim3 g(static_cast<unsigned>((p.N + rows_each - 1) / rows_each), static_cast<unsigned>(batch));
        auto narrow = [](long v) { return static_cast<int>(v); };
        const FewParams f{p.a, p.b, p.add, p.c, p.sa, p.sb, p.sc, p.sadd, p.ldc, p.ld_add, static_cast<std::uint16_t>(p.M), static_cast<std::uint16_t>(p.swapped),
                          narrow(p.N), narrow(p.K), narrow(p.lda), narrow(p.ldb), narrow(rows_each), p.alpha, p.beta};
        if (p.M <= 8)     { if (two) hipLaunchKernelGGL((stream_gemm_nt_kernel<T, 2, 1>), g, block, 0, s, f);
                            else     hipLaunchKernelGGL((stream_gemm_nt_kernel<T, 1, 1>), g, block, 0, s, f); }
        else if (mb <= 1) { if (two) hipLaunchKernelGGL((stream_gemm_nt_kernel<T, 2, 2>), g, block, 0, s, f);
                            else     hipLaunchKernelGGL((stream_gemm_nt_kernel<T, 1, 2>), g, block, 0, s, f); }
        else              { if (two) hipLaunchKernelGGL((stream_gemm_nt_kernel<T, 2, 4>), g, block, 0, s, f);
                            else     hipLaunchKernelGGL((stream_gemm_nt_kernel<T, 1, 4>), g, block, 0, s, f); }
        return;
    }
    const dim3 g1(static_cast<unsigned>((p.N + 15) / 16), static_cast<unsigned>(batch));
    const dim3 g2(static_cast<unsigned>((p.N + 31) / 32), static_cast<unsigned>(batch));
    const bool two = static_cast<long>(g2.x) * batch >= 256;
    if (mb <= 4) { if (two) hipLaunchKernelGGL((skinny_gemm_nt_kernel<T, 4, 2>), g2, block, 0, s, p);
                   else     hipLaunchKernelGGL((skinny_gemm_nt_kernel<T, 4, 1>), g1, block, 0, s, p); }
    else         { if (two) hipLaunchKernelGGL((skinny_gemm_nt_kernel<T, 8, 2>), g2, block, 0, s, p);
                   else     hipLaunchKernelGGL((skinny_gemm_nt_kernel<T, 8, 1>), g1, block, 0, s, p); }
}

// ---- few rows with a workspace: the same product with the activations read once per 128 weight
// rows instead of once per 16.  In the kernel above every workgroup re-reads all M x K activations
// from L2, which -- not the weights -- bounds it from M = 32 upwards.  Here the eight waves of a
// workgroup own eight blocks of 16 weight rows and walk the SAME part of the contraction, so a slab
// of activations (M rows x 256 elements) is brought into LDS once and shared; the contraction is
// split over workgroups instead (grid.x), each writes its fp32 partial result to the workspace, and
// a second kernel adds the partials in split order and applies the epilogue: deterministic, and
// 128 / 16 = 8 times fewer activation reads for a workspace of splits x M x N floats.
constexpr int kSlab = 256;                 // contraction elements per LDS slab (4 pieces of 64)
constexpr int kSlabLd = kSlab + 8;         // LDS row stride (elements): 16 consecutive rows hit distinct banks

template <typename T, int MB>
__global__ __launch_bounds__(512) void skinny_splitk_kernel(const DenseParams p, float* __restrict__ partial, int pieces_per_split) {
    __shared__ __attribute__((aligned(16))) std::uint16_t xs[2][MB * 16 * kSlabLd];
    const long bidx = blockIdx.z;
    const std::uint16_t* A = p.a + bidx * p.sa;
    const std::uint16_t* B = p.b + bidx * p.sb;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int r16 = lane & 15, kg = lane >> 4;
    // grid.x = split, grid.y = block of 128 weight rows: workgroups that run together read adjacent
    // parts of the same weight rows
    const long n0 = static_cast<long>(blockIdx.y) * 128 + wave * 16;
    long wrow = n0 + r16;
    if (wrow >= p.N) wrow = p.N - 1;                        // clamped rows are computed but never stored
    const std::uint16_t* wp = B + wrow * p.ldb + kg * 16;
    const long pieces = p.K / 64;
    const long pc0 = static_cast<long>(blockIdx.x) * pieces_per_split;
    const long pc1 = pc0 + pieces_per_split < pieces ? pc0 + pieces_per_split : pieces;
    // staging of a slab: MB*16 rows x 32 chunks of 16 bytes, 512 threads -> MB chunks per thread
    u32x4 stage[MB];
    auto load_slab = [&](long pc) {                         // pieces pc .. pc+3 (clamped to the split's end)
#pragma unroll
        for (int i = 0; i < MB; ++i) {
            const int c = tid + i * 512;
            long row = c >> 5;
            const long k = pc * 64 + (c & 31) * 8;
            if (row >= p.M) row = p.M - 1;
            stage[i] = k < pc1 * 64 ? load16(A + row * p.lda + k) : u32x4{0, 0, 0, 0};
        }
    };
    auto store_slab = [&](int buf) {
#pragma unroll
        for (int i = 0; i < MB; ++i) {
            const int c = tid + i * 512;
            *reinterpret_cast<u32x4*>(&xs[buf][(c >> 5) * kSlabLd + (c & 31) * 8]) = stage[i];
        }
    };
    float4_t acc[MB];
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) acc[mb] = float4_t{0.f, 0.f, 0.f, 0.f};
    // Weights and activations of slab s+1 are requested before the MFMAs of slab s, so that two
    // slabs' worth of loads are in flight per wave and a split of two slabs pays the memory latency
    // about once.
    u32x4 wv[4][2], wn[4][2];
    auto load_w = [&](long pc, u32x4 (&dst)[4][2]) {
#pragma unroll
        for (int u = 0; u < 4; ++u)
#pragma unroll
            for (int h = 0; h < 2; ++h)
                dst[u][h] = pc + u < pc1 ? load16(wp + (pc + u) * 64 + h * 8) : u32x4{0, 0, 0, 0};
    };
    // The slabs of the split are walked from a different starting slab in every block of weight rows
    // (and wrap around), so that the workgroups of one split do not read the same part of their rows
    // at the same time.
    const long nslabs = pc1 > pc0 ? (pc1 - pc0 + 3) / 4 : 0;
    const long rot = nslabs > 0 ? static_cast<long>(blockIdx.y) % nslabs : 0;
    auto slab_pc = [&](long i) {
        long r = i + rot;
        if (r >= nslabs) r -= nslabs;
        return pc0 + 4 * r;
    };
    if (nslabs > 0) {
        load_slab(slab_pc(0));
        load_w(slab_pc(0), wv);
        store_slab(0);
    }
    __syncthreads();
    int buf = 0;
    for (long i = 0; i < nslabs; ++i, buf ^= 1) {
        const bool more = i + 1 < nslabs;
        if (more) {
            load_slab(slab_pc(i + 1));
            load_w(slab_pc(i + 1), wn);
        }
#pragma unroll
        for (int u = 0; u < 4; ++u)
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int mb = 0; mb < MB; ++mb) {
                    const u32x4 xv = *reinterpret_cast<const u32x4*>(&xs[buf][(mb * 16 + r16) * kSlabLd + u * 64 + kg * 16 + h * 8]);
                    acc[mb] = Mma16<T>::run(wv[u][h], xv, acc[mb]);
                }
        if (more) {
            store_slab(buf ^ 1);
#pragma unroll
            for (int u = 0; u < 4; ++u)
#pragma unroll
                for (int h = 0; h < 2; ++h) wv[u][h] = wn[u][h];
        }
        __syncthreads();
    }
    // partial[(batch, split)][row][col]: lane holds row mb*16 + r16, columns n0 + 4 kg .. + 3
    float* dst = partial + (bidx * gridDim.x + blockIdx.x) * (p.M * p.N);
    const long col = n0 + 4 * kg;
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) {
        const long row = mb * 16 + r16;
        if (row >= p.M) continue;
#pragma unroll
        for (int r = 0; r < 4; ++r)
            if (col + r < p.N) dst[row * p.N + col + r] = acc[mb][r];
    }
}

template <typename T>
__global__ __launch_bounds__(256) void skinny_splitk_finish_kernel(const DenseParams p, const float* __restrict__ partial, int splits) {
    using El = Elem<T>;
    const long mn = p.M * p.N;
    const long i = static_cast<long>(blockIdx.x) * 256 + threadIdx.x;
    if (i >= mn) return;
    const long bidx = blockIdx.y;
    const float* src = partial + bidx * splits * mn + i;
    float t = 0.f;
    for (int sp = 0; sp < splits; ++sp) t += src[sp * mn];
    const long row = i / p.N, col = i % p.N;
    float v = p.alpha * t;
    if (p.add) v = fmaf(p.beta, El::to_f32((p.add + bidx * p.sadd)[row * p.ld_add + col]), v);
    (p.c + bidx * p.sc)[row * p.ldc + col] = El::from_f32(v);
}

// Few rows but many columns (a vocabulary projection, a fused gate-up projection at M = 64 ... 128):
// from about 200 tiles of 128 x 128 the tile kernel streams the weights faster than the few-row
// kernels do (M = 128, N = 128256, K = 4096: 267 against 649 us; N = 28672: 75 against 106 us; at
// N = 6144 the few-row kernels win, 47 against 67 us).  Up to 32 rows few_rows_up_to decides alone.
bool few_rows_by_tiles(long M, long N, long batch) {
    return M > 32 && M <= kSkinnyMaxM && (N + gemm::kBN - 1) / gemm::kBN * batch >= 192;
}

// From 33 rows on the staged tiles are faster but for short contractions of few weight rows, where their start is most of
// the call: few-row kernels / tiles, 33 x 512 x 512 4.3 / 4.9 us, 48 x 3072 x 512 4.8 / 5.2, 64 x 1024 x 512 5.0 / 5.1, 64 x 4096 x 256 4.1 / 4.4;
// 64 x 4096 x 512 5.7 / 5.4, 40 x 2048 x 1024 7.0 / 6.7, 64 x 1024 x 1024 7.2 / 6.5, 33 x 6144 x 512 6.5 / 5.3, 56 x 4384 x 256 4.9 / 4.4,
// 63 x 7192 x 1024 12.5 / 7.0, 108 x 7456 x 6656 110 / 36; 128 products of 64 x 64 x 64 3.7 / 4.2, two of 100 x 512 x 64 3.7 / 4.1,
// eight of 128 x 512 x 64 4.1 / 4.3; two of 100 x 128 x 128 4.0 / 4.0, 128 of 33 x 512 x 64 6.0 / 6.0.  Where the tiles want the contraction in parts and the caller has no workspace for
// them, and for paras_gemm_nt, the few-row kernels stay up to kSkinnyMaxM rows.
bool few_rows_up_to(long M, long N, long K, long batch, bool parts_or_whole) {
    // (17 to 32 rows read four times the activations that 8 do, for each block of weight rows: over a long contraction, and where the weight rows are few, 32 x 64 and
    // 64 x 64 tiles in parts are ahead.  This kernel and those, us: 32 x 4096 x 14336 32.4 / 26.5, 24 x 2048 x 7168 13.5 / 12.1, 20 x 320 x 9600 13.4 / 10.3,
    // 32 x 1024 x 14336 24.3 / 14.0, 17 x 64 x 14336 17.4 / 10.1; 32 x 1024 x 4096 8.8 / 9.0, 32 x 7168 x 2048 9.9 / 11.7, 17 x 8192 x 6400 24.2 / 25.9,
    // 20 x 14336 x 8192 46.6 / 53.3; 16 x 4096 x 14336 26.0 / 25.9, 16 x 2048 x 7168 11.4 / 11.8)
    if (M <= kFewRowsM) return M <= 16 || K < 6144 || N > 4096 || batch > 1 || !parts_or_whole;
    return M <= kSkinnyMaxM && (!parts_or_whole || (K <= 64 && M * N * batch <= 1 << 19) || (M <= 64 && M * K <= 36000 && N * batch <= 4096));
}

// Few output columns and many rows: the few-row kernels with the operands in each other's place.  Up to
// 32 columns (every workgroup re-reads the short operand, and from 48 rows of it on the tile kernel with
// the contraction in parts is faster: M = 16384, N = 128, K = 4096 80 us this way).
bool swapped_route(long M, long N, long batch) {
    return N <= 32 && M > kSkinnyMaxM && batch <= 65535 && (M + 15) / 16 <= 0x7fffffffL;
}

// Parts of the contraction for the 128 x 128 tile kernel with a workspace (0 = it does not apply): 49 to
// 128 rows and too few tiles to fill the chip; about 384 workgroups in all (measured 128 ... 1024: fewer
// leave CUs idle, more only add partial tiles for the finishing kernel to read), at least four k-tiles each.
// More rows than that with at most one tile per CU (a projection over 256 ... 1024 tokens: 64 ... 256
// tiles, each walking the whole contraction alone on its CU): the same, two parts from 193 tiles on.
int tile_splitk_plan(long M, long N, long K, long batch, long* k_per_split) {
    if (M <= 48 || K % 64 != 0 || N < 128) return 0;
    if (M <= kSkinnyMaxM && few_rows_by_tiles(M, N, batch)) return 0;
    const long m_tiles = (M + gemm::kBM - 1) / gemm::kBM;
    const long tiles = m_tiles * ((N + gemm::kBN - 1) / gemm::kBN) * batch;
    if (m_tiles > 1 && tiles > 256) return 0;
    const long k_tiles = K / 64;
    long splits = (m_tiles > 1 && tiles > 192) ? 2 : (384 + tiles - 1) / tiles;
    if (splits > k_tiles / 4) splits = k_tiles / 4;
    if (splits < 2) return 0;
    const long per = (k_tiles + splits - 1) / splits;
    splits = (k_tiles + per - 1) / per;
    if (splits < 2 || tiles * splits > 0x7fffffffL) return 0;
    *k_per_split = per * 64;
    return static_cast<int>(splits);
}

// Splits of the contraction for the workspace kernel (0 = it does not apply): enough workgroups to
// fill the chip twice, at least two slabs each.
int splitk_plan(long M, long N, long K, long batch, int* pieces_per_split) {
    if (M < 32 || M > kSkinnyMaxM || K % 64 != 0 || N < 512) return 0;   // up to 16 rows the activations are no load
    if (few_rows_by_tiles(M, N, batch)) return 0;
    const long pieces = K / 64;
    const long groups = (N + 127) / 128 * batch;
    long splits = (512 + groups - 1) / groups;
    if (splits > pieces / 8) splits = pieces / 8;
    if (splits < 2) return 0;
    long per = (pieces + splits - 1) / splits;
    per = (per + 3) / 4 * 4;                                  // whole slabs
    splits = (pieces + per - 1) / per;
    if (splits < 2 || (N + 127) / 128 > 65535) return 0;
    *pieces_per_split = static_cast<int>(per);
    return static_cast<int>(splits);
}

// ---- any float dtype, any contraction size, any alignment: the product for what the MFMA kernels
// do not take (fp32 / fp64 tensors, K not a multiple of 64, rows that are not 16-byte aligned), so
// that no GEMM leaves the device.  64 x 64 outputs per workgroup, 4 x 4 per thread, k-tiles of 16
// through LDS; fp32 accumulation (fp64 for fp64 tensors) and one rounding, as ATen-CPU does.
template <typename T>
__global__ __launch_bounds__(256) void gemm_nt_any_kernel(const typename Elem<T>::store_t* __restrict__ a,
                                                          const typename Elem<T>::store_t* __restrict__ b,
                                                          const typename Elem<T>::store_t* __restrict__ add,
                                                          typename Elem<T>::store_t* __restrict__ c, const DenseParams p) {
    using El = Elem<T>;
    using Acc = typename std::conditional<sizeof(typename El::store_t) == 8, double, float>::type;
    constexpr int BM = 64, BN = 64, BKK = 16;
    __shared__ Acc as[BKK][BM + 1], bs[BKK][BN + 1];
    const long bidx = blockIdx.z;
    const auto* A = a + bidx * p.sa;
    const auto* B = b + bidx * p.sb;
    const long row0 = static_cast<long>(blockIdx.y) * BM, col0 = static_cast<long>(blockIdx.x) * BN;
    const int tx = threadIdx.x & 15, ty = threadIdx.x >> 4;
    const int lrow = threadIdx.x >> 2, lk = (threadIdx.x & 3) * 4;     // staging: 64 rows x 16 k, 4 k per thread
    auto widen = [](typename El::store_t v) -> Acc {
        if constexpr (sizeof(typename El::store_t) == 8) return El::to_f64(v);
        else return El::to_f32(v);
    };
    Acc acc[4][4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = 0;
    for (long k0 = 0; k0 < p.K; k0 += BKK) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const long k = k0 + lk + e;
            const long ar = row0 + lrow, br = col0 + lrow;
            as[lk + e][lrow] = (ar < p.M && k < p.K) ? widen(A[ar * p.lda + k]) : Acc(0);
            bs[lk + e][lrow] = (br < p.N && k < p.K) ? widen(B[br * p.ldb + k]) : Acc(0);
        }
        __syncthreads();
#pragma unroll
        for (int kk = 0; kk < BKK; ++kk) {
            Acc av[4], bv[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) av[i] = as[kk][ty * 4 + i];
#pragma unroll
            for (int j = 0; j < 4; ++j) bv[j] = bs[kk][tx * 4 + j];
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j) acc[i][j] += av[i] * bv[j];
        }
        __syncthreads();
    }
    auto* C = c + bidx * p.sc;
    const auto* ADD = add ? add + bidx * p.sadd : nullptr;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const long row = row0 + ty * 4 + i;
        if (row >= p.M) continue;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const long col = col0 + tx * 4 + j;
            if (col >= p.N) continue;
            if constexpr (sizeof(typename El::store_t) == 8) {
                double v = static_cast<double>(p.alpha64) * acc[i][j];
                if (ADD) v += p.beta64 * El::to_f64(ADD[row * p.ld_add + col]);
                C[row * p.ldc + col] = El::from_f64(v);
            } else {
                float v = p.alpha * acc[i][j];
                if (ADD) v = fmaf(p.beta, El::to_f32(ADD[row * p.ld_add + col]), v);
                C[row * p.ldc + col] = El::from_f32(v);
            }
        }
    }
}

template <typename T>
int launch_any(const DenseParams& p, const void* a, const void* b, const void* add, void* c, long batch, hipStream_t s) {
    using S = typename Elem<T>::store_t;
    const long gx = (p.N + 63) / 64, gy = (p.M + 63) / 64;
    PARAS_REQUIRE(gx <= 0x7fffffffL && gy <= 65535 && batch <= 65535, "paras_gemm_nt: shape too large for the general kernel");
    hipLaunchKernelGGL((gemm_nt_any_kernel<T>), dim3(static_cast<unsigned>(gx), static_cast<unsigned>(gy), static_cast<unsigned>(batch)),
                       dim3(256), 0, s, static_cast<const S*>(a), static_cast<const S*>(b), static_cast<const S*>(add),
                       static_cast<S*>(c), p);
    PARAS_HIP_TRY(hipGetLastError());
    return PARAS_OK;
}

// How a product is carried out.
struct Route {
    enum Kind { Any, FewRows, FewRowsParts, FewColumns, Flex, F32 } kind = Any;
    int pieces = 0, splits = 0;          // FewRowsParts
    flex::Plan flex;
    f32::Plan f32;
    size_t workspace = 0;
};

flex::Problem flex_problem(const paras_gemm_args& g) {
    flex::Problem q{};
    q.a = static_cast<const std::uint16_t*>(g.a); q.b = static_cast<const std::uint16_t*>(g.b);
    q.add = static_cast<const std::uint16_t*>(g.addend); q.c = static_cast<std::uint16_t*>(g.c);
    q.M = g.M; q.N = g.N; q.K = g.K;
    q.lda = g.lda; q.ldb = g.ldb; q.ldc = g.ldc; q.ld_add = g.ld_add;
    q.sa = g.stride_a; q.sb = g.stride_b; q.sc = g.stride_c; q.sadd = g.stride_add; q.batch = g.batch;
    q.alpha = static_cast<float>(g.alpha); q.beta = static_cast<float>(g.beta);
    q.a_rows = g.a_rows != 0; q.b_rows = g.b_rows != 0;
    q.bf16 = g.dtype == PARAS_BF16;
    return q;
}
f32::Problem f32_problem(const paras_gemm_args& g, int causal_kind, long causal_first) {
    f32::Problem q{};
    q.a = static_cast<const float*>(g.a); q.b = static_cast<const float*>(g.b);
    q.add = static_cast<const float*>(g.addend); q.c = static_cast<float*>(g.c);
    q.M = g.M; q.N = g.N; q.K = g.K;
    q.lda = g.lda; q.ldb = g.ldb; q.ldc = g.ldc; q.ld_add = g.ld_add;
    q.sa = g.stride_a; q.sb = g.stride_b; q.sc = g.stride_c; q.sadd = g.stride_add; q.batch = g.batch;
    q.alpha = static_cast<float>(g.alpha); q.beta = static_cast<float>(g.beta);
    q.a_rows = g.a_rows != 0; q.b_rows = g.b_rows != 0;
    q.causal_kind = causal_kind; q.causal_first = causal_first;
    return q;
}

// `may_split`: the caller will bring the workspace the route asks for.  `nt_api`: the call came through
// paras_gemm_nt_ws, whose workspace function knows sizes only: the few-row forms and 128 x 128 tiles.
Route route_of(const paras_gemm_args& g, bool may_split, bool nt_api, int causal_kind, long causal_first) {
    Route r;
    if (g.dtype == PARAS_F32) {
        const auto q = f32_problem(g, causal_kind, causal_first);
        if (f32::takes(q)) {
            r.kind = Route::F32;
            r.f32 = f32::plan(q, may_split && !nt_api && causal_kind == 0);
            r.workspace = f32::workspace(q, r.f32);
        }
        return r;
    }
    if (g.dtype != PARAS_BF16 && g.dtype != PARAS_F16) return r;
    const auto q = flex_problem(g);
    if (!flex::takes(q)) return r;
    const bool nt64 = !g.a_rows && !g.b_rows && g.K % gemm::kBK == 0;
    if (nt64 && swapped_route(g.M, g.N, g.batch)) {
        r.kind = Route::FewColumns;
        return r;
    }
    r.kind = Route::Flex;
    if (nt_api) {
        if (may_split) {
            long kper = 0;
            const int parts = tile_splitk_plan(g.M, g.N, g.K, g.batch, &kper);
            if (parts >= 2) {
                r.flex.tile = flex::kTile128x128;
                r.flex.splits = parts;
                r.flex.k_per_split = kper;
                r.workspace = flex::workspace(q, r.flex);
                return r;
            }
            r.splits = splitk_plan(g.M, g.N, g.K, g.batch, &r.pieces);
        }
    }
    if (r.splits >= 2) {
        r.kind = Route::FewRowsParts;
        r.workspace = static_cast<size_t>(r.splits) * g.batch * g.M * g.N * sizeof(float);
        return r;
    }
    if (nt64 && few_rows_up_to(g.M, g.N, g.K, g.batch, may_split && !nt_api) && !few_rows_by_tiles(g.M, g.N, g.batch) && g.batch <= 65535) {
        r.kind = Route::FewRows;
        return r;
    }
    r.flex = flex::plan(q, may_split && !nt_api);
    r.workspace = flex::workspace(q, r.flex);
    return r;
}

int check_args(const paras_gemm_args& g) {
    PARAS_REQUIRE(g.M >= 0 && g.N >= 0 && g.K >= 0 && g.batch >= 0, "paras_gemm_nt: negative shape");
    if (g.M == 0 || g.N == 0 || g.batch == 0) return PARAS_OK;
    PARAS_REQUIRE(g.dtype == PARAS_BF16 || g.dtype == PARAS_F16 || g.dtype == PARAS_F32 || g.dtype == PARAS_F64,
                  "paras_gemm_nt: unknown dtype");
    PARAS_REQUIRE(g.c && (g.K == 0 || (g.a && g.b)), "paras_gemm_nt: null pointer");   // an empty contraction has no operands to read
    PARAS_REQUIRE(g.lda >= (g.a_rows ? g.M : g.K) && g.ldb >= (g.b_rows ? g.N : g.K) && g.ldc >= g.N &&
                      (g.addend == nullptr || g.ld_add == 0 || g.ld_add >= g.N),
                  "paras_gemm_nt: a leading dimension is smaller than its row");
    return PARAS_OK;
}

// Where a product's partial sums go: memory that the caller has, or a way to ask it for some.
struct Scratch {
    void* p = nullptr;
    size_t bytes = 0;
    paras_scratch_fn ask = nullptr;
    void* ctx = nullptr;
};

// The route is found once.  It is the one that paras_gemm_workspace answers for, and only where it wants more than the caller has
// another one is taken.
int run(const paras_gemm_args& g, const Scratch& scratch, void* stream, bool nt_api, int causal_kind, long causal_first) {
    int rc = check_args(g);
    if (rc != PARAS_OK || g.M == 0 || g.N == 0 || g.batch == 0) return rc;
    hipStream_t s = nullptr;
    rc = resolve_stream(stream, &s);
    if (rc != PARAS_OK) return rc;
    Route r = route_of(g, /*may_split=*/true, nt_api, causal_kind, causal_first);
    void* workspace = scratch.p;
    if (r.workspace > 0) {
        if (scratch.ask != nullptr) {
            workspace = scratch.ask(scratch.ctx, r.workspace);
            PARAS_REQUIRE(workspace != nullptr && (reinterpret_cast<uintptr_t>(workspace) & 15) == 0,
                          "paras_gemm_scratch: no memory for %zu bytes on a 16-byte boundary", r.workspace);
        } else if (workspace == nullptr || (reinterpret_cast<uintptr_t>(workspace) & 15) != 0 || r.workspace > scratch.bytes) {
            r = route_of(g, false, nt_api, causal_kind, causal_first);
        }
    }
    if (r.kind == Route::F32) return f32::launch(f32_problem(g, causal_kind, causal_first), r.f32, workspace, s);
    if (r.kind == Route::Flex) return flex::launch(flex_problem(g), r.flex, workspace, s);
    PARAS_REQUIRE(!g.a_rows && !g.b_rows, "paras_gemm: these sizes or alignments need operands that are contiguous along the contraction");
    DenseParams p{};
    p.a = static_cast<const std::uint16_t*>(g.a);
    p.b = static_cast<const std::uint16_t*>(g.b);
    p.add = static_cast<const std::uint16_t*>(g.addend);
    p.c = static_cast<std::uint16_t*>(g.c);
    p.M = g.M; p.N = g.N; p.K = g.K;
    p.lda = g.lda; p.ldb = g.ldb; p.ldc = g.ldc; p.ld_add = g.ld_add;
    p.sa = g.stride_a; p.sb = g.stride_b; p.sc = g.stride_c; p.sadd = g.stride_add;
    p.alpha = static_cast<float>(g.alpha); p.beta = static_cast<float>(g.beta);
    p.alpha64 = g.alpha; p.beta64 = g.beta;
    const bool bf = g.dtype == PARAS_BF16;
    if (r.kind == Route::FewColumns) {
        // Few output columns and many rows (a router's logits: tokens x experts): the product is bound by
        // reading a once, which 128 x 128 tiles on N / 128 of the CUs do badly (M = 16384, K = 4096:
        // N = 8 in 78 us, N = 128 in 78 us).  The few-row kernels stream a long operand with every CU and
        // keep the short one in registers, so the operands change places and the results are stored
        // transposed.
        DenseParams q = p;
        q.a = p.b; q.b = p.a;
        q.M = g.N; q.N = g.M;
        q.lda = g.ldb; q.ldb = g.lda;
        q.sa = g.stride_b; q.sb = g.stride_a;
        q.swapped = 1;
        if (bf) launch_skinny<bf16_t>(q, g.batch, s);
        else    launch_skinny<f16_t>(q, g.batch, s);
    } else if (r.kind == Route::FewRowsParts) {
        const dim3 grid(static_cast<unsigned>(r.splits), static_cast<unsigned>((g.N + 127) / 128), static_cast<unsigned>(g.batch));
        const int mb = static_cast<int>((g.M + 15) / 16);
        float* part = static_cast<float*>(workspace);
        if (mb <= 2)      { if (bf) hipLaunchKernelGGL((skinny_splitk_kernel<bf16_t, 2>), grid, dim3(512), 0, s, p, part, r.pieces);
                            else    hipLaunchKernelGGL((skinny_splitk_kernel<f16_t, 2>), grid, dim3(512), 0, s, p, part, r.pieces); }
        else if (mb <= 4) { if (bf) hipLaunchKernelGGL((skinny_splitk_kernel<bf16_t, 4>), grid, dim3(512), 0, s, p, part, r.pieces);
                            else    hipLaunchKernelGGL((skinny_splitk_kernel<f16_t, 4>), grid, dim3(512), 0, s, p, part, r.pieces); }
        else              { if (bf) hipLaunchKernelGGL((skinny_splitk_kernel<bf16_t, 8>), grid, dim3(512), 0, s, p, part, r.pieces);
                            else    hipLaunchKernelGGL((skinny_splitk_kernel<f16_t, 8>), grid, dim3(512), 0, s, p, part, r.pieces); }
        PARAS_HIP_TRY(hipGetLastError());
        const dim3 fgrid(static_cast<unsigned>((g.M * g.N + 255) / 256), static_cast<unsigned>(g.batch));
        if (bf) hipLaunchKernelGGL((skinny_splitk_finish_kernel<bf16_t>), fgrid, dim3(256), 0, s, p, part, r.splits);
        else    hipLaunchKernelGGL((skinny_splitk_finish_kernel<f16_t>), fgrid, dim3(256), 0, s, p, part, r.splits);
    } else if (r.kind == Route::FewRows) {
        if (bf) launch_skinny<bf16_t>(p, g.batch, s);
        else    launch_skinny<f16_t>(p, g.batch, s);
    } else {
        switch (g.dtype) {
            case PARAS_F32:  return launch_any<float>(p, g.a, g.b, g.addend, g.c, g.batch, s);
            case PARAS_F64:  return launch_any<double>(p, g.a, g.b, g.addend, g.c, g.batch, s);
            case PARAS_BF16: return launch_any<bf16_t>(p, g.a, g.b, g.addend, g.c, g.batch, s);
            default:         return launch_any<f16_t>(p, g.a, g.b, g.addend, g.c, g.batch, s);
        }
    }
    PARAS_HIP_TRY(hipGetLastError());
    return PARAS_OK;
}

}  // namespace

// paras_gemm_nt_ws with two hints for causal attention (Problem in gemm_f32_host.h); also declared in sdpa_internal.h
int gemm_nt_causal(const void* a, const void* b, const void* addend, void* c, int64_t M, int64_t N, int64_t K,
                   int64_t lda, int64_t ldb, int64_t ldc, int64_t ld_add, int64_t batch, int64_t stride_a,
                   int64_t stride_b, int64_t stride_c, int64_t stride_add, double alpha, double beta, int dtype,
                   void* workspace, size_t workspace_bytes, void* stream, int causal_kind, long causal_first) {
    paras_gemm_args g{};
    g.a = a; g.b = b; g.addend = addend; g.c = c;
    g.M = M; g.N = N; g.K = K;
    g.lda = lda; g.ldb = ldb; g.ldc = ldc; g.ld_add = ld_add;
    g.batch = batch; g.stride_a = stride_a; g.stride_b = stride_b; g.stride_c = stride_c; g.stride_add = stride_add;
    g.alpha = alpha; g.beta = beta; g.dtype = dtype;
    return run(g, {workspace, workspace_bytes}, stream, /*nt_api=*/true, causal_kind, causal_first);
}
}  // namespace paras

extern "C" {

size_t paras_gemm_nt_workspace(int64_t M, int64_t N, int64_t K, int64_t batch, int dtype) {
    using namespace paras;
    if (M <= 0 || N <= 0 || K <= 0 || batch <= 0 || (dtype != PARAS_BF16 && dtype != PARAS_F16)) return 0;
    int per = 0;
    long kper = 0;
    if (K % gemm::kBK == 0 && swapped_route(M, N, batch)) return 0;
    int splits = tile_splitk_plan(M, N, K, batch, &kper);
    if (splits == 0) splits = splitk_plan(M, N, K, batch, &per);
    return static_cast<size_t>(splits) * static_cast<size_t>(batch) * static_cast<size_t>(M) * static_cast<size_t>(N) * sizeof(float);
}

int paras_gemm_nt(const void* a, const void* b, const void* addend, void* c, int64_t M, int64_t N, int64_t K,
                  int64_t lda, int64_t ldb, int64_t ldc, int64_t ld_add, int64_t batch, int64_t stride_a,
                  int64_t stride_b, int64_t stride_c, int64_t stride_add, double alpha, double beta, int dtype,
                  void* stream) {
    return paras_gemm_nt_ws(a, b, addend, c, M, N, K, lda, ldb, ldc, ld_add, batch, stride_a, stride_b, stride_c, stride_add,
                            alpha, beta, dtype, nullptr, 0, stream);
}

int paras_gemm_nt_ws(const void* a, const void* b, const void* addend, void* c, int64_t M, int64_t N, int64_t K,
                     int64_t lda, int64_t ldb, int64_t ldc, int64_t ld_add, int64_t batch, int64_t stride_a,
                     int64_t stride_b, int64_t stride_c, int64_t stride_add, double alpha, double beta, int dtype,
                     void* workspace, size_t workspace_bytes, void* stream) {
    return paras::gemm_nt_causal(a, b, addend, c, M, N, K, lda, ldb, ldc, ld_add, batch, stride_a, stride_b, stride_c, stride_add, alpha, beta,
                                 dtype, workspace, workspace_bytes, stream, 0, 0);
}

size_t paras_gemm_workspace(const paras_gemm_args* args) {
    using namespace paras;
    if (args == nullptr || args->M <= 0 || args->N <= 0 || args->K <= 0 || args->batch <= 0) return 0;
    return route_of(*args, true, false, 0, 0).workspace;
}

int paras_gemm(const paras_gemm_args* args, void* workspace, size_t workspace_bytes, void* stream) {
    PARAS_REQUIRE(args != nullptr, "paras_gemm: null argument block");
    return paras::run(*args, {workspace, workspace_bytes}, stream, /*nt_api=*/false, 0, 0);
}

int paras_gemm_scratch(const paras_gemm_args* args, paras_scratch_fn scratch, void* ctx, void* stream) {
    PARAS_REQUIRE(args != nullptr && scratch != nullptr, "paras_gemm_scratch: null argument");
    return paras::run(*args, {nullptr, 0, scratch, ctx}, stream, /*nt_api=*/false, 0, 0);
}

}  // extern "C"
