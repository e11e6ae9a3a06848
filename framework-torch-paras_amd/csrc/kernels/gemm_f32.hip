// fp32 products on the matrix cores, either operand either way round:
//   C = alpha op(A) op(B)^T + beta addend
// v_mfma_f32_16x16x4_f32 multiplies and accumulates in full fp32.  A workgroup is four waves, 2 x 2, a
// wave computes MI x NJ blocks of 16 x 16: tiles of 32 MI x 32 NJ, from 128 x 128 (bound by the matrix
// cores: 157 TFLOP/s published) down to 32 x 64 for products too small to fill the chip otherwise, and
// the contraction is split over workgroups where there are still too few tiles.  Before, small products
// ran on scalar FMAs in 64 x 64 tiles (12 x 384 x 256: 34 us against the 5 us of a launch and its
// latency) and a transposed operand was copied first.
//
// k-tile 32: global -> registers (the next tile in flight during the MFMAs) -> LDS as [k][row], two
// stages, one barrier per tile.  A fragment is one word per lane (row lane % 16, step lane / 16), so an
// operand that is contiguous along its rows is stored as it lies and one that is contiguous along the
// contraction is turned by its stores: eight lanes hold eight k-quads of a row, and with a row stride
// of rows + 2 words their stores fall 8 banks apart.  (The reads then overlap two ways, which costs
// nothing: 2 LDS cycles per 32-cycle MFMA.)  Buffer loads against the operand's extent return zeros
// past its end and need no alignment beyond the element's.
#include <hip/hip_runtime.h>

#include "core/device_context.h"
#include "core/device_math.h"
#include "core/status.h"
#include "kernels/gemm_f32_host.h"
#include "paras_hip.h"

namespace paras {
namespace f32 {
namespace {

constexpr int kThreads = 256;
constexpr int kBK = 32;
constexpr std::uint32_t kOutOfRange = 0xF0000000u;
constexpr long kMaxExtent = 0xE0000000L;

struct Params {
    const float* a;
    const float* b;
    const float* add;
    float* c;
    long M, N, K;
    long lda, ldb, ldc, ld_add;
    long sa, sb, sc, sadd;
    int  m_tiles, n_tiles, splits;
    long k_per_split;
    float* partial;             // splits > 1: [batch][split][M][N]
    float alpha, beta;
    int  causal_kind;           // for causal attention: 1 = the product is a score matrix of which row r only needs columns
                                // <= r + causal_first (tiles wholly beyond are left unwritten); 2 = a is such a matrix after
                                // its softmax (zeros beyond), so a row tile contracts as far as its last row needs; 0 = neither
    long causal_first;
};

template <int W, bool R> struct Operand {
    static constexpr int kRows = 32 * W;
    static constexpr int kLd = kRows + 2;
    const char* base;
    long left, step;
    std::uint32_t off[W];
    int kq4;                     // contraction steps: first of this thread's quads within a tile
    int kcount;

    __device__ __forceinline__ void init(const float* p, long ld, long rows, long row0, long k_first, long k_count) {
        const int tid = threadIdx.x;
        kcount = static_cast<int>(k_count);
        kq4 = (tid & 7) * 4;
        if constexpr (R) {
            base = reinterpret_cast<const char*>(p + k_first * ld + row0);
            left = ((k_count - 1) * ld + (rows - row0)) * 4;
            step = kBK * ld * 4;
#pragma unroll
            for (int i = 0; i < W; ++i) {
                const int c = tid + i * kThreads;
                off[i] = static_cast<std::uint32_t>((c / (8 * W)) * ld * 4 + (c % (8 * W)) * 16);
            }
        } else {
            base = reinterpret_cast<const char*>(p + row0 * ld + k_first);
            left = ((rows - row0 - 1) * ld + k_count) * 4;
            step = kBK * 4;
#pragma unroll
            for (int i = 0; i < W; ++i) off[i] = static_cast<std::uint32_t>(((tid >> 3) + i * 32) * ld * 4 + kq4 * 4);
        }
    }
    __device__ __forceinline__ void load(int kt, u32x4 (&st)[W]) const {
        const long l = left - kt * step;
        const long n = l < 0 ? 0 : (l > kMaxExtent ? kMaxExtent : l);
        const auto r = __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(base + kt * step), 0, static_cast<int>(static_cast<std::uint32_t>(n)), 0x00020000);
#pragma unroll
        for (int i = 0; i < W; ++i) st[i] = __builtin_amdgcn_raw_buffer_load_b128(r, static_cast<int>(off[i]), 0, 0);
        if constexpr (!R) {
            if ((kt + 1) * kBK > kcount) {              // the last tile, cut short: what lies past K is the next row's
#pragma unroll
                for (int i = 0; i < W; ++i)
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        if (kt * kBK + kq4 + e >= kcount) st[i][e] = 0;
            }
        }
    }
    __device__ __forceinline__ void store(float* tile, const u32x4 (&st)[W]) const {
#pragma unroll
        for (int i = 0; i < W; ++i) {
            const int c = static_cast<int>(threadIdx.x) + i * kThreads;
            if constexpr (R) {
                float* q = tile + (c / (8 * W)) * kLd + (c % (8 * W)) * 4;
                *reinterpret_cast<u32x2*>(q) = u32x2{st[i][0], st[i][1]};
                *reinterpret_cast<u32x2*>(q + 2) = u32x2{st[i][2], st[i][3]};
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const std::uint32_t bits = st[i][e];        // (a copy: a bit cast of the element itself reads element 0)
                    tile[(kq4 + e) * kLd + (c >> 3)] = __builtin_bit_cast(float, bits);
                }
            }
        }
    }
};

template <int MI, int NJ, bool AR, bool BR>
__global__ __launch_bounds__(kThreads, (MI * NJ >= 16 ? 2 : 3)) void gemm_f32_kernel(const Params p) {
    using OA = Operand<MI, AR>;
    using OB = Operand<NJ, BR>;
    __shared__ __attribute__((aligned(16))) float as[2][kBK * OA::kLd];
    __shared__ __attribute__((aligned(16))) float bs[2][kBK * OB::kLd];
    // column tiles innermost, parts of the contraction outermost
    const unsigned r = blockIdx.x / static_cast<unsigned>(p.n_tiles), nt = blockIdx.x - r * p.n_tiles;
    const unsigned split_v = r / static_cast<unsigned>(p.m_tiles);
    const int split = __builtin_amdgcn_readfirstlane(static_cast<int>(split_v));
    const long batch = blockIdx.y;
    const long row0 = static_cast<long>(__builtin_amdgcn_readfirstlane(static_cast<int>(r - split_v * p.m_tiles))) * (32 * MI);
    const long col0 = static_cast<long>(__builtin_amdgcn_readfirstlane(static_cast<int>(nt))) * (32 * NJ);
    if (p.causal_kind == 1 && col0 > row0 + (32 * MI - 1) + p.causal_first) return;
    long K = p.K;
    if (p.causal_kind == 2) {
        const long upto = row0 + 32 * MI + p.causal_first;
        if (upto < K) K = upto;
    }
    const long k_first = static_cast<long>(split) * p.k_per_split;
    const long k_count = K - k_first < p.k_per_split ? K - k_first : p.k_per_split;     // (one part wherever K is cut)
    OA oa;
    OB ob;
    oa.init(p.a + batch * p.sa, p.lda, p.M, row0, k_first, k_count);
    ob.init(p.b + batch * p.sb, p.ldb, p.N, col0, k_first, k_count);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int l16 = lane & 15, kq = lane >> 4;
    const int a_at = kq * OA::kLd + (wave >> 1) * 16 * MI + l16, b_at = kq * OB::kLd + (wave & 1) * 16 * NJ + l16;
    float4_t acc[MI][NJ];
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j) acc[i][j] = float4_t{0.f, 0.f, 0.f, 0.f};
    u32x4 a_st[MI], b_st[NJ];
    const int k_tiles = static_cast<int>((k_count + kBK - 1) / kBK);
    oa.load(0, a_st);
    ob.load(0, b_st);
    oa.store(as[0], a_st);
    ob.store(bs[0], b_st);
    __syncthreads();
    for (int kt = 0; kt < k_tiles; ++kt) {
        const int cur = kt & 1;
        const bool more = kt + 1 < k_tiles;
        if (more) {
            oa.load(kt + 1, a_st);
            ob.load(kt + 1, b_st);
        }
#pragma unroll
        for (int kk = 0; kk < kBK; kk += 4) {
            float af[MI], bf[NJ];
#pragma unroll
            for (int i = 0; i < MI; ++i) af[i] = as[cur][a_at + kk * OA::kLd + i * 16];
#pragma unroll
            for (int j = 0; j < NJ; ++j) bf[j] = bs[cur][b_at + kk * OB::kLd + j * 16];
#pragma unroll
            for (int j = 0; j < NJ; ++j)
#pragma unroll
                for (int i = 0; i < MI; ++i) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(bf[j], af[i], acc[i][j], 0, 0, 0);
        }
        if (more) {
            oa.store(as[cur ^ 1], a_st);      // the other stage: last read before the previous barrier
            ob.store(bs[cur ^ 1], b_st);
        }
        __syncthreads();
    }
    // the B fragment is the first operand: lane (l16, kq) of block (i, j) holds row i*16 + l16, columns j*16 + 4*kq .. + 3
    const bool part = p.splits > 1;
    float* C = part ? p.partial + (batch * p.splits + split) * (p.M * p.N) : p.c + batch * p.sc;
    const long ldc = part ? p.N : p.ldc;
    const float* ADD = !part && p.add ? p.add + batch * p.sadd : nullptr;
    const float alpha = part ? 1.0f : p.alpha;
    const bool vec = ldc % 4 == 0 && (reinterpret_cast<uintptr_t>(C) & 15) == 0;
#pragma unroll
    for (int i = 0; i < MI; ++i) {
        const long row = row0 + (wave >> 1) * 16 * MI + i * 16 + l16;
        if (row >= p.M) continue;
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
            const long col = col0 + (wave & 1) * 16 * NJ + j * 16 + 4 * kq;
            float4_t v;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                v[r] = alpha * acc[i][j][r];
                if (ADD && col + r < p.N) v[r] = fmaf(p.beta, ADD[row * p.ld_add + col + r], v[r]);
            }
            if (vec && col + 3 < p.N) {
                *reinterpret_cast<float4_t*>(C + row * ldc + col) = v;
            } else {
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    if (col + r < p.N) C[row * ldc + col + r] = v[r];
            }
        }
    }
}

// adds the parts in order and applies the epilogue
__global__ __launch_bounds__(256) void gemm_f32_finish_kernel(const Params p) {
    const long mn = p.M * p.N, i = static_cast<long>(blockIdx.x) * 256 + threadIdx.x;
    if (i >= mn) return;
    const long batch = blockIdx.y;
    const float* src = p.partial + batch * p.splits * mn + i;
    float t = 0.f;
    for (int sp = 0; sp < p.splits; ++sp) t += src[sp * mn];
    const long row = i / p.N, col = i - row * p.N;
    float v = p.alpha * t;
    if (p.add) v = fmaf(p.beta, (p.add + batch * p.sadd)[row * p.ld_add + col], v);
    (p.c + batch * p.sc)[row * p.ldc + col] = v;
}

template <int MI, int NJ>
void launch_tile(bool ar, bool br, const Params& p, dim3 g, hipStream_t s) {
    if (ar)      hipLaunchKernelGGL((gemm_f32_kernel<MI, NJ, true, true>), g, dim3(kThreads), 0, s, p);
    else if (br) hipLaunchKernelGGL((gemm_f32_kernel<MI, NJ, false, true>), g, dim3(kThreads), 0, s, p);
    else         hipLaunchKernelGGL((gemm_f32_kernel<MI, NJ, false, false>), g, dim3(kThreads), 0, s, p);
}

// Per tile shape: rows, columns, workgroups a CU holds at once.
struct Tile { int m, n, per_cu; };
constexpr Tile kTiles[] = {{128, 128, 2}, {64, 128, 3}, {64, 64, 4}, {32, 64, 4}};
constexpr int kTileCount = 4;

}  // namespace

bool takes(const Problem& q) {
    if (q.a_rows && !q.b_rows) return false;
    const long ld_max = 1L << 21;
    return q.K > 0 && q.K < (1L << 30) && q.lda <= ld_max && q.ldb <= ld_max && q.batch <= 65535 && q.M < (1L << 30) && q.N < (1L << 30) &&
           ((q.M + 31) / 32) * ((q.N + 63) / 64) < (1L << 31);
}

// The least estimated time over tile shapes and numbers of parts: rounds of workgroups times the time of a
// tile's contraction.  A k-tile of 32 steps is 8 MI NJ MFMAs of 32 cycles per wave (MI NJ / 8 us) when the CU
// has work for its matrix cores, and no less than the latency of a load and a barrier otherwise.
Plan plan(const Problem& q, bool may_split) {
    Plan best;
    double best_us = 1e30;
    const long k_tiles = (q.K + kBK - 1) / kBK;
    for (int t = 0; t < kTileCount; ++t) {
        const Tile& tl = kTiles[t];
        const double step = tl.m / 32 * (tl.n / 32) * 0.125;
        const long tiles = (q.M + tl.m - 1) / tl.m * ((q.N + tl.n - 1) / tl.n) * q.batch;
        for (int s = 1; s <= (may_split ? 32 : 1) && s * 2 <= (k_tiles < 2 ? 2 : k_tiles); s = s < 4 ? s + 1 : s + s / 2) {
            const long per = (k_tiles + s - 1) / s, parts = (k_tiles + per - 1) / per;
            const long wgs = tiles * parts, slots = 256L * tl.per_cu, full = wgs / slots, rest = (wgs - full * slots + 255) / 256;
            auto round = [&](long n) { const double c = step * n; return per * (c > 0.75 ? c : 0.75); };
            double us = full * round(tl.per_cu) + (rest > 0 ? round(rest) : 0.0) + 3.0;
            if (parts > 1) us += 2.5 + static_cast<double>(q.M) * q.N * q.batch * (8.0 * parts + 4.0) / 6e6;
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

size_t workspace(const Problem& q, const Plan& pl) {
    return pl.splits > 1 ? static_cast<size_t>(pl.splits) * q.batch * q.M * q.N * sizeof(float) : 0;
}

int launch(const Problem& q, const Plan& pl, void* ws, hipStream_t s) {
    Params p{};
    p.a = q.a; p.b = q.b; p.add = q.add; p.c = q.c;
    p.M = q.M; p.N = q.N; p.K = q.K;
    p.lda = q.lda; p.ldb = q.ldb; p.ldc = q.ldc; p.ld_add = q.ld_add;
    p.sa = q.sa; p.sb = q.sb; p.sc = q.sc; p.sadd = q.sadd;
    p.alpha = q.alpha; p.beta = q.beta;
    p.causal_kind = q.causal_kind; p.causal_first = q.causal_first;
    const Tile& t = kTiles[pl.tile];
    p.n_tiles = static_cast<int>((q.N + t.n - 1) / t.n);
    p.splits = pl.splits;
    p.k_per_split = pl.k_per_split;
    p.partial = static_cast<float*>(ws);
    p.m_tiles = static_cast<int>((q.M + t.m - 1) / t.m);
    const dim3 g(static_cast<unsigned>(p.n_tiles) * static_cast<unsigned>(p.m_tiles) * static_cast<unsigned>(pl.splits), static_cast<unsigned>(q.batch));
    switch (pl.tile) {
        case 0: launch_tile<4, 4>(q.a_rows, q.b_rows, p, g, s); break;
        case 1: launch_tile<2, 4>(q.a_rows, q.b_rows, p, g, s); break;
        case 2: launch_tile<2, 2>(q.a_rows, q.b_rows, p, g, s); break;
        default: launch_tile<1, 2>(q.a_rows, q.b_rows, p, g, s); break;
    }
    PARAS_HIP_TRY(hipGetLastError());
    if (pl.splits > 1) {
        hipLaunchKernelGGL(gemm_f32_finish_kernel, dim3(static_cast<unsigned>((q.M * q.N + 255) / 256), static_cast<unsigned>(q.batch)), dim3(256), 0, s, p);
        PARAS_HIP_TRY(hipGetLastError());
    }
    return PARAS_OK;
}

}  // namespace f32
}  // namespace paras
