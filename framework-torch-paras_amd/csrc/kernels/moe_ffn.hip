// MoE grouped expert FFN for gfx950: two grouped GEMMs on bf16/fp16 MFMA with
// fp32 accumulation, and the weighted combine.
//
//   GEMM 1   h[p, :] = T( silu(T(xp W_gate[e]^T)) * T(xp W_up[e]^T) )
//            xp = x[order[p] / k] is gathered inside the A-tile load (no
//            permuted copy of x is ever written); gate and up columns of the
//            same tile are accumulated side by side and the SwiGLU runs in
//            the epilogue on the values already rounded to T, as the composed
//            reference would see them (mm -> T, paras::swiglu -> T).
//   GEMM 2   y[p, :] = T( h[p, :] W_down[e]^T )
//   combine  out[t] = T( sum_slot T( y[inv_order[t*k+slot]] * T(topw[t][slot]) ) )
//
// Both products are "NT": A rows and weight rows are contiguous along the
// contraction dim, which is exactly the 8-element-per-lane operand layout of
// v_mfma_f32_32x32x16, so neither operand needs a transpose.
//
// Tiling: 32 to 256 routed rows x 64 to 256 weight rows (gate and up rows of the same columns for GEMM 1), k-tile 64, four
// waves on v_mfma_f32_16x16x32 with loads straight to LDS (gemm_flex.h; grouped_tile_kernel, grouped_gemm_direct_kernel), the
// tile chosen by an estimate (grouped_tiles); few rows per expert on kernels that stream the weights (grouped_few_rows_kernel); an x
// beyond a 32-bit byte offset on register-staged 256-row tiles (gemm_tile.h; grouped_gemm_kernel).  Rows of one
// expert are contiguous in the routed order; m-tiles never straddle experts (the grid is sized for the
// worst case and surplus workgroups exit).
#include <hip/hip_runtime.h>
#include <cstdlib>
#include <type_traits>

#include "core/device_context.h"
#include "core/device_math.h"
#include "core/status.h"
#include "kernels/gemm_flex.h"
#include "kernels/gemm_tile.h"
#include "kernels/moe_forms.h"
#include "kernels/stream_rows.h"
#include "kernels/swiglu_math.h"

namespace paras {
namespace {

using namespace gemm;

struct FfnGemmParams {
    const std::uint16_t* a;     // x [T, K] (gathered) or h [R, K]
    const std::uint16_t* b;     // weights of column group 0, [E, Nw, K]
    const std::uint16_t* b2;    // weights of column group 1 (same layout)
    std::uint16_t* c;           // [R, N]
    const long* order;          // gather index (routed row -> flat (token, slot)); null = direct rows
    const long* offsets;        // [E+1]
    long a_bytes;               // extent of a (few-row and direct kernels)
    long K, N, Nw, R;           // contraction, output columns, weight rows per expert, routed rows
    int E, k;
    int mt_total;               // upper bound on m-tiles
    int n_units;                // column units (128 output columns for GEMM 1, 256 for GEMM 2)
    int ngt;                    // column units an XCD sweeps together (register-staged tiles); 256 x 256 tiles: 1 = dealt one by one
    unsigned div_m;             // flat (token, slot) index / k as a multiplication: (x * div_m) >> div_s
    int div_s;                  // for every x < 2^30 (a 64-bit division per gathered row is ~150 instructions)
};

// Multiplier and shift with floor(x / d) == (x * m) >> s for all 0 <= x < 2^30, 1 <= d < 2^30:
// s = 30 + ceil(log2 d), m = ceil(2^s / d) < 2^31; the error x * (m d - 2^s) stays below 2^s.
inline void division_by(unsigned d, unsigned* m, int* s) {
    int lg = 0;
    while ((1ull << lg) < d) ++lg;
    *s = 30 + lg;
    *m = static_cast<unsigned>(((1ull << *s) + d - 1) / d);
}

// ---- register-staged 256-row tiles, for an x whose rows are out of a 32-bit byte offset's reach (from 3.76 GB; also
// PARAS_GEMM_EIGHT_WAVES).  8 experts, top-2, H 4096: 8192 tokens, I 14336 5149 us, on the other tiles 4956; 65536 tokens, I 1792
// 5834 and 5620; H 2048, I 4096, 1024 tokens 206 and 200.
template <typename T, bool kSwiglu>
__global__ __launch_bounds__(wide::kThreads, 2) void grouped_gemm_kernel(const FfnGemmParams p) {
    using El = Elem<T>;
    constexpr int kBM = wide::kBM, kThreads = wide::kThreads, kShortRows = 64;
    __shared__ __attribute__((aligned(16))) wide::TileLds lds;

    // ---- tile coordinates.  Linear id L: xcd = L % 8 (hardware round-robin);
    // within an XCD walk (column group, m-tile, column-in-group).
    int mt, nu;
    {
        const long L = blockIdx.x;
        const int xcd = static_cast<int>(L & 7);
        const long j = L >> 3;
        const long per_group = static_cast<long>(p.mt_total) * p.ngt;
        const long g = j / per_group, rem = j % per_group;
        mt = static_cast<int>(rem / p.ngt);
        nu = static_cast<int>((g * 8 + xcd) * p.ngt + rem % p.ngt);
        if (nu >= p.n_units) return;
    }
    // m-tile -> (expert, first row)
    int e = 0;
    long row0 = 0, row_end = 0;
    {
        int tiles_before = 0;
        bool found = false;
        for (int i = 0; i < p.E; ++i) {
            const long lo = p.offsets[i], hi = p.offsets[i + 1];
            const int tiles = static_cast<int>((hi - lo + kBM - 1) / kBM);
            if (!found && mt < tiles_before + tiles) {
                e = i;
                row0 = lo + static_cast<long>(mt - tiles_before) * kBM;
                row_end = hi;
                found = true;
            }
            tiles_before += tiles;
        }
        if (!found) return;
    }
    const long n0 = static_cast<long>(nu) * (kSwiglu ? kBN : 2 * kBN);

    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int lr = lane & 31, lh = lane >> 5;
    const int wm = wave >> 1, wn = wave & 1;

    // ---- global -> register staging: 16-byte chunks, 8 per row of a k-tile
    unsigned a_off[4], b_off[2][2];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int c = tid + i * kThreads;
        long prow = row0 + (c >> 3);
        if (prow >= row_end) prow = row_end - 1;  // clamp: result rows beyond the expert are not stored
        const long src = p.order ? static_cast<long>((static_cast<unsigned long long>(static_cast<unsigned>(p.order[prow])) * p.div_m) >> p.div_s) : prow;
        a_off[i] = static_cast<unsigned>(src * p.K + (c & 7) * 8);
    }
    // weights of this expert: a uniform base per column group, rows as 32-bit offsets
    const std::uint16_t* const b_base[2] = {p.b + static_cast<long>(e) * p.Nw * p.K, p.b2 + static_cast<long>(e) * p.Nw * p.K};
#pragma unroll
    for (int g = 0; g < 2; ++g)
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const int c = tid + i * kThreads;
            long wrow = (kSwiglu ? n0 : n0 + g * kBN) + (c >> 3);
            if (wrow >= p.Nw) wrow = p.Nw - 1;
            b_off[g][i] = static_cast<unsigned>(wrow * p.K + (c & 7) * 8);
        }
    // An expert's last tile with few rows: the waves share those rows (same sums, a fraction of
    // the time) instead of most of them idling through the contraction.
    if (row_end - row0 <= kShortRows) {
        float16_t sacc[2];
        wide::short_tile_mainloop<T>(p.a, a_off[0], b_base, b_off, p.K, lds, sacc);
        const long col = n0 + (wave & 3) * 32 + lr;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const long prow = row0 + (wave >> 2) * 32 + (r >> 2) * 8 + 4 * lh + (r & 3);
            if (prow >= row_end) continue;
            if (kSwiglu) {
                if (col < p.N) p.c[prow * p.N + col] = swiglu_from_acc<T>(sacc[0][r], sacc[1][r]);
            } else {
                if (col < p.N) p.c[prow * p.N + col] = El::from_f32(sacc[0][r]);
                if (col + kBN < p.N) p.c[prow * p.N + col + kBN] = El::from_f32(sacc[1][r]);
            }
        }
        return;
    }
    float16_t acc[2][2][2];
    wide::tile_mainloop<T>(p.a, a_off, b_base, b_off, p.K, lds, acc);

    // ---- epilogue.  Accumulator lane (column lr, half lh) holds rows (r/4)*8 + 4*lh + r%4.
    // One uniform base, a 32-bit byte offset per lane (the launcher sends output rows of 2^22
    // elements or more elsewhere), rows and columns checked against counts in 32-bit registers,
    // narrowing by the conversion instruction; a 32 x 32 block of the plain product in which a NaN
    // turns up is narrowed again in software, which writes NaNs as the host's types do.
    {
        char* cb = reinterpret_cast<char*>(p.c + row0 * p.N + n0);       // uniform
        const long rows_left = row_end - row0, cols_left = p.N - n0;
        const int nrows = static_cast<int>(rows_left < kBM ? rows_left : kBM) - (wm * 64 + 4 * lh);
        const int ncols = static_cast<int>(cols_left < 2 * kBN ? cols_left : 2 * kBN) - (wn * 64 + lr);
        const unsigned ld2 = static_cast<unsigned>(p.N) * 2u;
        unsigned lane_b = static_cast<unsigned>(wm * 64 + 4 * lh) * ld2 + static_cast<unsigned>(wn * 64 + lr) * 2u;
        asm volatile("" : "+v"(lane_b));       // one add per store from here on
        const bool full = rows_left >= kBM && cols_left >= (kSwiglu ? kBN : 2 * kBN);    // uniform
#pragma unroll
        for (int mi = 0; mi < 2; ++mi)
#pragma unroll
            for (int ni = 0; ni < 2; ++ni) {
                if (kSwiglu) {
                    if (ni * 32 >= ncols) continue;
                    std::uint16_t o[16];
#pragma unroll
                    for (int r = 0; r < 16; ++r) o[r] = swiglu_from_acc<T>(acc[0][mi][ni][r], acc[1][mi][ni][r]);
                    if (full) store_block<true>(cb + ni * 64, lane_b, ld2, mi, nrows, o);
                    else      store_block<false>(cb + ni * 64, lane_b, ld2, mi, nrows, o);
                } else {
#pragma unroll
                    for (int g = 0; g < 2; ++g) {
                        if (g * kBN + ni * 32 >= ncols) continue;
                        std::uint16_t o[16];
                        narrow_block<T>(acc[g][mi][ni], o);
                        char* blk = cb + (g * kBN + ni * 32) * 2;
                        if (full) store_block<true>(blk, lane_b, ld2, mi, nrows, o);
                        else      store_block<false>(blk, lane_b, ld2, mi, nrows, o);
                    }
                }
            }
    }
}

// f(integral_constant<int, I>) for I = 0 .. N-1
template <int... I, typename F>
__device__ __forceinline__ void static_for_impl(std::integer_sequence<int, I...>, F&& f) {
    (f(std::integral_constant<int, I>{}), ...);
}
template <int N, typename F>
__device__ __forceinline__ void static_for(F&& f) {
    static_for_impl(std::make_integer_sequence<int, N>{}, static_cast<F&&>(f));
}

// A wave's queue of SwiGLU values that left the common tier (four of one lane per entry): laid over the second half of one
// of the four tile stages once the contraction is done (the first half is for the wave's rows on their way out).
struct SwigluQueue {
    static constexpr unsigned kEntries = 448;
    unsigned where[kEntries];       // the first of the four in the wave's rows (RowsOut)
    flex::float4v gate[kEntries], up[kEntries];
};
__device__ __forceinline__ unsigned scalar_of(unsigned v) { return static_cast<unsigned>(__builtin_amdgcn_readfirstlane(static_cast<int>(v))); }
constexpr int kTileBand = 8;        // m-tiles whose column units an XCD walks through together: they share the experts' weights in its L2
constexpr int kStageElems = 256 * kBK;          // a stage of either operand: 256 rows of a k-tile
constexpr int kQueueAt = 128 * 64;               // elements: the rows of a wave, 64 columns each
static_assert(sizeof(SwigluQueue) <= (kStageElems - kQueueAt) * 2, "a queue in a tile stage");
static_assert(kBK == kFormStep, "moe_forms.h");

// The weight rows of a 256-column tile that come as two groups of 128: a wave's 128 rows of the LDS tile are 64 rows of
// group 0 and the 64 rows of group 1 with the same index, so that the accumulators of a gate column and of its up
// column belong to the same lane.  (An LDS tile row r: wave r / 128, block r % 128 / 16, of which four are group 0's.)
struct TwoGroups : flex::Operand<8, false> {
    const char* base2;
    struct Rsrc { __amdgpu_buffer_rsrc_t g[2]; };
    // b, b2: row 0 of the groups, of each of which rows_left exist (<= 0: none)
    __device__ __forceinline__ void aim(const std::uint16_t* b, const std::uint16_t* b2, long K, long rows_left, int w) {
        const int lane = threadIdx.x & 63, l16 = lane & 15, kq = lane >> 4;
        base = reinterpret_cast<const char*>(b);
        base2 = reinterpret_cast<const char*>(b2);
        left = rows_left * K * 2;
        step = kBK * 2;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const int r = (i * 4 + flex::wave_id()) * 8 + (lane >> 3);
            const long row = (r >> 7) * 64 + ((r >> 4) & 3) * 16 + (r & 15);
            off[i] = static_cast<std::uint32_t>(row * K * 2 + ((lane & 7) ^ (lane >> 3)) * 16);
        }
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) fb[ks] = (w * 128 + l16) * kBK + ((ks * 4 + kq) ^ (l16 & 7)) * 8;
    }
    __device__ __forceinline__ Rsrc rsrc(int kt, int k_tiles) const {
        const long l = left - kt * step;
        const int n = static_cast<int>(static_cast<std::uint32_t>(l < 0 || kt >= k_tiles ? 0 : (l > flex::kMaxExtent ? flex::kMaxExtent : l)));
        return {{__builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(base + kt * step), 0, n, 0x00020000),
                 __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(base2 + kt * step), 0, n, 0x00020000)}};
    }
    __device__ __forceinline__ void request(const Rsrc& r, std::uint16_t* tile, int i) const {
        flex::Operand<8, false>::request((i & 2) ? r.g[1] : r.g[0], tile, i);
    }
};

// The experts' m-tiles, counted expert by expert: every lane looks at one expert (64 at a time; one after the other the offsets of
// 64 experts are 64 round trips before a workgroup's first load).  `tiles_of(rows)`: the tiles of an expert with that many.
struct ExpertTiles {
    int lo, hi, tiles, upto;        // of 64 experts, by lane: rows [lo, hi), tiles, and those of the 64 up to this one
    template <typename Tiles> __device__ __forceinline__ void look(const FfnGemmParams& p, int e0, Tiles tiles_of) {
        const int lane = threadIdx.x & 63, i = e0 + lane;
        lo = i < p.E ? static_cast<int>(p.offsets[i]) : 0;
        hi = i < p.E ? static_cast<int>(p.offsets[i + 1]) : 0;
        count(tiles_of);
    }
    template <typename Tiles> __device__ __forceinline__ void count(Tiles tiles_of) {
        tiles = tiles_of(hi - lo);
        upto = tiles;
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
            const int o = __shfl_up(upto, d, 64);
            if (static_cast<int>(threadIdx.x & 63) >= d) upto += o;
        }
    }
    __device__ __forceinline__ int all() const { return __builtin_amdgcn_readlane(upto, 63); }
};

// `head`: experts 0 to 63
template <typename Tiles> __device__ __forceinline__ int count_tiles(const FfnGemmParams& p, const ExpertTiles& head, Tiles tiles_of) {
    int n = head.all();
    for (int e0 = 64; e0 < p.E; e0 += 64) {
        ExpertTiles more;
        more.look(p, e0, tiles_of);
        n += more.all();
    }
    return n;
}

// m-tile `mt`, one of those counted: its expert, that expert's rows and which of its tiles it is
struct TileOf { int e, lo, hi, nth; };
template <typename Tiles> __device__ __forceinline__ TileOf find_tile(const FfnGemmParams& p, int mt, const ExpertTiles& head, Tiles tiles_of) {
    ExpertTiles at = head;
    int before = 0, e0 = 0;
    while (e0 + 64 < p.E && mt >= before + at.all()) {
        before += at.all();
        e0 += 64;
        at.look(p, e0, tiles_of);
    }
    const int first = before + at.upto - at.tiles;
    const int l = __builtin_ctzll(__builtin_amdgcn_ballot_w64(mt >= first && mt < first + at.tiles) | 1ull << 63);
    return {e0 + l, __builtin_amdgcn_readlane(at.lo, l), __builtin_amdgcn_readlane(at.hi, l), mt - __builtin_amdgcn_readlane(first, l)};
}

// The same on the four-wave 256 x 256 tile of v_mfma_f32_16x16x32 whose loads go straight to LDS (gemm_flex.h): what the
// layer runs on when the experts are big enough for 256-row tiles.  Tile coordinates and the search for the
// m-tile's expert as above; the routed rows are gathered by the addresses the lanes fetch from.  A lane of accumulator
// block (i, j) holds row i*16 + lane%16 and columns 4*(lane/16) .. + 3 of column block j; of the gate-up product that is group j / 4
// (TwoGroups), columns wn*64 + (j % 4)*16 of it, so gate and up of one output sit in blocks j and j + 4 of the same lane.  Results leave through LDS in
// whole rows (RowsOut).  Bound by the matrix cores' power and the LDS reads.
template <typename T, bool kSwiglu>
__global__ __launch_bounds__(flex::kThreads, 1) void grouped_gemm_direct_kernel(const FfnGemmParams p) {
    using El = Elem<T>;
    constexpr int kBM = 256;
    __shared__ __attribute__((aligned(1024))) std::uint16_t a0[kStageElems];
    __shared__ __attribute__((aligned(1024))) std::uint16_t a1[kStageElems];
    __shared__ __attribute__((aligned(1024))) std::uint16_t b0[kStageElems];
    __shared__ __attribute__((aligned(1024))) std::uint16_t b1[kStageElems];
    // Super-tiles of kSuperM row tiles x kSuperN column units, the 32 workgroups an XCD runs together: they fetch 8 panels of
    // routed rows and 4 to 8 of weights between them (a sweep of all row tiles over two column units: 18 to 20).
    // They are dealt to the XCDs one after the other, columns first, so that the XCDs share the rows' panels.
    // (8192 tokens, 8 experts, H 4096, I 14336, the layer: 8 x 4 4675 us, 4 x 8 4750, 16 x 2 4760, 32 x 1 for the plain product 4820.)
    // m-tile -> (expert, first row): first every expert's tiles with more than 64 rows, then the short last ones, which
    // take a fraction of the time and fill in at the end of every XCD's list
    int mt, nu;
    int e;
    long row0, row_end;
    {
        ExpertTiles head;
        TileOf at;
        if (p.ngt != 0) {
            // A few rounds of tiles: a contiguous run of the tiles that there are for every XCD, as grouped_tile_kernel deals them, since a few
            // super-tiles, some of them half empty, are not the same number for all (down in bf16, 5595 tokens, top-2, 8 experts, H 2112,
            // I 5760: 368 us in super-tiles, 272; gate-up in fp16, 1668 tokens, top-1, 4 experts, 832 x 3264, less than a round: 61 on tiles of
            // 128 x 128, 41).  Expert by expert: with the short tiles at the end of the list one XCD has most of them (3056 tokens, top-6,
            // 64 experts, 1472 x 768, the layer: 290, and 271 so).
            auto tiles_of = [](int rows) { return (rows + kBM - 1) / kBM; };
            head.look(p, 0, tiles_of);
            const unsigned m_tiles = static_cast<unsigned>(count_tiles(p, head, tiles_of)), units = static_cast<unsigned>(p.n_units);
            const unsigned total = m_tiles * units, q = total / 8, r = total % 8, x = blockIdx.x % 8, i = blockIdx.x / 8;
            if (i >= q + (x < r ? 1 : 0)) return;
            const unsigned lin = x * q + (x < r ? x : r) + i;
            const unsigned band = scalar_of(lin / (kTileBand * units)), in = lin - band * kTileBand * units;
            const unsigned left = m_tiles - band * kTileBand, rows = left < kTileBand ? left : kTileBand;
            nu = static_cast<int>(scalar_of(in / rows));
            mt = static_cast<int>(band * kTileBand + (in - static_cast<unsigned>(nu) * rows));
            at = find_tile(p, mt, head, tiles_of);
        } else {
            const unsigned xcd = blockIdx.x & 7, j = blockIdx.x >> 3;
            const unsigned super = j / (kSuperM * kSuperN) * 8 + xcd, in = j % (kSuperM * kSuperN);
            const unsigned across = (static_cast<unsigned>(p.n_units) + kSuperN - 1) / kSuperN;
            // (quotients come from vector arithmetic: what depends on them is to stay in scalar registers)
            const unsigned mb = static_cast<unsigned>(__builtin_amdgcn_readfirstlane(static_cast<int>(super / across)));
            mt = static_cast<int>(mb * kSuperM + in % kSuperM);
            nu = static_cast<int>((super - mb * across) * kSuperN + in / kSuperM);
            if (nu >= p.n_units) return;
            auto whole = [](int rows) { return rows / kBM + (rows % kBM > 64); };
            auto ends = [](int rows) { return static_cast<int>(rows % kBM > 0 && rows % kBM <= 64); };
            head.look(p, 0, whole);
            const int n_whole = count_tiles(p, head, whole);
            if (mt < n_whole) {
                at = find_tile(p, mt, head, whole);
            } else {
                head.count(ends);
                if (mt - n_whole >= count_tiles(p, head, ends)) return;
                at = find_tile(p, mt - n_whole, head, ends);
                at.nth = (at.hi - at.lo) / kBM;
            }
        }
        e = at.e;
        row0 = at.lo + static_cast<long>(at.nth) * kBM;
        row_end = at.hi;
    }
    const long n0 = static_cast<long>(nu) * (kSwiglu ? kBN : 2 * kBN);
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int l16 = lane & 15, kq = lane >> 4;
    const int wm = wave >> 1, wn = wave & 1;

    // W requests per wave of the routed rows: rows past the expert's last are not fetched (their results are not stored)
    auto aim_rows = [&](auto& oa, int w) __attribute__((always_inline)) {
        constexpr int W = sizeof(oa.off) / sizeof(oa.off[0]);
        oa.base = reinterpret_cast<const char*>(p.order ? p.a : p.a + row0 * p.K);
        oa.left = p.order ? p.a_bytes : (row_end - row0) * p.K * 2;
        oa.step = kBK * 2;
#pragma unroll
        for (int i = 0; i < W; ++i) {
            const long r = (i * 4 + flex::wave_id()) * 8 + (lane >> 3);
            const bool live = row0 + r < row_end;
            long src = r;
            if (p.order) src = static_cast<long>((static_cast<unsigned long long>(static_cast<unsigned>(p.order[live ? row0 + r : row0])) * p.div_m) >> p.div_s);
            oa.off[i] = live ? static_cast<std::uint32_t>(src * p.K * 2 + ((lane & 7) ^ (lane >> 3)) * 16) : flex::kOutOfRange;
        }
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) oa.fb[ks] = (w * 16 * W + l16) * kBK + ((ks * 4 + kq) ^ (l16 & 7)) * 8;
    };
    typename std::conditional<kSwiglu, TwoGroups, flex::Operand<8, false>>::type ob;
    {
        const long first = static_cast<long>(e) * p.Nw * p.K;
        if constexpr (kSwiglu) ob.aim(p.b + first + n0 * p.K, p.b2 + first + n0 * p.K, p.K, p.Nw - n0, wn);
        else                   ob.init(p.b + first, p.K, p.Nw, n0, 0, p.K, wn);
    }
    // The tile with 32 MI of its rows: an expert's last tile takes the fewest that hold its rows, with the same sums in the
    // same order (64 rows about a third of a full tile's time, 128 rows two thirds).
    auto tile = [&](auto mi) __attribute__((always_inline)) {
    constexpr int MI = decltype(mi)::value;
    flex::Operand<MI, false> oa;
    aim_rows(oa, wm);
    flex::float4v acc[MI][8];
    flex::mainloop<T, MI, 8, 2>(oa, ob, static_cast<int>(p.K), {a0, a1}, {b0, b1}, acc);
    if constexpr (kSwiglu) {
        // About one value in a thousand leaves the common tier of SwiGLU, and where one lane of the 64 does,
        // the whole wave walks through the fp64 formula: at 128 values a lane that happened eight times a tile
        // and cost 4 % of the kernel.  A lane whose four values do not all pass queues them (the accumulators
        // and where they go) in one of the tile stages, which nobody reads any more; after
        // the last row block (or when the next one might not fit) the wave works its queue off, one value per lane.
        __syncthreads();
        // (the lane's coordinates derived again, from a value the compiler cannot trace: none of this is to
        // occupy a register during the contraction, which has none to spare)
        int t = threadIdx.x;
        asm volatile("" : "+v"(t));
        const int lane = t & 63, wave = t >> 6, l16 = t & 15, kq = (t >> 4) & 3, wm = t >> 7, wn = (t >> 6) & 1;
        std::uint16_t* const stage = wave == 0 ? a0 : (wave == 1 ? a1 : (wave == 2 ? b0 : b1));
        SwigluQueue& q = *reinterpret_cast<SwigluQueue*>(stage + kQueueAt);
        flex::lds_u16* const out = (flex::lds_u16*)stage;
        using Out = flex::RowsOut<4>;
        const unsigned long long lanes_below = (1ull << lane) - 1ull;
        unsigned queued = 0;      // uniform
        auto work_off = [&]() __attribute__((always_inline)) {
            lds_exchange_in_wave();
            for (unsigned idx = lane; idx < 4 * queued; idx += 64) {
                const unsigned e = idx >> 2, r = idx & 3, where = q.where[e];
                const float a0 = reinterpret_cast<const float*>(&q.gate[e])[r];
                const float a1 = reinterpret_cast<const float*>(&q.up[e])[r];
                out[where + r] = swiglu_from_acc<T>(a0, a1);
            }
            lds_exchange_in_wave();
            queued = 0;
        };
        const long rows_left = row_end - row0 - wm * 16 * MI, cols_left = p.N - n0 - wn * 64;
        static_for<MI>([&](auto I) __attribute__((always_inline)) {
            constexpr int i = decltype(I)::value;
#pragma unroll
            for (int jb = 0; jb < 4; ++jb) {
                const int row = i * 16 + l16, at = Out::at(row, jb, kq);
                const bool live = row < rows_left && jb * 16 + 4 * kq < cols_left;
                std::uint16_t o[4];
                const bool ok = swiglu4_common_tier<T>(acc[i][jb], acc[i][4 + jb], o);
                *(flex::lds_u32x2*)(out + at) = u32x2{o[0] | (static_cast<std::uint32_t>(o[1]) << 16), o[2] | (static_cast<std::uint32_t>(o[3]) << 16)};
                const unsigned long long left = __builtin_amdgcn_ballot_w64(live && !ok);
                if (left != 0) {
                    if (live && !ok) {
                        const unsigned slot = queued + static_cast<unsigned>(__builtin_popcountll(left & lanes_below));
                        q.where[slot] = static_cast<unsigned>(at);
                        q.gate[slot] = acc[i][jb];
                        q.up[slot] = acc[i][4 + jb];
                    }
                    queued += static_cast<unsigned>(__builtin_popcountll(left));
                }
            }
            // a row block queues 4 x 64 entries at most
            if (i == MI - 1 || queued > SwigluQueue::kEntries - 256) work_off();
        });
        flex::store_rows<T, MI, 4>(out, p.c + (row0 + wm * 16 * MI) * p.N + n0 + wn * 64, p.N, rows_left, cols_left, true, false);
        return;
    } else {
        flex::lds_u16* const out = (flex::lds_u16*)(wave == 0 ? a0 : (wave == 1 ? a1 : (wave == 2 ? b0 : b1)));
        __syncthreads();
        float probe = 0.f;
        static_for<MI>([&](auto I) __attribute__((always_inline)) {
            constexpr int i = decltype(I)::value;
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                const flex::float4v v = flex::in_turn<0>(acc[i][j]);
                probe += (v[0] + v[1]) + (v[2] + v[3]);
                flex::RowsOut<8>::lay(out, i * 16 + l16, j, kq, flex::pack4<T>(v));
            }
        });
        const bool nan_here = __builtin_amdgcn_ballot_w64(probe != probe) != 0;      // (an infinity minus an infinity counts as well)
        const long r0 = row0 + wm * 16 * MI, c0 = n0 + wn * 128;
        flex::store_rows<T, MI, 8>(out, p.c + r0 * p.N + c0, p.N, row_end - r0, p.N - c0, true, nan_here);
    }
    };      // tile
    const long rows = row_end - row0;
    if (rows > 192)      tile(std::integral_constant<int, 8>{});
    else if (rows > 128) tile(std::integral_constant<int, 6>{});
    else if (rows > 64)  tile(std::integral_constant<int, 4>{});
    else                 tile(std::integral_constant<int, 2>{});
}

// ---- experts of a few dozen to a few hundred rows: tiles of 32 MI rows on the staged mainloop of gemm_flex.h, with enough
// stages in flight that one or two workgroups per CU do not wait for each tile's way from L2, which is what bounds these sizes (the
// register-staged 128-row tiles that they replace had one tile under way).
// The weight rows of a tile are 32 NJ columns of the result or, for gate and up, 16 NJ of each: of a wave's NJ blocks of 16 the
// first half are gate rows and the second half the up rows of the same columns, so that both accumulators of an output belong to one lane.
template <int NJ> struct GateUp : flex::Operand<NJ, false> {
    const char* base2;
    struct Rsrc { __amdgpu_buffer_rsrc_t g[2]; };
    __device__ __forceinline__ void aim(const std::uint16_t* gate, const std::uint16_t* up, long K, long rows_left, int w) {
        static_assert(NJ % 4 == 0 || NJ == 2, "the rows that a wave requests at once belong to one of the two");
        const int lane = threadIdx.x & 63, l16 = lane & 15, kq = lane >> 4;
        this->base = reinterpret_cast<const char*>(gate);
        base2 = reinterpret_cast<const char*>(up);
        this->left = rows_left * K * 2;
        this->step = kBK * 2;
#pragma unroll
        for (int i = 0; i < NJ; ++i) {
            const int r = (i * 4 + flex::wave_id()) * 8 + (lane >> 3), block = (r >> 4) % NJ;
            const long row = ((r >> 4) / NJ * (NJ / 2) + block % (NJ / 2)) * 16 + (r & 15);
            this->off[i] = static_cast<std::uint32_t>(row * K * 2 + ((lane & 7) ^ (lane >> 3)) * 16);
        }
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) this->fb[ks] = (w * 16 * NJ + l16) * kBK + ((ks * 4 + kq) ^ (l16 & 7)) * 8;
    }
    __device__ __forceinline__ Rsrc rsrc(int kt, int k_tiles) const {
        const long l = this->left - kt * this->step;
        const int n = static_cast<int>(static_cast<std::uint32_t>(l < 0 || kt >= k_tiles ? 0 : (l > flex::kMaxExtent ? flex::kMaxExtent : l)));
        const char* first = NJ == 2 && flex::wave_id() >= 2 ? base2 : this->base;          // (NJ == 2: half of the waves' requests are for one matrix, half for the other)
        return {{__builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(first + kt * this->step), 0, n, 0x00020000),
                 __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(base2 + kt * this->step), 0, n, 0x00020000)}};
    }
    __device__ __forceinline__ void request(const Rsrc& r, std::uint16_t* tile, int i) const {
        flex::Operand<NJ, false>::request(NJ > 2 && (2 * i) % NJ >= NJ / 2 ? r.g[1] : r.g[0], tile, i);
    }
};

template <typename T, bool kSwiglu, int MI, int NJ, int ST>
__global__ __launch_bounds__(flex::kThreads, (MI * NJ >= 32 || ST * (MI + NJ) > 20 ? 1 : 2)) void grouped_tile_kernel(const FfnGemmParams p) {
    using OA = flex::Operand<MI, false>;
    using OB = typename std::conditional<kSwiglu, GateUp<NJ>, flex::Operand<NJ, false>>::type;
    constexpr int kBM = 32 * MI, kCols = kSwiglu ? 16 * NJ : 32 * NJ;
    __shared__ __attribute__((aligned(1024))) std::uint16_t a0[OA::kElems];
    __shared__ __attribute__((aligned(1024))) std::uint16_t a1[OA::kElems];
    __shared__ __attribute__((aligned(1024))) std::uint16_t a2[OA::kElems];     // (stages past ST are never named, and take no memory)
    __shared__ __attribute__((aligned(1024))) std::uint16_t a3[OA::kElems];
    __shared__ __attribute__((aligned(1024))) std::uint16_t b0[OB::kElems];
    __shared__ __attribute__((aligned(1024))) std::uint16_t b1[OB::kElems];
    __shared__ __attribute__((aligned(1024))) std::uint16_t b2[OB::kElems];
    __shared__ __attribute__((aligned(1024))) std::uint16_t b3[OB::kElems];
    // Workgroup w runs on XCD w % 8: every XCD takes a contiguous run of the list of tiles.  Of the tiles that there are: the grid has room for
    // any spread of the rows, and with runs of that room the last XCDs have nothing
    // (64 experts, 150 layers: 1.15 to 1.2 times the time; 8 experts: 1.07 to 1.1 times).
    auto tiles_of = [](int rows) { return (rows + kBM - 1) / kBM; };
    ExpertTiles head;
    head.look(p, 0, tiles_of);
    const unsigned m_tiles = static_cast<unsigned>(count_tiles(p, head, tiles_of)), units = static_cast<unsigned>(p.n_units);
    int mt, nu;
    {
        const unsigned total = m_tiles * units, q = total / 8, r = total % 8, x = blockIdx.x % 8, i = blockIdx.x / 8;
        if (i >= q + (x < r ? 1 : 0)) return;
        const unsigned lin = x * q + (x < r ? x : r) + i;
        const unsigned band = scalar_of(lin / (kTileBand * units)), in = lin - band * kTileBand * units;
        const unsigned left = m_tiles - band * kTileBand, rows = left < kTileBand ? left : kTileBand;
        nu = static_cast<int>(scalar_of(in / rows));
        mt = static_cast<int>(band * kTileBand + (in - static_cast<unsigned>(nu) * rows));
    }
    const TileOf at = find_tile(p, mt, head, tiles_of);
    const int e = at.e;
    const long row0 = at.lo + static_cast<long>(at.nth) * kBM, row_end = at.hi;
    const long n0 = static_cast<long>(nu) * kCols;
    const int lane = threadIdx.x & 63, wave = flex::wave_id(), l16 = lane & 15, kq = lane >> 4;
    const int wm = wave >> 1, wn = wave & 1;

    OA oa;          // rows past the expert's last are not fetched (their results are not stored)
    oa.base = reinterpret_cast<const char*>(p.order ? p.a : p.a + row0 * p.K);
    oa.left = p.order ? p.a_bytes : (row_end - row0) * p.K * 2;
    oa.step = kBK * 2;
#pragma unroll
    for (int i = 0; i < MI; ++i) {
        const long r = (i * 4 + wave) * 8 + (lane >> 3);
        const bool live = row0 + r < row_end;
        long src = r;
        if (p.order) src = static_cast<long>((static_cast<unsigned long long>(static_cast<unsigned>(p.order[live ? row0 + r : row0])) * p.div_m) >> p.div_s);
        oa.off[i] = live ? static_cast<std::uint32_t>(src * p.K * 2 + ((lane & 7) ^ (lane >> 3)) * 16) : flex::kOutOfRange;
    }
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) oa.fb[ks] = (wm * 16 * MI + l16) * kBK + ((ks * 4 + kq) ^ (l16 & 7)) * 8;
    OB ob;
    const long first = static_cast<long>(e) * p.Nw * p.K;
    if constexpr (kSwiglu) ob.aim(p.b + first + n0 * p.K, p.b2 + first + n0 * p.K, p.K, p.Nw - n0, wn);
    else                   ob.init(p.b + first, p.K, p.Nw, n0, 0, p.K, wn);
    flex::float4v acc[MI][NJ];
    const int K = static_cast<int>(p.K);
    if constexpr (ST == 2)      flex::mainloop<T, MI, NJ, 2>(oa, ob, K, {a0, a1}, {b0, b1}, acc);
    else if constexpr (ST == 3) flex::mainloop<T, MI, NJ, 3>(oa, ob, K, {a0, a1, a2}, {b0, b1, b2}, acc);
    else                        flex::mainloop<T, MI, NJ, 4>(oa, ob, K, {a0, a1, a2, a3}, {b0, b1, b2, b3}, acc);

    // (N is a multiple of 64 here and the rows are 16-byte aligned)
    constexpr int OJ = kSwiglu ? NJ / 2 : NJ;               // column blocks of the result per wave
    using Out = flex::RowsOut<OJ>;
    static_assert(16 * MI * 16 * OJ <= OA::kElems && 16 * MI * 16 * OJ <= OB::kElems, "a wave's rows in a stage");
    flex::lds_u16* const out = wave == 0 ? (flex::lds_u16*)a0 : wave == 1 ? (flex::lds_u16*)a1 : wave == 2 ? (flex::lds_u16*)b0 : (flex::lds_u16*)b1;
    const long r0 = row0 + wm * 16 * MI, c0 = n0 + wn * 16 * OJ;
    __syncthreads();                                        // (no wave's requests are on their way to the stages)
    float probe = 0.f;
#pragma unroll
    for (int i = 0; i < MI; ++i) {
        const long prow = r0 + i * 16 + l16;
        if constexpr (kSwiglu) {
#pragma unroll
            for (int j = 0; j < NJ / 2; ++j) {
                std::uint16_t o[4];
                const bool ok = swiglu4_common_tier<T>(acc[i][j], acc[i][NJ / 2 + j], o);
                if (!ok && prow < row_end) {
#pragma unroll 1
                    for (int r = 0; r < 4; ++r) {
                        const float g = r < 2 ? (r == 0 ? acc[i][j][0] : acc[i][j][1]) : (r == 2 ? acc[i][j][2] : acc[i][j][3]);
                        const float u = r < 2 ? (r == 0 ? acc[i][NJ / 2 + j][0] : acc[i][NJ / 2 + j][1]) : (r == 2 ? acc[i][NJ / 2 + j][2] : acc[i][NJ / 2 + j][3]);
                        const std::uint16_t v = swiglu_from_acc<T>(g, u);
                        o[0] = r == 0 ? v : o[0];
                        o[1] = r == 1 ? v : o[1];
                        o[2] = r == 2 ? v : o[2];
                        o[3] = r == 3 ? v : o[3];
                    }
                }
                Out::lay(out, i * 16 + l16, j, kq, u32x2{o[0] | (static_cast<std::uint32_t>(o[1]) << 16), o[2] | (static_cast<std::uint32_t>(o[3]) << 16)});
            }
        } else {
#pragma unroll
            for (int j = 0; j < NJ; ++j) {
                const flex::float4v v = acc[i][j];
                probe += (v[0] + v[1]) + (v[2] + v[3]);
                Out::lay(out, i * 16 + l16, j, kq, flex::pack4<T>(v));
            }
        }
    }
    const bool nan_here = !kSwiglu && __builtin_amdgcn_ballot_w64(probe != probe) != 0;      // (an infinity minus an infinity counts as well)
    flex::store_rows<T, MI, OJ>(out, p.c + r0 * p.N + c0, p.N, row_end - r0, p.N - c0, true, nan_here);
}

// ---- few rows per expert (decode-time batches): the layer is bound by streaming every active
// expert's weights once, which 128-row tiles with a handful of live rows do at half the memory
// rate (and a single token, two active experts, at a fifth of it: its down-projection is 32
// workgroups).  A workgroup owns 16 weight rows of one expert (for the gate-up GEMM the 16 gate rows and
// the 16 up rows of the same columns) and its eight waves split the contraction (stream_rows.h).  An expert's
// rows are taken up to 8, 16 or 32 at a time, whichever holds them, so any count works (the weights of a second
// pass come from L2); experts without rows return at once.
// (The SwiGLU of a workgroup's blocks waits until its last one: its fp64 tier would not fit into the registers beside
// the requests under way.  Until then the sums stay in LDS, kFewBlocks blocks of them.)
constexpr int kFewBlocks = 2;

template <typename T, bool kSwiglu, int XQ>
__device__ __forceinline__ void few_rows(const FfnGemmParams& p, int e, long row_lo, long row_hi, std::uint16_t* lds, float4_t* kept) {
    using El = Elem<T>;
    using S = stream::Shape<(kSwiglu ? 2 : 1), 1, XQ>;
    constexpr int NB = S::kBlocks, MB = S::kXBlocks;
    const int lane = threadIdx.x & 63;
    const long n0 = static_cast<long>(blockIdx.x) * 16, step = static_cast<long>(gridDim.x) * 16;
    const int count = static_cast<int>((p.Nw - n0 + step - 1) / step);
    const long first = (static_cast<long>(e) * p.Nw + n0) * p.K;
    const std::uint16_t* w[NB];
    w[0] = p.b + first;
    if constexpr (kSwiglu) w[1] = p.b2 + first;
    for (long chunk = row_lo; chunk < row_hi; chunk += XQ * 8) {
        std::uint32_t x_off[XQ];
#pragma unroll
        for (int q = 0; q < XQ; ++q) {
            long prow = chunk + q * 8 + (lane >> 3);
            if (prow >= row_hi) prow = row_hi - 1;
            const long src = p.order ? static_cast<long>((static_cast<unsigned long long>(static_cast<unsigned>(p.order[prow])) * p.div_m) >> p.div_s) : prow;
            x_off[q] = static_cast<std::uint32_t>(src * p.K * 2);
        }
        // value r of lane l in row block m of column block j: routed row l % 16 of the row block, column 4 (l / 16) + r
        auto put = [&](int j, int m, int l, int r, float g, float u) __attribute__((always_inline)) {
            const long prow = chunk + m * 16 + (l & 15), col = n0 + j * step + 4 * (l >> 4) + r;
            if (prow >= row_hi || (XQ == 1 && (l & 15) >= 8) || col >= p.N) return;
            if constexpr (kSwiglu) p.c[prow * p.N + col] = swiglu_from_acc<T>(g, u);
            else                   p.c[prow * p.N + col] = El::from_f32(g);
        };
        stream::products<T, NB, 1, XQ, false>(w, p.K, p.Nw - n0, step, count, p.K, p.a, p.a_bytes, x_off, lds,
                                       [&](int j, const float4_t (&acc)[NB][MB]) __attribute__((always_inline)) {
            stream::share<NB, MB>(lds, acc);
            const int m = stream::wave_id();             // wave m finishes row block m
            if (m < MB) {
                if constexpr (kSwiglu) {
#pragma unroll
                    for (int b = 0; b < 2; ++b) kept[((j * MB + m) * 2 + b) * 64 + lane] = stream::sum_of<NB, MB>(lds, b, m);
                } else {
                    const float4_t g = stream::sum_of<NB, MB>(lds, 0, m);
#pragma unroll
                    for (int r = 0; r < 4; ++r) put(j, m, lane, r, g[r], 0.f);
                }
            }
            lds_barrier();                               // the LDS is free for the next block
        });
        if constexpr (kSwiglu) {
            const float* v = reinterpret_cast<const float*>(kept);
            for (int i = threadIdx.x; i < count * MB * 256; i += stream::kThreads) {
                const int jm = i >> 8, in = i & 255;
                put(jm / MB, jm % MB, in >> 2, in & 3, v[jm * 512 + in], v[jm * 512 + 256 + in]);
            }
            lds_barrier();                               // the kept sums are free for the next rows
        }
    }
}

template <typename T, bool kSwiglu>
__global__ __launch_bounds__(stream::kThreads, 4) void grouped_few_rows_kernel(const FfnGemmParams p) {
    __shared__ __attribute__((aligned(1024))) std::uint16_t lds[stream::Shape<(kSwiglu ? 2 : 1), 1, 4>::kLdsElems];
    __shared__ float4_t kept[kSwiglu ? kFewBlocks * 2 * 2 * 64 : 1];
    const int e = blockIdx.y;
    const long row_lo = p.offsets[e], row_hi = p.offsets[e + 1];
    const int rows = __builtin_amdgcn_readfirstlane(static_cast<int>(row_hi - row_lo));
    if (rows <= 0) return;
    if (rows <= 8)       few_rows<T, kSwiglu, 1>(p, e, row_lo, row_hi, lds, kept);
    else if (rows <= 16) few_rows<T, kSwiglu, 2>(p, e, row_lo, row_hi, lds, kept);
    else                 few_rows<T, kSwiglu, 4>(p, e, row_lo, row_hi, lds, kept);
}

// out[t, :] = T( sum_slot T( y[inv[t*k+slot], :] * T(w[t, slot]) ) ), 8 columns per lane, the sum in double.  KC slots at a time, which divides k: their places and
// weights are asked for together, and then their rows, so a lane waits for two trips to memory and not for two per slot.  (A product of two 16-bit values is
// exact in fp32, or rounded as from double; so is the sum of two.  One slot after the other with 64-bit divisions for the place, in double throughout,
// and this: 8192 tokens, top-2, 4096 columns 44.0 and 36.5 us; 555, top-6, 2496 9.2 and 7.0; 2344, top-1, 1088 5.3 and 4.5.)
template <typename T, int KC, bool kAll>
__global__ __launch_bounds__(kThreads) void moe_combine_kernel(const std::uint16_t* __restrict__ y, const float* __restrict__ topw, const long* __restrict__ inv_order,
                                                              std::uint16_t* __restrict__ out, unsigned total, unsigned hv, int k) {
    using El = Elem<T>;
    typedef typename std::conditional<(kAll && KC <= 2), float, double>::type sum_t;
    for (unsigned i = blockIdx.x * kThreads + threadIdx.x; i < total; i += gridDim.x * kThreads) {
        const unsigned t = i / hv, c = i - t * hv;
        const long first = static_cast<long>(t) * k;
        sum_t acc[8] = {};
        for (int s = 0; s < (kAll ? KC : k); s += KC) {
            float w[KC];
            u32x4 v[KC];
#pragma unroll
            for (int u = 0; u < KC; ++u) w[u] = El::to_f32(El::from_f32(topw[first + s + u]));        // w.to(T)
#pragma unroll
            for (int u = 0; u < KC; ++u) v[u] = load16(y + (inv_order[first + s + u] * hv + c) * 8);
#pragma unroll
            for (int u = 0; u < KC; ++u)
#pragma unroll
                for (int j = 0; j < 8; ++j) acc[j] += static_cast<sum_t>(El::to_f32(El::from_f32(El::to_f32(static_cast<std::uint16_t>(v[u][j >> 1] >> (16 * (j & 1)))) * w[u])));
        }
        u32x4 o;
#pragma unroll
        for (int j = 0; j < 4; ++j)
            o[j] = El::from_f32(static_cast<float>(acc[2 * j])) | static_cast<std::uint32_t>(El::from_f32(static_cast<float>(acc[2 * j + 1]))) << 16;
        store16(out + static_cast<std::uint64_t>(i) * 8, o);
    }
}

template <typename T>
void launch_combine(const std::uint16_t* y, const float* topw, const long* inv_order, void* out, long tokens, int k, long H, hipStream_t s) {
    const unsigned hv = static_cast<unsigned>(H / 8), total = static_cast<unsigned>(tokens * (H / 8));          // (paras_moe_ffn: T H < 2^32)
    const unsigned blocks = (total + kThreads - 1) / kThreads;
    auto launch = [&](auto slots, auto all) {
        hipLaunchKernelGGL((moe_combine_kernel<T, decltype(slots)::value, decltype(all)::value>), dim3(blocks), dim3(kThreads), 0, s, y, topw, inv_order,
                           static_cast<std::uint16_t*>(out), total, hv, k);
    };
    if (k == 1)          launch(std::integral_constant<int, 1>{}, std::true_type{});
    else if (k == 2)     launch(std::integral_constant<int, 2>{}, std::true_type{});
    else if (k == 4)     launch(std::integral_constant<int, 4>{}, std::true_type{});
    else if (k % 4 == 0) launch(std::integral_constant<int, 4>{}, std::false_type{});
    else if (k % 3 == 0) launch(std::integral_constant<int, 3>{}, std::false_type{});
    else if (k % 2 == 0) launch(std::integral_constant<int, 2>{}, std::false_type{});
    else                 launch(std::integral_constant<int, 1>{}, std::false_type{});
}

// ---- sizes the MFMA tiles do not take (hidden or intermediate size not a multiple of 64) -------
// One thread per output element: the routed row's expert is looked up in `offsets`, the dot
// products over the contraction dim accumulate in fp32 (one rounding to T, like the tile kernels),
// the SwiGLU of GEMM 1 is applied to the narrowed gate and up values.  No alignment or size
// requirement; two orders of magnitude slower than the tiles, so it only serves odd shapes.
template <typename T, bool kSwiglu>
__global__ __launch_bounds__(kThreads) void grouped_any_kernel(const FfnGemmParams p) {
    using El = Elem<T>;
    const long prow = blockIdx.y;
    const long col = static_cast<long>(blockIdx.x) * kThreads + threadIdx.x;
    if (col >= p.N) return;
    int e = 0;
    while (e + 1 < p.E && prow >= p.offsets[e + 1]) ++e;
    const long src = p.order ? p.order[prow] / p.k : prow;
    const std::uint16_t* a = p.a + src * p.K;
    const std::uint16_t* w0 = p.b + (static_cast<long>(e) * p.Nw + col) * p.K;
    float acc0 = 0.f, acc1 = 0.f;
    if (kSwiglu) {
        const std::uint16_t* w1 = p.b2 + (static_cast<long>(e) * p.Nw + col) * p.K;
        for (long kk = 0; kk < p.K; ++kk) {
            const float av = El::to_f32(a[kk]);
            acc0 = fmaf(av, El::to_f32(w0[kk]), acc0);
            acc1 = fmaf(av, El::to_f32(w1[kk]), acc1);
        }
        p.c[prow * p.N + col] = swiglu_one<T>(El::from_f32(acc0), El::from_f32(acc1));
    } else {
        for (long kk = 0; kk < p.K; ++kk) acc0 = fmaf(El::to_f32(a[kk]), El::to_f32(w0[kk]), acc0);
        p.c[prow * p.N + col] = El::from_f32(acc0);
    }
}

// The combine for any H: one element per thread.
template <typename T>
__global__ __launch_bounds__(kThreads) void moe_combine_any_kernel(const std::uint16_t* __restrict__ y, const float* __restrict__ topw,
                                                                  const long* __restrict__ inv_order, std::uint16_t* __restrict__ out,
                                                                  long T_, int k, long H) {
    using El = Elem<T>;
    const long total = T_ * H;
    for (long i = static_cast<long>(blockIdx.x) * kThreads + threadIdx.x; i < total; i += static_cast<long>(gridDim.x) * kThreads) {
        const long t = i / H, c = i % H;
        double acc = 0.0;
        for (int s = 0; s < k; ++s) {
            const double w = El::to_f64(El::from_f32(topw[t * k + s]));
            acc += El::to_f64(El::from_f64(El::to_f64(y[inv_order[t * k + s] * H + c]) * w));
        }
        out[t * H + c] = El::from_f64(acc);
    }
}

size_t align_up(size_t v, size_t a) { return (v + a - 1) / a * a; }

template <typename T>
int run_ffn_any(const void* x, const void* w_gate, const void* w_up, const void* w_down, const float* topw, const long* order,
                const long* inv_order, const long* offsets, void* out, void* workspace, long T_, int E, int k, long H, long I,
                hipStream_t s) {
    const long R = T_ * k;
    auto* h = static_cast<std::uint16_t*>(workspace);
    auto* y = reinterpret_cast<std::uint16_t*>(static_cast<char*>(workspace) + align_up(static_cast<size_t>(R) * I * 2, 256));
    PARAS_REQUIRE(R <= 65535, "paras_moe_ffn: at most 65535 routed rows when the hidden or intermediate size is not a multiple of %d", kBK);
    FfnGemmParams g1{};
    g1.a = static_cast<const std::uint16_t*>(x);
    g1.b = static_cast<const std::uint16_t*>(w_gate);
    g1.b2 = static_cast<const std::uint16_t*>(w_up);
    g1.c = h;
    g1.order = order;
    g1.offsets = offsets;
    g1.K = H; g1.N = I; g1.Nw = I; g1.R = R; g1.E = E; g1.k = k;
    hipLaunchKernelGGL((grouped_any_kernel<T, true>), dim3(static_cast<unsigned>((I + kThreads - 1) / kThreads), static_cast<unsigned>(R)),
                       dim3(kThreads), 0, s, g1);
    PARAS_HIP_TRY(hipGetLastError());
    FfnGemmParams g2{};
    g2.a = h;
    g2.b = static_cast<const std::uint16_t*>(w_down);
    g2.b2 = g2.b;
    g2.c = y;
    g2.order = nullptr;
    g2.offsets = offsets;
    g2.K = I; g2.N = H; g2.Nw = H; g2.R = R; g2.E = E; g2.k = k;
    hipLaunchKernelGGL((grouped_any_kernel<T, false>), dim3(static_cast<unsigned>((H + kThreads - 1) / kThreads), static_cast<unsigned>(R)),
                       dim3(kThreads), 0, s, g2);
    PARAS_HIP_TRY(hipGetLastError());
    long blocks = (T_ * H + kThreads - 1) / kThreads;
    if (blocks > 256L * 16) blocks = 256L * 16;
    hipLaunchKernelGGL((moe_combine_any_kernel<T>), dim3(static_cast<unsigned>(blocks)), dim3(kThreads), 0, s, y, topw, inv_order,
                       static_cast<std::uint16_t*>(out), T_, k, H);
    PARAS_HIP_TRY(hipGetLastError());
    return PARAS_OK;
}

template <typename T, bool kSwiglu>
void launch_form(int form, FfnGemmParams g, hipStream_t s) {
    const GroupedForm f = kAllForms[form];
    const long cols = kSwiglu ? f.n / 2 : f.n;
    g.mt_total = static_cast<int>((g.R + f.m - 1) / f.m + (g.R < g.E ? g.R : g.E));      // an upper bound: workgroups past the last tile return
    g.n_units = static_cast<int>((g.N + cols - 1) / cols);
    const dim3 block(flex::kThreads), grid(static_cast<unsigned>(static_cast<long>(g.mt_total) * g.n_units));
    const long supers = static_cast<long>((g.mt_total + kSuperM - 1) / kSuperM) * ((g.n_units + kSuperN - 1) / kSuperN);
    switch (form) {
        case 0: hipLaunchKernelGGL((grouped_tile_kernel<T, kSwiglu, 4, 4, 2>), grid, block, 0, s, g); break;
        case 1: hipLaunchKernelGGL((grouped_tile_kernel<T, kSwiglu, 4, 4, 3>), grid, block, 0, s, g); break;
        case 2: hipLaunchKernelGGL((grouped_tile_kernel<T, kSwiglu, 2, 4, 2>), grid, block, 0, s, g); break;
        case 3: hipLaunchKernelGGL((grouped_tile_kernel<T, kSwiglu, 2, 4, 4>), grid, block, 0, s, g); break;
        case 4: hipLaunchKernelGGL((grouped_tile_kernel<T, kSwiglu, 1, 4, 4>), grid, block, 0, s, g); break;
        case 7: hipLaunchKernelGGL((grouped_tile_kernel<T, kSwiglu, 1, 2, 4>), grid, block, 0, s, g); break;
        case 8: hipLaunchKernelGGL((grouped_tile_kernel<T, kSwiglu, 2, 2, 4>), grid, block, 0, s, g); break;
        case 9: hipLaunchKernelGGL((grouped_tile_kernel<T, kSwiglu, 3, 2, 4>), grid, block, 0, s, g); break;
        case 10: hipLaunchKernelGGL((grouped_tile_kernel<T, kSwiglu, 3, 4, 2>), grid, block, 0, s, g); break;
        case 11: hipLaunchKernelGGL((grouped_tile_kernel<T, kSwiglu, 6, 4, 2>), grid, block, 0, s, g); break;
        case 12:
            if constexpr (kSwiglu) hipLaunchKernelGGL((grouped_tile_kernel<T, kSwiglu, 5, 4, 2>), grid, block, 0, s, g);
            break;
        case 13:
            if constexpr (!kSwiglu) hipLaunchKernelGGL((grouped_tile_kernel<T, kSwiglu, 6, 8, 2>), grid, block, 0, s, g);
            break;
        case 14:
            if constexpr (!kSwiglu) hipLaunchKernelGGL((grouped_tile_kernel<T, kSwiglu, 4, 8, 3>), grid, block, 0, s, g);
            break;
        default: {
            g.ngt = form == kOneByOne ? 1 : 0;
            const long wgs = form == kOneByOne ? (static_cast<long>(g.mt_total) * g.n_units + 7) / 8 * 8 : (supers + 7) / 8 * 8 * kSuperM * kSuperN;
            hipLaunchKernelGGL((grouped_gemm_direct_kernel<T, kSwiglu>), dim3(static_cast<unsigned>(wgs)), block, 0, s, g);
        }
    }
}

// The register-staged tiles' grid: an XCD sweeps up to two column units together (one expert's weight panel for them is
// 4 MB at K = 4096, the size of an XCD's L2; 4 units measured 8 % slower), fewer when there are not enough units to keep all 8
// XCDs busy.
template <typename T, bool kSwiglu>
void launch_register_staged(FfnGemmParams g, hipStream_t s) {
    const long cols = kSwiglu ? kBN : 2 * kBN;
    g.mt_total = static_cast<int>((g.R + wide::kBM - 1) / wide::kBM) + g.E;
    g.n_units = static_cast<int>((g.N + cols - 1) / cols);
    g.ngt = g.n_units < 16 ? 1 : 2;
    const long groups = (g.n_units + 8 * g.ngt - 1) / (8 * g.ngt);
    hipLaunchKernelGGL((grouped_gemm_kernel<T, kSwiglu>), dim3(static_cast<unsigned>(groups * 8 * g.ngt * g.mt_total)), dim3(wide::kThreads), 0, s, g);
}

template <typename T>
int run_ffn_tiles(const void* x, const void* w_gate, const void* w_up, const void* w_down, const float* topw,
            const long* order, const long* inv_order, const long* offsets, void* out, void* workspace, long T_,
            int E, int k, long H, long I, hipStream_t s) {
    const long R = T_ * k;
    auto* h = static_cast<std::uint16_t*>(workspace);
    auto* y = reinterpret_cast<std::uint16_t*>(static_cast<char*>(workspace) + align_up(static_cast<size_t>(R) * I * 2, 256));
    // By form, unless x is out of a 32-bit byte offset's reach (weights are aimed at from a tile's first row: paras_moe_ffn's limit on H and I
    // is theirs).  PARAS_GEMM_EIGHT_WAVES: the register-staged tiles whatever the size, for tests and measurements; looked up per call.
    const bool by_form = T_ * H * 2 <= flex::kMaxExtent && std::getenv("PARAS_GEMM_EIGHT_WAVES") == nullptr;

    FfnGemmParams g1{};
    g1.a = static_cast<const std::uint16_t*>(x);
    g1.b = static_cast<const std::uint16_t*>(w_gate);
    g1.b2 = static_cast<const std::uint16_t*>(w_up);
    g1.c = h;
    g1.order = order;
    g1.offsets = offsets;
    g1.a_bytes = T_ * H * 2;
    g1.K = H; g1.N = I; g1.Nw = I; g1.R = R; g1.E = E; g1.k = k;
    division_by(static_cast<unsigned>(k), &g1.div_m, &g1.div_s);
    if (by_form) launch_form<T, true>(grouped_tiles(true, E, R, I, H), g1, s);
    else         launch_register_staged<T, true>(g1, s);
    PARAS_HIP_TRY(hipGetLastError());

    FfnGemmParams g2{};
    g2.a = h;
    g2.b = static_cast<const std::uint16_t*>(w_down);
    g2.b2 = g2.b;  // (register-staged) column group 1 = the next 128 weight rows, selected through the row index
    g2.c = y;
    g2.order = nullptr;
    g2.offsets = offsets;
    g2.K = I; g2.N = H; g2.Nw = H; g2.R = R; g2.E = E; g2.k = k;
    if (by_form) launch_form<T, false>(grouped_tiles(false, E, R, H, I), g2, s);
    else         launch_register_staged<T, false>(g2, s);
    PARAS_HIP_TRY(hipGetLastError());

    launch_combine<T>(y, topw, inv_order, out, T_, k, H, s);
    PARAS_HIP_TRY(hipGetLastError());
    return PARAS_OK;
}

template <typename T>
int run_ffn_few_rows(const void* x, const void* w_gate, const void* w_up, const void* w_down, const float* topw,
                     const long* order, const long* inv_order, const long* offsets, void* out, void* workspace, long T_,
                     int E, int k, long H, long I, hipStream_t s) {
    const long R = T_ * k;
    // Column blocks per workgroup: two save a start each where the rows of an expert take long to multiply (8 experts,
    // 64 tokens 578 -> 557 us), one spreads better where they do not (2 tokens 203 -> 192, 5 tokens 430 -> 415).
    const long each = R > 4L * E ? 2 : 1;
    static_assert(kFewBlocks >= 2, "the sums a workgroup keeps");
    auto* h = static_cast<std::uint16_t*>(workspace);
    auto* y = reinterpret_cast<std::uint16_t*>(static_cast<char*>(workspace) + align_up(static_cast<size_t>(R) * I * 2, 256));
    FfnGemmParams g1{};
    g1.a = static_cast<const std::uint16_t*>(x);
    g1.b = static_cast<const std::uint16_t*>(w_gate);
    g1.b2 = static_cast<const std::uint16_t*>(w_up);
    g1.c = h;
    g1.order = order;
    g1.offsets = offsets;
    g1.a_bytes = T_ * H * 2;
    g1.K = H; g1.N = I; g1.Nw = I; g1.R = R; g1.E = E; g1.k = k;
    division_by(static_cast<unsigned>(k), &g1.div_m, &g1.div_s);
    hipLaunchKernelGGL((grouped_few_rows_kernel<T, true>), dim3(static_cast<unsigned>((I / 16 + each - 1) / each), static_cast<unsigned>(E)),
                       dim3(stream::kThreads), 0, s, g1);
    PARAS_HIP_TRY(hipGetLastError());
    FfnGemmParams g2{};
    g2.a = h;
    g2.b = static_cast<const std::uint16_t*>(w_down);
    g2.b2 = g2.b;
    g2.c = y;
    g2.order = nullptr;
    g2.offsets = offsets;
    g2.a_bytes = R * I * 2;
    g2.K = I; g2.N = H; g2.Nw = H; g2.R = R; g2.E = E; g2.k = k;
    hipLaunchKernelGGL((grouped_few_rows_kernel<T, false>), dim3(static_cast<unsigned>((H / 16 + each - 1) / each), static_cast<unsigned>(E)),
                       dim3(stream::kThreads), 0, s, g2);
    PARAS_HIP_TRY(hipGetLastError());
    launch_combine<T>(y, topw, inv_order, out, T_, k, H, s);
    PARAS_HIP_TRY(hipGetLastError());
    return PARAS_OK;
}

template <typename T>
int run_ffn(const void* x, const void* w_gate, const void* w_up, const void* w_down, const float* topw,
            const long* order, const long* inv_order, const long* offsets, void* out, void* workspace, long T_,
            int E, int k, long H, long I, hipStream_t s) {
    const long R = T_ * k;
    // The few-row kernels (an expert with more than 32 rows takes them 32 at a time) spend a workgroup's start on every 16 weight rows
    // of every expert, and a row's products on all of them; the tiles' down-projection is E H / 128 workgroups that walk the whole of I each.
    // So: the fewer rows and experts and the longer I.  1410 layers (1 to 64 experts, 0.4 to 64 rows each, H 512 to 4096, I 512 to 14336): this rule
    // costs 1.1 % over the better of the two in the mean and 8 % at the 95th percentile, the best limit on rows per expert alone 3.4 % and 21 %.
    // Few-row kernels / tiles: 4 experts of 11 rows, H 1280, I 9920 81 / 105 us; 8 of 10, 704 x 3072 38 / 45; 8 experts, top-2, 4096 x 14336, 1 token
    // 128 / 168, 5 tokens 369 / 380, 64 tokens 507 / 479, 128 tokens 757 / 509; 64 of 4, 768 x 1472 118 / 94; 32 of 13, 704 x 3200 115 / 97.  Beyond
    // 16 rows on average some experts have more than 32: 4 of 30, 1088 x 2176 46 / 28.
    // PARAS_MOE_FEW_ROWS = n: up to n rows per expert instead (0: never); looked up per call.
    const char* env = std::getenv("PARAS_MOE_FEW_ROWS");
    const bool few = env != nullptr ? R <= std::atol(env) * E : 4 * R * E <= I && R <= 16L * E;
    if (few && E <= 65535 && T_ * H * 2 <= stream::kMaxExtent && R * I * 2 <= stream::kMaxExtent)
        return run_ffn_few_rows<T>(x, w_gate, w_up, w_down, topw, order, inv_order, offsets, out, workspace, T_, E, k, H, I, s);
    return run_ffn_tiles<T>(x, w_gate, w_up, w_down, topw, order, inv_order, offsets, out, workspace, T_, E, k, H, I, s);
}

}  // namespace
}  // namespace paras

extern "C" {

size_t paras_moe_ffn_workspace(int64_t T, int64_t k, int64_t H, int64_t I, int dtype) {
    (void)dtype;
    if (T <= 0 || k <= 0 || H <= 0 || I <= 0) return 0;
    const size_t R = static_cast<size_t>(T) * k;
    return paras::align_up(R * I * 2, 256) + paras::align_up(R * H * 2, 256);
}

int paras_moe_ffn(const void* x, const void* w_gate, const void* w_up, const void* w_down, const float* topw,
                  const int64_t* order, const int64_t* inv_order, const int64_t* offsets, void* out,
                  void* workspace, int64_t T, int64_t E, int64_t k, int64_t H, int64_t I, int dtype, void* stream) {
    using namespace paras;
    PARAS_REQUIRE(T >= 0 && E >= 1 && k >= 1 && H >= 1 && I >= 1, "paras_moe_ffn: bad shape");
    if (T == 0) return PARAS_OK;
    PARAS_REQUIRE(dtype == PARAS_BF16 || dtype == PARAS_F16, "paras_moe_ffn: dtype must be bf16 or f16");
    PARAS_REQUIRE(x && w_gate && w_up && w_down && topw && order && inv_order && offsets && out && workspace,
                  "paras_moe_ffn: null pointer");
    // The MFMA tiles take hidden and intermediate sizes that are multiples of 64 and 16-byte aligned
    // tensors; anything else goes to the general kernels (any size, any alignment).
    const bool aligned = ((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(w_gate) | reinterpret_cast<uintptr_t>(w_up) |
                           reinterpret_cast<uintptr_t>(w_down) | reinterpret_cast<uintptr_t>(out) | reinterpret_cast<uintptr_t>(workspace)) & 15) == 0;
    const bool tiles = H % kBK == 0 && I % kBK == 0 && aligned && H < flex::kMaxLd && I < flex::kMaxLd;   // (the tiles' loads and stores use 32-bit byte offsets within a tile)
    PARAS_REQUIRE(T * k <= 0x3fffffffLL, "paras_moe_ffn: too many routed rows");
    if (T * H >= (1LL << 32) || T * k * I >= (1LL << 32) || I * H >= (1LL << 32))
        return fail(PARAS_ERR_UNSUPPORTED, "paras_moe_ffn: an operand (x, the routed intermediate, or one expert's weight matrix) spans 2^32 elements or more");
    hipStream_t s = nullptr;
    int rc = resolve_stream(stream, &s);
    if (rc != PARAS_OK) return rc;
    const long* ord = reinterpret_cast<const long*>(order);
    const long* inv = reinterpret_cast<const long*>(inv_order);
    const long* off = reinterpret_cast<const long*>(offsets);
    if (!tiles) {
        if (dtype == PARAS_BF16)
            return run_ffn_any<bf16_t>(x, w_gate, w_up, w_down, topw, ord, inv, off, out, workspace, T, (int)E, (int)k, H, I, s);
        return run_ffn_any<f16_t>(x, w_gate, w_up, w_down, topw, ord, inv, off, out, workspace, T, (int)E, (int)k, H, I, s);
    }
    if (dtype == PARAS_BF16)
        return run_ffn<bf16_t>(x, w_gate, w_up, w_down, topw, ord, inv, off, out, workspace, T, (int)E, (int)k, H, I, s);
    return run_ffn<f16_t>(x, w_gate, w_up, w_down, topw, ord, inv, off, out, workspace, T, (int)E, (int)k, H, I, s);
}

}  // extern "C"
