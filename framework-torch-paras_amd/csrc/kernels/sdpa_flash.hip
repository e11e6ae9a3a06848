// Flash-attention forward for gfx950 (bf16 / fp16 MFMA, fp32 accumulate).
//
// out = softmax(q k^T * scale [+ causal mask]) v, computed tile by tile with an
// online softmax; the [Lq, Lk] score matrix never exists in memory (the
// reference materialises it: csrc/ops/attention_ops.cpp:101,128).
//
// Work decomposition
//   workgroup = 4 wavefronts = 128 queries of one (batch, head); each wave owns
//   32 queries.  K/V are streamed in tiles of 64 keys through LDS (two buffers
//   each, one barrier per tile), shared by the 4 waves.  Tiles go from global
//   memory straight into LDS (buffer_load_dwordx4 ... lds: no staging registers,
//   no LDS store instructions; the buffer descriptor's range check supplies the
//   zeros for rows outside [0, Lk)); rows are unpadded and the 16-byte chunks of a
//   row are XOR-swizzled so that operand reads stay conflict free.
//
// The products are formed transposed so that a lane always owns ONE query:
//   S^T = K Q^T    A = K tile from LDS (lane: key l%32, 8 consecutive d),
//                  B = Q^T from registers (lane: query l%32, same 8 d)
//                  -> accumulator lane (query l%32, half h=l/32) holds, for a
//                  32-key block, keys (r/4)*8 + 4h + r%4, r = 0..15
//   row max / row sum: in-lane over the accumulator registers plus one
//                  v_permlane32_swap between the two half-waves
//   O^T = V^T P^T  B = P^T straight from the S^T accumulators (converted to
//                  16 bit, no shuffle: the accumulator's key order is simply
//                  used as the contraction order),
//                  A = V^T read from the row-major V tile with
//                  ds_read_b64_tr_b16, which transposes 4 keys x 16 d per
//                  16-lane group in the LDS crossbar
//   rescaling O by exp(m_old - m_new) is a per-lane scalar multiply, and it
//                  is lazy: the running max is only raised (and O, l rescaled)
//                  when a block's row max exceeds it by more than 2^8 in the
//                  exponent domain, so after the first block the rescale is
//                  skipped almost always; the same (possibly stale) max is used
//                  for P and for the row sum, so out = O / l is unchanged.
//   row sums       fp32 adds of the exponentials before they are rounded to the
//                  16-bit operand of the PV product
//
// Software pipeline inside a wave: the unit of work is a 32-key block and the
// score MFMAs run one block ahead,
//
//   block j:   [ S(j+1) = K(j+1) Q^T  MFMAs  |  exp / pack / row-sum of S(j) ]   one fenced schedule,
//              [ O^T += V(j)^T P(j)^T MFMAs  |  in-lane row max of S(j+1)    ]   an MFMA per slot
//              mask S(j+1) on the diagonal / at the end of K; raise the running max if needed (rare branch)
//
// so the matrix pipe has independent work in flight under the softmax VALU
// work of the same wave.  K is staged half a tile ahead of V: K tile u holds
// keys [64u-32, 64u+32) (tile 0 only 0 .. 31, in a buffer of its own), so the two blocks whose scores are computed during V
// tile t (blocks 2t+1, 2t+2) both live in K tile t+1, and K and V need only two
// LDS buffers each with a single barrier per tile.  The operand fragments run
// through a register ring that carries across the two blocks of a tile, and a
// tile's first fragments are requested before the next tile pair is.
//
// Three things in the structure exist to keep the compiler's wait insertion
// exact (it is conservative in ways that serialise this loop otherwise): the
// tiles come through buffer loads (an LDS-direct global load makes every later
// LDS wait a full one), each buffer is its own __shared__ array named at
// compile time in the main loop (an LDS read waits for all direct loads in
// flight unless the variables prove them disjoint), and nothing with a branch
// sits between a fragment's request and the MFMA that consumes it.
//
// An optional mask (bytes, nonzero = attend; or additive values of the tensor type;
// broadcast over any of batch / head / query, any stride along the keys) is applied
// to the finished scores of a block; the mask bytes of block j+1 are requested when
// block j starts.  Queries with no visible key so far carry a running maximum of
// -inf and contribute zeros; a query with no visible key at all ends as 0/0 = NaN,
// like the reference's softmax.
//
// A problem with fewer query tiles than CUs shares its keys out as well: two halves per workgroup or parts of the keys in
// workgroups of their own (plan_shares).
//
// v_mfma_f32_32x32x16_{bf16,f16}: 32 MFMAs per wave per 64-key tile at D=128.
#include <hip/hip_runtime.h>

#include <cmath>
#include <type_traits>

#include "core/device_context.h"
#include "core/device_math.h"
#include "core/status.h"
#include "kernels/sdpa_flash_common.h"
#include "kernels/sdpa_flash_deal.h"
#include "kernels/sdpa_internal.h"

namespace paras {
namespace {

using namespace flash;

constexpr int kBM = 128;   // queries per workgroup: 4 waves x 32

// Tiles of keys that the queries of a tile see.
template <bool kCausal>
__device__ __forceinline__ int tiles_of(const FlashParams& p, int qblock) {
    const int keys = kCausal ? min(min(qblock * kBM + kBM, p.Lq), p.Lk) : p.Lk;
    return (keys + kBN - 1) / kBN;
}

// The keys of (batch, head) up to the last one that a mask shared by all queries opens, to the next 16 or so; all of them if the
// mask is not of that kind or the row is so short that the look at it costs more than it saves (S91 D128 7.6 -> 7.9 us, S424 16.2 ->
// 15.6).  From the end of the row, 1024 bytes at a time.
__device__ __forceinline__ int open_keys(const FlashParams& p, int b, int hq, int lane) {
    if (p.ms_q != 0 || p.ms_k != 1 || p.Lk <= 256) return p.Lk;
    typedef u32x4 u32x4_any __attribute__((aligned(1)));
    const unsigned char* row = p.mask + static_cast<long>(b) * p.ms_b + static_cast<long>(hq) * p.ms_h;
    for (int k0 = (p.Lk - 1) / 1024 * 1024; k0 >= 0; k0 -= 1024) {
        const int at = k0 + 16 * lane;
        std::uint32_t any = 0;
        if (at < p.Lk) {
            const u32x4 w = *reinterpret_cast<const u32x4_any*>(row + min(at, p.Lk - 16));
            any = w[0] | w[1] | w[2] | w[3];
        }
        const unsigned long long lanes = __builtin_amdgcn_ballot_w64(any != 0);
        if (lanes != 0) return min(p.Lk, k0 + 16 * (64 - __builtin_clzll(lanes)));
    }
    return 0;
}

// Keys first .. last - 1 are closed to every query: their weights are 0, and so is their share of the outputs, but for the columns
// in which a value is an infinity or a NaN, since 0 times those is NaN.  All the workgroup's threads look (8 columns each); it has finished
// its tiles.  (What it saves is arithmetic, scores, narrowings and exponentials: with lengths from half to all of the longest, fp16 B6 H12
// S777 D64 26.7 -> 24.0 us, bf16 B13 H4 S1837 D128 134 -> 106, B4 H16 S5283 D64 738 -> 532, the same bits.)
template <typename T, int D, int DBLK, int kThreads>
__device__ __forceinline__ void close_columns(const FlashParams& p, const std::uint16_t* v, int first, int last, int* flags, int lh, float16_t (&oacc)[DBLK]) {
    constexpr std::uint32_t kExp = std::is_same<T, bf16_t>::value ? 0x7F807F80u : 0x7C007C00u, kUnit = std::is_same<T, bf16_t>::value ? 0x00800080u : 0x04000400u;
    constexpr int kChunks = D / 8, kRows = kThreads / kChunks;
    const int tid = threadIdx.x, col = tid % kChunks;
    const std::uint16_t* at = v + col * 8;
    u32x4 bad = {0, 0, 0, 0};
#pragma unroll 4
    for (int r = first + tid / kChunks; r < last; r += kRows) {
        const u32x4 w = *reinterpret_cast<const u32x4*>(at + static_cast<long>(r) * p.vs_l);
#pragma unroll
        for (int i = 0; i < 4; ++i) bad[i] |= (w[i] & kExp) + kUnit;       // an exponent of all ones carries into the sign's place
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) bad[i] &= 0x80008000u;
    if (__builtin_expect(__syncthreads_or((bad[0] | bad[1] | bad[2] | bad[3]) != 0), 0)) {
        for (int i = tid; i < D; i += kThreads) flags[i] = 0;
        __syncthreads();
#pragma unroll
        for (int i = 0; i < 8; ++i)
            if ((bad[i / 2] >> (16 * (i & 1) + 15)) & 1u) flags[col * 8 + i] = 1;
        __syncthreads();
#pragma unroll
        for (int db = 0; db < DBLK; ++db)
#pragma unroll
            for (int r = 0; r < 16; ++r)
                if (flags[db * 32 + (r >> 2) * 8 + 4 * lh + (r & 3)] != 0) oacc[db][r] = __builtin_nanf("");
        __syncthreads();                       // the flags' place may be written again
    }
}

// The weight of a share of the keys whose maximum is m beside one with M >= m.  A share in which the query saw no key counts
// with weight zero (and hands on a NaN that its values left there, as 0 x NaN does in the product).
__device__ __forceinline__ float weight_of(float m, float M, float scale_log2) {
    return m == -INFINITY ? 0.f : __builtin_amdgcn_exp2f((m - M) * scale_log2);
}

// One query's outputs from its lanes (half lh of the lanes holds, of each 32 columns, 8 g + 4 lh .. + 3) divided by the sum
// of its weights, and the logarithm of that sum where it is asked for; columns d0 .. d0 + 32 DBLK.
template <typename T, int D, int DBLK>
__device__ __forceinline__ void store_rows(const FlashParams& p, int b, int hq, int my_q, int lh, const float16_t (&oacc)[DBLK], float m, float l, int d0 = 0) {
    if (my_q >= p.Lq) return;
    const float inv_l = 1.0f / l;
    std::uint16_t* op = p.out + ((static_cast<long>(b) * p.Hq + hq) * p.Lq + my_q) * D + d0;
#pragma unroll
    for (int db = 0; db < DBLK; ++db)
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            const int d = db * 32 + g * 8 + 4 * lh;
            u32x2 w;
            w[0] = Mma<T>::pack2(oacc[db][4 * g + 0] * inv_l, oacc[db][4 * g + 1] * inv_l);
            w[1] = Mma<T>::pack2(oacc[db][4 * g + 2] * inv_l, oacc[db][4 * g + 3] * inv_l);
            *reinterpret_cast<u32x2*>(op + d) = w;
        }
    if (p.lse != nullptr && lh == 0) p.lse[(static_cast<long>(b) * p.Hq + hq) * p.Lq + my_q] = m * p.scale + logf(l);
}

// kMask: 0 none, 1 bytes (nonzero = attend), 2 additive values of type T.
// kHalves = 2: a workgroup is eight waves, four for the first half of the keys and four for the second, each half with tiles of its
// own; the second half's unnormalised outputs, maxima and sums reach the first through LDS at the end.
// kParts: the keys of a query tile are shared out to several workgroups, p.part_tiles tiles each, which leave their
// unnormalised outputs, maxima and sums to flash_combine_kernel.
// A wave sees its keys as keys 0 .. Lk - 1.
template <typename T, int D, bool kCausal, int kMask, bool kParts, int kHalves>
__global__ __launch_bounds__(256 * kHalves, (D > 128 || kHalves > 1 ? 1 : 2)) void flash_fwd_kernel(const FlashParams p) {
    static_assert(!(kCausal && kMask != 0), "a mask and the causal rule are mutually exclusive");
    // 32-query blocks per wave.  The code is written for any QB; 2 halves the LDS operand
    // traffic per query but needs one wave per SIMD and measured 30 % slower (nothing hides
    // LDS / barrier latency then), so 1 it is: two waves per SIMD, 256 registers each.
    constexpr int QB     = 1;
    constexpr int NW     = 4;
    constexpr int WQ     = 32 * QB;          // queries per wave
    static_assert(kBM == NW * WQ, "workgroup shape");
    constexpr int KSTEPS = D / 16;
    constexpr int DBLK   = D / 32;
    constexpr int CHUNKS = D / 8;
    constexpr int RPI    = 64 / CHUNKS;
    constexpr int NI     = kBN / (RPI * NW);
    auto ksw = [](int row) { return D >= 128 ? (row & 15) : ((row >> 1) & 7); };
    auto vsw = [](int row) { return D >= 128 ? ((row & 3) << 2) : (((row >> 1) & 1) << 2); };

    // LDS: two tiles each of K and V and the first half tile of K (72 KiB per workgroup at D = 128, two workgroups per
    // CU).  They are four separate arrays on purpose: the compiler makes an LDS read wait for
    // every direct-to-LDS load in flight unless it can prove from the variables involved that the
    // two do not overlap, and the point of the double buffer is to read one tile while the next
    // one streams in.  The main loop therefore names its buffers at compile time (`Par`), the
    // rarely taken paths pick them at run time (`AnyPar`) and accept the wait.
    __shared__ __attribute__((aligned(1024))) std::uint16_t k_lds0[kHalves * kBN * D];
    __shared__ __attribute__((aligned(1024))) std::uint16_t k_lds1[kHalves * kBN * D];
    __shared__ __attribute__((aligned(1024))) std::uint16_t v_lds0[kHalves * kBN * D];
    __shared__ __attribute__((aligned(1024))) std::uint16_t v_lds1[kHalves * kBN * D];
    // Keys 0..31, whose scores come before the loop.  (Not the upper half of K tile 0: K tile 2 is requested into that buffer
    // while another wave may still read them, and a barrier in between costs a problem of two tiles 5 %.)
    __shared__ __attribute__((aligned(1024))) std::uint16_t k_first[kHalves * 32 * D];
    using Par0 = std::integral_constant<int, 0>;
    using Par1 = std::integral_constant<int, 1>;
    struct AnyPar { int value; };
    const int tid = threadIdx.x, lane = tid & 63;
    const int half = kHalves == 1 ? 0 : __builtin_amdgcn_readfirstlane(tid >> 8);
    const int wave = __builtin_amdgcn_readfirstlane(kHalves == 1 ? tid >> 6 : (tid >> 6) & 3);      // within its half
    const int own = half * kBN * D;            // where this half's tiles are in the arrays
    // buffer of tile index parity `par`; `flip` selects the other one
    auto kbuf = [&](auto par, bool flip) -> std::uint16_t* {
        if constexpr (std::is_same<decltype(par), AnyPar>::value) return (((par.value ^ (flip ? 1 : 0)) & 1) ? k_lds1 : k_lds0) + own;
        else return ((decltype(par)::value != 0) != flip ? k_lds1 : k_lds0) + own;
    };
    auto vbuf = [&](auto par, bool flip) -> std::uint16_t* {
        if constexpr (std::is_same<decltype(par), AnyPar>::value) return (((par.value ^ (flip ? 1 : 0)) & 1) ? v_lds1 : v_lds0) + own;
        else return ((decltype(par)::value != 0) != flip ? v_lds1 : v_lds0) + own;
    };

    // (One fetch for all the arguments on the way to the first loads: left to itself the compiler fetches the pointers behind the
    // quotients, a second way to memory in front of everything: 11.9 us for 11.7.  Not with 256 elements, B2 H8 S6968 791 -> 796 us, nor where a
    // mask's arguments join them in parts of the keys, B2 H3 S2055 padded 29.1 -> 30.1.)
    if constexpr (kMask == 0 ? D <= 128 : !kParts)
        asm volatile("" ::"s"(p.q), "s"(p.k), "s"(p.v), "s"(p.rep), "s"(p.magic_group), "s"(p.magic_heads), "s"(p.magic_hq), "s"(p.magic_rep), "s"(p.head_group));
    if constexpr (kMask != 0 && !kParts) asm volatile("" ::"s"(p.mask), "s"(p.ms_b), "s"(p.ms_h), "s"(p.ms_q), "s"(p.ms_k));
    const int nq = p.n_qblocks;
    const int BH = p.B * p.Hq;
    int bh, qi;
    {
        const int idx = kParts ? blockIdx.x % (BH * nq) : blockIdx.x;
        if (BH % 8 == 0) {           // the heads are dealt to the XCDs, head_group at a time, longest query tiles first
            const int xcd = idx & 7, j = idx >> 3, G = p.head_group;
            const int g = quotient(j, G * nq, p.magic_group), r = j - g * G * nq;
            qi = quotient(r, G, p.magic_heads);
            bh = (g * G + r - qi * G) * 8 + xcd;
        } else if (kCausal) {        // the longest tiles of all heads first (B10 H1 S5121 D128: 102 -> 86 us; head by head the last heads' longest start late)
            qi = quotient(idx, BH, p.magic_group);
            bh = idx - qi * BH;
        } else {
            bh = quotient(idx, nq, p.magic_group);
            qi = idx - bh * nq;
        }
    }
    const int qblock = nq - 1 - qi;
    const int b = quotient(bh, p.Hq, p.magic_hq), hq = bh - b * p.Hq;
    int n_tiles = tiles_of<kCausal>(p, qblock);
    int first = 0;                             // this wave's first tile of keys
    const bool whole = !kParts || n_tiles <= p.part_tiles;
    const int part = kParts ? static_cast<int>(blockIdx.x) / (BH * nq) : 0;
    if constexpr (kParts) {
        first = part * p.part_tiles;
        if (first >= n_tiles) return;
        n_tiles = min(n_tiles - first, p.part_tiles);
    }
    // A key-padding mask: the tiles past the last open key of the sequence are left out of the loop (close_columns).  Not for
    // heads of 256: the registers it takes are spilled there (B14 H1 S117 13.9 -> 17.1 us, B1 H4 S2402 48 -> 55).
    constexpr bool kLeaveOut = kMask == 1 && D <= 128;
    int closed0 = 0, closed1 = 0;              // keys of this workgroup that are left out
    if constexpr (kLeaveOut) {
        const int open = max(min((open_keys(p, b, hq, lane) + kBN - 1) / kBN - first, n_tiles), 0);
        closed0 = (first + open) * kBN;
        closed1 = min(p.Lk, (first + n_tiles) * kBN);
        n_tiles = open;
    }
    const int turns = kHalves == 1 ? n_tiles : (n_tiles + 1) / 2;       // tiles between the workgroup's barriers
    if constexpr (kHalves == 2) {
        first += half * turns;
        n_tiles = half == 0 ? turns : n_tiles - turns;                  // (the second half of a single tile has none)
    }
    const int key0 = first * kBN;
    const int Lk = kParts || kHalves == 2 || kLeaveOut ? min(p.Lk - key0, n_tiles * kBN) : p.Lk;
    const int hkv = quotient(hq, p.rep, p.magic_rep);

    const int lq = lane & 31, lh = lane >> 5;
    const int q0 = qblock * kBM + wave * WQ;   // first query of this wave; query block qb starts at q0 + 32 qb
    const int q0k = q0 - key0;                 // the same, counted from this workgroup's first key (the causal rule)

    i16x8 qreg[QB][KSTEPS];
#pragma unroll
    for (int qb = 0; qb < QB; ++qb) {
        const int my_q = q0 + 32 * qb + lq;
        const int qrow = my_q < p.Lq ? my_q : p.Lq - 1;
        const std::uint16_t* qp = p.q + b * p.qs_b + hq * p.qs_h + static_cast<long>(qrow) * p.qs_l;
#pragma unroll
        for (int ks = 0; ks < KSTEPS; ++ks) qreg[qb][ks] = *reinterpret_cast<const i16x8*>(qp + ks * 16 + lh * 8);
    }

    const std::uint16_t* kbase = p.k + b * p.ks_b + hkv * p.ks_h + static_cast<long>(key0) * p.ks_l;
    const std::uint16_t* vbase = p.v + b * p.vs_b + hkv * p.vs_h + static_cast<long>(key0) * p.vs_l;
    // (keys may lie wholly beyond a wave's last query: no tiles, and zeros with a maximum of -inf)
    const int wave_tiles = !kCausal ? n_tiles : ((kParts || kHalves == 2) && q0k + WQ - 1 < 0 ? 0 : min(n_tiles, (q0k + WQ - 1) / kBN + 1));

    // ---- staging: 64 LDS rows <- global rows first .. first+63, straight from memory into LDS
    // with buffer loads.  The buffer descriptor spans rows [0, Lk) of this (batch, kv head), so
    // rows outside it (past the end of K in the last tiles)
    // arrive as zeros without a branch: the hardware range-checks every dword of every lane.
    const int srow = wave * RPI + lane / CHUNKS;
    const int slot = lane % CHUNKS;
    const int k_row_bytes = static_cast<int>(p.ks_l) * 2, v_row_bytes = static_cast<int>(p.vs_l) * 2;
    const int k_lane = srow * k_row_bytes + ((slot ^ ksw(srow)) * 16);
    const int v_lane = srow * v_row_bytes + ((slot ^ vsw(srow)) * 16);
    // Request i of a tile fills rows i * RPI * NW + srow.  That is a multiple of 16 rows further on
    // for heads of up to 128 elements, so the swizzle of the row is the swizzle of srow; with 256
    // elements a request covers 8 rows and every other one lands 8 rows on: bit 3 of the K swizzle flips.
    const int k_lane_odd = D > 128 ? srow * k_row_bytes + ((slot ^ ksw(srow + 8)) * 16) : k_lane;
    static_assert((RPI * NW) % 16 == 0 || (RPI * NW == 8 && D == 256), "the staging swizzle assumes whole groups of 16 (or 8) rows per request");
    typedef __attribute__((address_space(3))) void* lptr_t;
    auto make_rsrc = [&](const std::uint16_t* base, int row_bytes) {
        const int bytes = (kHalves == 2 || kLeaveOut) && Lk <= 0 ? 0 : (Lk - 1) * row_bytes + D * 2;           // < 2^31: checked by flash_supported
        return __builtin_amdgcn_make_buffer_rsrc(const_cast<std::uint16_t*>(base), 0, bytes, 0x00020000);
    };
    const __amdgpu_buffer_rsrc_t k_rsrc = make_rsrc(kbase, k_row_bytes);
    const __amdgpu_buffer_rsrc_t v_rsrc = make_rsrc(vbase, v_row_bytes);
    struct OfK {}; struct OfV {};
    auto stage_one = [&](__amdgpu_buffer_rsrc_t rsrc, auto which, int row_bytes, int first, std::uint16_t* tile, int i) {
        const int r0 = i * RPI * NW;
        constexpr bool is_k = std::is_same<decltype(which), OfK>::value;
        const int lane_off = is_k ? ((i & 1) ? k_lane_odd : k_lane) : v_lane;      // (i is a constant wherever this is called)
        // a negative offset is a huge unsigned one: out of range like the rows past the end
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (lptr_t)(tile + (r0 + wave * RPI) * D), 16,
                                                 lane_off + (first + r0) * row_bytes, 0, 0, 0);
    };
    auto stage_rows = [&](__amdgpu_buffer_rsrc_t rsrc, auto which, int row_bytes, int first, std::uint16_t* tile) {
#pragma unroll
        for (int i = 0; i < NI; ++i) stage_one(rsrc, which, row_bytes, first, tile, i);
    };
    // Requests the pair tile t's blocks need beyond K tile t: K tile t+1 and V tile t (`par` = parity of t).
    auto stage_pair = [&](int t, auto par) {
        stage_rows(k_rsrc, OfK{}, k_row_bytes, (t + 1) * kBN - 32, kbuf(par, true));
        stage_rows(v_rsrc, OfV{}, v_row_bytes, t * kBN, vbuf(par, false));
    };
    // Barrier that publishes every tile requested so far.
    auto publish = [&]() {
        // s_waitcnt simm16 on gfx9: vmcnt in bits 3:0 and 15:14, expcnt 6:4, lgkmcnt 11:8.  The
        // builtin (not inline asm) so that the compiler's own wait bookkeeping sees the loads retire.
        __builtin_amdgcn_s_waitcnt(0x0F70);
        __syncthreads();
    };

    float16_t oacc[QB][DBLK];
    float m_run[QB], l_run[QB];
#pragma unroll
    for (int qb = 0; qb < QB; ++qb) {
        m_run[qb] = -INFINITY;
        l_run[qb] = 0.f;
#pragma unroll
        for (int i = 0; i < DBLK; ++i)
#pragma unroll
            for (int r = 0; r < 16; ++r) oacc[qb][i][r] = 0.f;
    }

#pragma unroll
    for (int i = 0; i < NI / 2; ++i) stage_one(k_rsrc, OfK{}, k_row_bytes, 0, k_first + half * 32 * D, i);
    stage_pair(0, Par0{});
    publish();

    const int grp = lane >> 4, m16 = lane & 15;
    int k_rd[KSTEPS], v_rd[DBLK];
#pragma unroll
    for (int ks = 0; ks < KSTEPS; ++ks) k_rd[ks] = lq * D + (((2 * ks + lh) ^ ksw(lq)) * 8);
    {
        const int vrow = 4 * lh + (m16 >> 2);
#pragma unroll
        for (int db = 0; db < DBLK; ++db)
            v_rd[db] = vrow * D + (((4 * db + 2 * (grp & 1) + ((m16 & 3) >> 1)) ^ vsw(vrow)) * 8) + 4 * (m16 & 1);
    }
    const float lazy_margin = 8.0f / p.scale_log2;

    auto needs_mask = [&](int j, int qb) { return (kCausal && j * 32 + 31 > q0k + 32 * qb) || j * 32 + 32 > Lk; };
    auto apply_mask = [&](int j, int qb, float16_t& sc) {
        const int my_q = q0k + 32 * qb + lq;
        const int last_visible = kCausal ? min(my_q, Lk - 1) : Lk - 1;
        const int rel = last_visible - j * 32 - 4 * lh;
#pragma unroll
        for (int r = 0; r < 16; ++r)
            if ((r >> 2) * 8 + (r & 3) > rel) sc[r] = -INFINITY;
    };
    // ---- optional user mask.  Lane (query, half lh) needs, for block j, keys j*32 + 8g + 4 lh + i
    // (g, i = 0..3; accumulator register 4g + i): four runs of four consecutive keys.  The runs of
    // block j+1 are requested at the start of block j and applied when its scores are finished.
    constexpr int MREGS = kMask == 0 ? 1 : (kMask == 1 ? 4 : 8);
    const unsigned char* mrow = nullptr;
    if constexpr (kMask != 0) {
        const int my_q = q0 + lq;
        const long qrow = my_q < p.Lq ? my_q : p.Lq - 1;
        mrow = p.mask + (static_cast<long>(b) * p.ms_b + static_cast<long>(hq) * p.ms_h + qrow * p.ms_q + key0 * p.ms_k) * (kMask == 1 ? 1 : 2);
    }
    // A mask that is contiguous along the keys, with Lk >= 4: a run that hangs over the end of the
    // row is read from the row's last four elements and shifted down, so no load leaves the row and
    // no branch is needed; keys >= Lk get zero bits and are masked by the end-of-K rule.  Any other
    // stride along the keys (0: a view that broadcasts one value per query over the keys; > 1: slices
    // and transposed views) is read element by element into the same registers -- sixteen small
    // loads per block instead of four, requested a block ahead like the runs.
    //   A block that lies wholly inside a contiguous row is not read as four runs per lane (a wavefront's
    // 64 lanes then touch 64 different places four times over) but as one 16-byte piece per lane of
    // the block's 32 (bool) or 64 (additive: two pieces) bytes of its query's row: half lh holds keys
    // 16 lh .. 16 lh + 15 and needs keys 8 g + 4 lh .. + 3, so the two halves of a query swap every
    // other run when the mask is applied (v_permlane32_swap: lanes l and l + 32).
    const bool mask_runs = p.ms_k == 1 && Lk >= 4;       // uniform
    auto mask_whole_block = [&](int j) { return mask_runs && j * 32 + 32 <= Lk; };      // uniform
    auto mask_load = [&](int j, std::uint32_t (&mr)[MREGS]) {
        if constexpr (kMask != 0) {
            typedef std::uint32_t u32_any __attribute__((aligned(1)));
            typedef u32x4 u32x4_any __attribute__((aligned(1)));
            if (mask_whole_block(j)) {
                constexpr int ES = kMask == 1 ? 1 : 2;
                const unsigned char* at = mrow + (j * 32 + 16 * lh) * ES;
#pragma unroll
                for (int h = 0; h < ES; ++h) {
                    const u32x4 w = *reinterpret_cast<const u32x4_any*>(at + 16 * h);
#pragma unroll
                    for (int i = 0; i < 4; ++i) mr[4 * h + i] = w[i];
                }
                return;
            }
            if (!mask_runs) {
                constexpr int ES = kMask == 1 ? 1 : 2;
#pragma unroll
                for (int g = 0; g < 4; ++g) {
                    std::uint32_t e[4];
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        const int key = min(j * 32 + 8 * g + 4 * lh + i, Lk - 1);   // (keys past the end: any value, the end-of-K rule masks them)
                        const unsigned char* at = mrow + static_cast<long>(key) * p.ms_k * ES;
                        if constexpr (kMask == 1) e[i] = *at;
                        else                      e[i] = *reinterpret_cast<const std::uint16_t*>(at);
                    }
                    if constexpr (kMask == 1) {
                        mr[g] = e[0] | (e[1] << 8) | (e[2] << 16) | (e[3] << 24);
                    } else {
                        mr[2 * g] = e[0] | (e[1] << 16);
                        mr[2 * g + 1] = e[2] | (e[3] << 16);
                    }
                }
                return;
            }
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                const int key = j * 32 + 8 * g + 4 * lh;
                const int at = min(key, Lk - 4);
                const unsigned sh = static_cast<unsigned>(key - at);          // 0 unless the run hangs over
                if constexpr (kMask == 1) {
                    const std::uint32_t w = *reinterpret_cast<const u32_any*>(mrow + at);
                    mr[g] = sh < 4 ? w >> (8 * sh) : 0u;
                } else {
                    const std::uint64_t w = static_cast<std::uint64_t>(*reinterpret_cast<const u32_any*>(mrow + 2 * at)) |
                                            (static_cast<std::uint64_t>(*reinterpret_cast<const u32_any*>(mrow + 2 * at + 4)) << 32);
                    const std::uint64_t v = sh < 4 ? w >> (16 * sh) : 0ull;
                    mr[2 * g] = static_cast<std::uint32_t>(v);
                    mr[2 * g + 1] = static_cast<std::uint32_t>(v >> 32);
                }
            }
        }
    };
    // With a mask the scores are narrowed where the host engine narrows them (attention_ops.cpp:101-128:
    // the product, the scaled product and the sum with an additive mask are tensors of T): a row that
    // sees few keys is decided by one or two scores, and a 2^-9 step on one of them is several per cent
    // on its weight.  The scores leave here scaled; the kernel's scale is 1 in these variants.
    auto round_T = [](float x) { return Elem<T>::to_f32(Elem<T>::from_f32_finite(x)); };
    // A block's scores narrowed, scaled and narrowed, two at a time.  fp16: with a scale that is itself an fp16 number the
    // product of two such numbers is exact in fp32, so the fp16 multiplication rounds the same value once.  (fp16 B6 H12 S777
    // D64, key-padding mask 29.9 -> 26.4 us, the same bits; the kernel is bound by the arithmetic per score.)
    const bool scale_is_T = std::is_same<T, f16_t>::value && static_cast<float>(static_cast<_Float16>(p.score_scale)) == p.score_scale;   // uniform
    auto narrow_and_scale = [&](float16_t& sc) {
        if constexpr (std::is_same<T, bf16_t>::value) {
            auto halves = [](std::uint32_t w, float& lo, float& hi) {
                lo = __builtin_bit_cast(float, w << 16);
                hi = __builtin_bit_cast(float, w & 0xFFFF0000u);
            };
#pragma unroll
            for (int r = 0; r < 16; r += 2) {
                float lo, hi;
                halves(Mma<T>::pack2(sc[r], sc[r + 1]), lo, hi);
                halves(Mma<T>::pack2(lo * p.score_scale, hi * p.score_scale), lo, hi);
                sc[r] = lo;
                sc[r + 1] = hi;
            }
        } else if (scale_is_T) {
            typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
            const _Float16 k = static_cast<_Float16>(p.score_scale);
#pragma unroll
            for (int r = 0; r < 16; r += 2) {
                const f16x2 v = f16x2{static_cast<_Float16>(sc[r]), static_cast<_Float16>(sc[r + 1])} * f16x2{k, k};
                sc[r] = static_cast<float>(v[0]);
                sc[r + 1] = static_cast<float>(v[1]);
            }
        } else {
#pragma unroll
            for (int r = 0; r < 16; ++r) sc[r] = round_T(round_T(sc[r]) * p.score_scale);
        }
    };
    auto mask_apply = [&](int j, const std::uint32_t (&loaded)[MREGS], float16_t& sc) {
        std::uint32_t mr[MREGS];
#pragma unroll
        for (int i = 0; i < MREGS; ++i) mr[i] = loaded[i];
        if constexpr (kMask == 1) {
            // Every key of the block open to every query of the wave, as in all but the last blocks of a row under a
            // key-padding mask: nothing to swap and nothing to select (fp16 B6 H12 S777 D64 30.8 -> 29.9 us).
            if (mask_whole_block(j) && __builtin_amdgcn_ballot_w64((mr[0] & mr[1] & mr[2] & mr[3]) != 0x01010101u) == 0) {
                narrow_and_scale(sc);
                return;
            }
        }
        if constexpr (kMask != 0) {
            if (mask_whole_block(j)) {
                // registers as loaded: the lane's own sixteen keys.  Lower half: keeps its runs 0 and 2 (bool:
                // one register each; additive: two), gets runs 0 and 2 of the upper half for its runs 1 and 3.
                auto swap = [&](int x, int y) {       // upper half of register x <-> lower half of register y
                    const auto r = __builtin_amdgcn_permlane32_swap(mr[x], mr[y], false, false);
                    mr[x] = r[0];
                    mr[y] = r[1];
                };
                if constexpr (kMask == 1) {
                    swap(0, 1);
                    swap(2, 3);
                    const std::uint32_t t = mr[1];    // runs in order: registers 0, 2, 1, 3
                    mr[1] = mr[2];
                    mr[2] = t;
                } else {
                    swap(0, 2);
                    swap(1, 3);
                    swap(4, 6);
                    swap(5, 7);
                    const std::uint32_t t2 = mr[2], t3 = mr[3];     // runs in order: registers (0,1), (4,5), (2,3), (6,7)
                    mr[2] = mr[4];
                    mr[3] = mr[5];
                    mr[4] = t2;
                    mr[5] = t3;
                }
            }
            narrow_and_scale(sc);
        }
        if constexpr (kMask == 1) {
#pragma unroll
            for (int r = 0; r < 16; ++r)
                if (((mr[r >> 2] >> (8 * (r & 3))) & 0xffu) == 0) sc[r] = -INFINITY;
        } else if constexpr (kMask == 2) {
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const std::uint16_t bits = static_cast<std::uint16_t>(mr[r >> 1] >> (16 * (r & 1)));
                sc[r] = round_T(sc[r] + Elem<T>::to_f32(bits));
            }
        }
    };
    auto lane_max = [](const float16_t& sc) {
        float mx = sc[0];
#pragma unroll
        for (int r = 1; r < 16; ++r) mx = fmaxf(mx, sc[r]);
        return mx;
    };
    // Raise the running max of query block qb if block max `mx` (this lane's half) needs it.  The
    // test runs on each lane's own half of the keys; the two halves of a query are only brought
    // together inside the rare branch.
    auto raise_max = [&](float (&mx)[QB]) {
        // (the compare builtin hands back the wavefront's lane mask as it stands; a bool fed to the
        // ballot builtin is first turned into 0 / 1 per lane and compared again)
        unsigned long long grow = 0;
#pragma unroll
        for (int qb = 0; qb < QB; ++qb) grow |= __builtin_amdgcn_fcmpf(mx[qb], m_run[qb] + lazy_margin, 2 /* ordered greater than */);
        if (__builtin_expect(grow != 0, 0)) {  // wave-uniform, rare after block 0: the common path falls through
#pragma unroll
            for (int qb = 0; qb < QB; ++qb) {
                const float m_new = fmaxf(m_run[qb], half_swap_max(mx[qb]));
                // (equal covers -inf on both sides: a query that has seen no key yet keeps its zeros)
                const float alpha = m_run[qb] == m_new ? 1.f : __builtin_amdgcn_exp2f((m_run[qb] - m_new) * p.scale_log2);
                m_run[qb] = m_new;
                l_run[qb] *= alpha;
#pragma unroll
                for (int i = 0; i < DBLK; ++i)
#pragma unroll
                    for (int r = 0; r < 16; ++r) oacc[qb][i][r] *= alpha;
            }
        }
    };
    // Mask where needed, then raise.  `mx` holds the unmasked in-lane maxima on entry.
    auto finish_scores = [&](int j, float16_t (&sc)[QB], float (&mx)[QB], const std::uint32_t (&mr)[MREGS]) {
#pragma unroll
        for (int qb = 0; qb < QB; ++qb) {
            if constexpr (kMask != 0) mask_apply(j, mr, sc[qb]);
            if (__builtin_expect(needs_mask(j, qb), 0)) apply_mask(j, qb, sc[qb]);
            if (kMask != 0 || needs_mask(j, qb)) mx[qb] = lane_max(sc[qb]);
        }
        raise_max(mx);
    };

    // One block: exponentials of `cur` = S(j) and, if kNext, the MFMAs of S(j+1) into `nxt`,
    // then PV(j).  The MFMA part is a fixed schedule of KSTEPS + 2*DBLK slots (QB MFMAs per
    // slot, sharing one LDS fragment), fenced so that the compiler keeps the order.  Fragment
    // reads run two slots ahead through a ring of four registers that lives across blocks: a
    // block expects the operands of its first two slots in flight and, in its last two slots,
    // requests those of its successor (`tail`: KFirst = a block that starts with score MFMAs,
    // VFirst = one that only has PV left, NoTail = the successor's rows are not resident yet).
    // The 8*QB exp pairs (2 fma + 2 exp + cvt + 2 add each) are spread between the MFMAs so the
    // matrix pipe has an instruction in flight while the VALU works.  P(s2=0) is complete
    // before the first PV MFMA, P(s2=1) before the first PV MFMA that uses it; the row maxima
    // of S(j+1) are reduced as a tree in the slots after the last exp pair, so the rescale
    // decision is ready when the last MFMA issues.
    i16x8 frag[4];
    constexpr int NS = KSTEPS + 2 * DBLK;                 // slot c >= KSTEPS: PV(s2 = (c-KSTEPS)/DBLK, db = (c-KSTEPS)%DBLK)
    static_assert(NS % 4 == 0 && KSTEPS % 4 == 0, "the fragment ring is indexed by slot % 4 across blocks");
    // `par` is the parity of block j's tile (j >> 1): V(j) lives in the V buffer of that parity,
    // the K rows of block j+1 in the K buffer of the other one.
    auto fetch = [&](int j, int c, auto par) {            // operand of slot c of block j -> frag[c % 4]
        if (c < KSTEPS) {
            const std::uint16_t* kt = kbuf(par, true) + ((j + 2) & 1) * 32 * D;   // rows of block j+1
            frag[c % 4] = *reinterpret_cast<const i16x8*>(kt + k_rd[c]);
        } else {
            const std::uint16_t* vt = vbuf(par, false) + (j & 1) * 32 * D;
            const int s2 = (c - KSTEPS) / DBLK, db = (c - KSTEPS) % DBLK;
            const std::uint16_t* vp = vt + v_rd[db] + 16 * s2 * D;
            const i16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4*)(vp));
            const i16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4*)(vp + 8 * D));
            frag[c % 4] = i16x8{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
        }
    };
    struct KFirst {}; struct VFirst {}; struct NoTail {};
    auto first_fetches = [&](int j, auto kind, auto par) {   // what block j's first two slots consume
        constexpr int s0 = std::is_same<decltype(kind), KFirst>::value ? 0 : KSTEPS;
        fetch(j, s0, par);
        fetch(j, s0 + 1, par);
    };
    auto block = [&](int j, float16_t (&cur)[QB], float16_t (&nxt)[QB], auto next_tag, auto tail, auto par, auto stage_tag) {
        constexpr bool kNext = decltype(next_tag)::value;
        constexpr bool kStage = decltype(stage_tag)::value;
        constexpr bool kTail = !std::is_same<decltype(tail), NoTail>::value;
        constexpr int S0 = kNext ? 0 : KSTEPS;           // first slot that exists
        static_assert(QB == 1, "the max tree below is written for one query block per wave");
        float mc[QB];
#pragma unroll
        for (int qb = 0; qb < QB; ++qb) {
            mc[qb] = m_run[qb] * p.scale_log2;
            // every key so far masked out: the reference point is arbitrary, and it must not be -inf
            if constexpr (kMask != 0) mc[qb] = m_run[qb] == -INFINITY ? 0.f : mc[qb];
        }
        std::uint32_t mnext[MREGS];
        if constexpr (kNext) mask_load(j + 1, mnext);
        u32x4 pw[QB][2];
        float mx[QB], t3[5], t2[2];
        auto exp_pair = [&](int qb, int i) {              // elements 2i, 2i+1 of cur[qb]
            const float e0 = __builtin_amdgcn_exp2f(fmaf(cur[qb][2 * i], p.scale_log2, -mc[qb]));
            const float e1 = __builtin_amdgcn_exp2f(fmaf(cur[qb][2 * i + 1], p.scale_log2, -mc[qb]));
            const std::uint32_t w = Mma<T>::pack2(e0, e1);
            // Plain adds of the unrounded exponentials: v_dot2_f32_bf16 on the packed pair is one
            // instruction instead of two, but it runs on the matrix pipe's side and stalls the
            // MFMA next to it (measured: 4 % of the kernel).
            l_run[qb] += e0 + e1;
            asm volatile("" : "+v"(l_run[qb]));           // keeps the row-sum update in this slot
            pw[qb][i / 4][i % 4] = w;
        };
        // pair (qb, i) is issued just before the MFMAs of slot pair_slot(qb, i)
        auto pair_slot = [](int qb, int i) {
            if (i < 4) return kNext ? (qb * 4 + i) * KSTEPS / (4 * QB) : KSTEPS;
            return KSTEPS + (qb * 4 + i - 4) * DBLK / (4 * QB);
        };
        constexpr int MAX0 = KSTEPS + DBLK + (DBLK >= 4 ? 1 : 0);   // after the last exp pair; S(j+1) finished KSTEPS slots ago

#pragma unroll
        for (int c = S0; c < NS; ++c) {
#pragma unroll
            for (int qb = 0; qb < QB; ++qb)
#pragma unroll
                for (int i = 0; i < 8; ++i)
                    if (pair_slot(qb, i) == c) exp_pair(qb, i);
            if (c < KSTEPS) {
#pragma unroll
                for (int qb = 0; qb < QB; ++qb) {
                    if (c == 0) {
#pragma unroll
                        for (int r = 0; r < 16; ++r) nxt[qb][r] = 0.f;
                    }
                    nxt[qb] = Mma<T>::run(frag[c % 4], qreg[qb][c], nxt[qb]);
                }
            } else {
                const int s2 = (c - KSTEPS) / DBLK, db = (c - KSTEPS) % DBLK;
#pragma unroll
                for (int qb = 0; qb < QB; ++qb)
                    oacc[qb][db] = Mma<T>::run(frag[c % 4], __builtin_bit_cast(i16x8, pw[qb][s2]), oacc[qb][db]);
            }
            if constexpr (kStage) {
                // The next tile pair (K tile t+2, V tile t+1), one request every other slot: all of
                // them at the start of the tile, from every wave at once right after the barrier,
                // cost 1.5 % (they queue up in front of the waves' first MFMAs).
                static_assert(2 * (2 * NI - 1) < NS, "the requests fit the block's slots");
                if (c % 2 == 0 && c / 2 < 2 * NI) {
                    const int i = c / 2, t = j >> 1;
                    if (i < NI) stage_one(k_rsrc, OfK{}, k_row_bytes, (t + 2) * kBN - 32, kbuf(par, false), i);
                    else        stage_one(v_rsrc, OfV{}, v_row_bytes, (t + 1) * kBN, vbuf(par, true), i - NI);
                }
            }
            if (c + 2 < NS) fetch(j, c + 2, par);
            else if constexpr (kTail)    // only ever the second block of the same tile: same parity
                fetch(j + 1, (std::is_same<decltype(tail), KFirst>::value ? 0 : KSTEPS) + (c + 2 - NS), par);
            if constexpr (kNext && kMask == 0) {      // (with a user mask the maxima are taken after masking)
                const float16_t& sv = nxt[0];
                if (c == MAX0) {
#pragma unroll
                    for (int g = 0; g < 5; ++g) {
                        t3[g] = fmaxf(fmaxf(sv[3 * g], sv[3 * g + 1]), sv[3 * g + 2]);
                        asm volatile("" : "+v"(t3[g]));   // keeps the reduction in this slot
                    }
                }
                if (c == MAX0 + 1) {
                    t2[0] = fmaxf(fmaxf(t3[0], t3[1]), t3[2]);
                    t2[1] = fmaxf(fmaxf(t3[3], t3[4]), sv[15]);
                    mx[0] = fmaxf(t2[0], t2[1]);
                    asm volatile("" : "+v"(mx[0]));
                }
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        if constexpr (kNext) finish_scores(j + 1, nxt, mx, mnext);
    };
    using Yes = std::true_type;
    using No  = std::false_type;

    float16_t s_a[QB], s_b[QB];
    if (wave_tiles > 0) {
        // S(0): keys 0..31
        float mx[QB];
#pragma unroll
        for (int qb = 0; qb < QB; ++qb) {
#pragma unroll
            for (int r = 0; r < 16; ++r) s_a[qb][r] = 0.f;
#pragma unroll
            for (int ks = 0; ks < KSTEPS; ++ks)
                s_a[qb] = Mma<T>::run(*reinterpret_cast<const i16x8*>(&k_first[half * 32 * D + k_rd[ks]]), qreg[qb][ks], s_a[qb]);
            mx[qb] = lane_max(s_a[qb]);
        }
        std::uint32_t m0[MREGS];
        mask_load(0, m0);
        finish_scores(0, s_a, mx, m0);
    }
    // One tile of the main loop (`par` = parity of t, a compile-time name for the buffers; two
    // tiles per trip).  The tile's first block also requests the next tile pair (= stage_pair(t + 1)).
    auto tile = [&](int t, auto par) {
        first_fetches(2 * t, KFirst{}, par);
        __builtin_amdgcn_sched_barrier(0);                // keep the reads ahead of the requests
        block(2 * t, s_a, s_b, Yes{}, KFirst{}, par, Yes{});
        block(2 * t + 1, s_b, s_a, Yes{}, NoTail{}, par, No{}); // its successor's K rows arrive with the barrier below
        publish();
    };
    int t_main = 0;
    for (; t_main + 2 < wave_tiles; t_main += 2) {
        tile(t_main, Par0{});
        tile(t_main + 1, Par1{});
    }
    if (t_main + 1 < wave_tiles) {
        tile(t_main, Par0{});
        ++t_main;
    }
    if (wave_tiles > 0) {  // the wave's last tile: nothing to compute ahead in its second block
        const int t = wave_tiles - 1;
        const AnyPar par{t};
        if (t + 1 < n_tiles) stage_pair(t + 1, AnyPar{t + 1});
        // The tile's second block contributes nothing when it starts past the end of K or, for a
        // causal wave, past the wave's last query (every other wave's diagonal tile).
        const int second0 = (2 * t + 1) * 32;
        if (second0 >= Lk || (kCausal && second0 > q0k + WQ - 1)) {
            first_fetches(2 * t, VFirst{}, par);
            block(2 * t, s_a, s_b, No{}, NoTail{}, par, No{});
        } else {
            first_fetches(2 * t, KFirst{}, par);
            block(2 * t, s_a, s_b, Yes{}, VFirst{}, par, No{});
            block(2 * t + 1, s_b, s_a, No{}, NoTail{}, par, No{});
        }
        publish();
    }
    for (int t = wave_tiles; t < turns; ++t) {             // done early (causal): keep staging for the other waves
        if (t + 1 < n_tiles) stage_pair(t + 1, AnyPar{t + 1});
        publish();
    }

    if constexpr (kLeaveOut) {
        if (closed0 < closed1) close_columns<T, D, DBLK, 256 * kHalves>(p, p.v + b * p.vs_b + hkv * p.vs_h, closed0, closed1, reinterpret_cast<int*>(k_first), lh, oacc[0]);
    }
    float l_tot[QB];
#pragma unroll
    for (int qb = 0; qb < QB; ++qb) l_tot[qb] = half_swap_sum(l_run[qb]);
    if constexpr (kHalves == 2) {
        static_assert(QB == 1 && kHalves * kBN * D * 2 >= DBLK * 4 * 64 * 16, "a wave's outputs fit one of the arrays, whose tiles are done with");
        __shared__ float ml[NW][2][64];
        std::uint16_t* const mine = wave == 0 ? k_lds0 : (wave == 1 ? k_lds1 : (wave == 2 ? v_lds0 : v_lds1));
        float4_t* const po = reinterpret_cast<float4_t*>(mine) + lane;
        if (half == 1) {
#pragma unroll
            for (int i = 0; i < DBLK * 4; ++i)
                po[i * 64] = float4_t{oacc[0][i / 4][4 * (i % 4)], oacc[0][i / 4][4 * (i % 4) + 1], oacc[0][i / 4][4 * (i % 4) + 2], oacc[0][i / 4][4 * (i % 4) + 3]};
            ml[wave][0][lane] = m_run[0];
            ml[wave][1][lane] = l_tot[0];
        }
        __syncthreads();
        if (half == 1) return;
        const float m1 = ml[wave][0][lane], l1 = ml[wave][1][lane], M = fmaxf(m_run[0], m1);
        const float f0 = weight_of(m_run[0], M, p.scale_log2), f1 = weight_of(m1, M, p.scale_log2);
#pragma unroll
        for (int i = 0; i < DBLK * 4; ++i) {
            const float4_t v = po[i * 64];
#pragma unroll
            for (int r = 0; r < 4; ++r) oacc[0][i / 4][4 * (i % 4) + r] = fmaf(f1, v[r], f0 * oacc[0][i / 4][4 * (i % 4) + r]);
        }
        l_tot[0] = fmaf(f1, l1, f0 * l_tot[0]);
        m_run[0] = M;
    }
    if constexpr (kParts) {
        if (!whole) {
            static_assert(QB == 1, "one query block per wave in a slot");
            const long slot = (static_cast<long>(bh) * nq + qblock) * p.n_parts + part;
            float4_t* po = reinterpret_cast<float4_t*>(p.part_o) + (slot * NW + wave) * (DBLK * 4 * 64) + lane;
#pragma unroll
            for (int i = 0; i < DBLK * 4; ++i)
                po[i * 64] = float4_t{oacc[0][i / 4][4 * (i % 4)], oacc[0][i / 4][4 * (i % 4) + 1], oacc[0][i / 4][4 * (i % 4) + 2], oacc[0][i / 4][4 * (i % 4) + 3]};
            float* ml = p.part_ml + (slot * NW + wave) * 64;
            ml[lane] = lh == 0 ? m_run[0] : l_tot[0];
            return;
        }
    }
#pragma unroll
    for (int qb = 0; qb < QB; ++qb) store_rows<T, D, DBLK>(p, b, hq, q0 + 32 * qb + lq, lh, oacc[qb], m_run[qb], l_tot[qb]);
}

// The parts of a query tile brought together: O = sum of exp(m_s - M) O_s over sum of exp(m_s - M) l_s, in part order.
// A workgroup takes 32 columns of a tile's 128 queries, lane for lane as the parts were stored.
template <typename T, int D, bool kCausal>
__global__ __launch_bounds__(256) void flash_combine_kernel(const FlashParams p) {
    constexpr int DBLK = D / 32, NW = 4, kAhead = 4;
    const int tile = blockIdx.x / DBLK, db = blockIdx.x % DBLK;
    const int bh = tile / p.n_qblocks, qblock = tile % p.n_qblocks;
    const int parts = (tiles_of<kCausal>(p, qblock) + p.part_tiles - 1) / p.part_tiles;
    if (parts <= 1) return;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, lq = lane & 31, lh = lane >> 5;
    const long slot = static_cast<long>(tile) * p.n_parts;
    const float* ml = p.part_ml + (slot * NW + wave) * 64;
    const float4_t* po = reinterpret_cast<const float4_t*>(p.part_o) + (slot * NW + wave) * (DBLK * 4 * 64) + db * 256 + lane;
    float M = -INFINITY;
#pragma unroll 8
    for (int s = 0; s < parts; ++s) M = fmaxf(M, ml[s * (NW * 64) + lq]);
    float L = 0.f;
    float16_t o;
#pragma unroll
    for (int r = 0; r < 16; ++r) o[r] = 0.f;
    for (int s0 = 0; s0 < parts; s0 += kAhead) {        // four parts in flight
        float4_t v[kAhead][4];
        float m[kAhead], l[kAhead];
#pragma unroll
        for (int u = 0; u < kAhead; ++u) {
            const int s = min(s0 + u, parts - 1);
            m[u] = ml[s * (NW * 64) + lq];
            l[u] = ml[s * (NW * 64) + 32 + lq];
#pragma unroll
            for (int g = 0; g < 4; ++g) v[u][g] = po[static_cast<long>(s) * (NW * DBLK * 4 * 64) + g * 64];
        }
#pragma unroll
        for (int u = 0; u < kAhead; ++u) {
            if (s0 + u >= parts) break;
            const float f = weight_of(m[u], M, p.scale_log2);
            L = fmaf(f, l[u], L);
#pragma unroll
            for (int g = 0; g < 4; ++g)
#pragma unroll
                for (int r = 0; r < 4; ++r) o[4 * g + r] = fmaf(f, v[u][g][r], o[4 * g + r]);
        }
    }
    const int b = bh / p.Hq, hq = bh % p.Hq;
    const float16_t oacc[1] = {o};
    FlashParams q = p;
    if (db != 0) q.lse = nullptr;                       // (one workgroup of the tile writes it)
    store_rows<T, D, 1>(q, b, hq, qblock * kBM + wave * 32 + lq, lh, oacc, M, L, db * 32);
}

template <typename T, int D, bool kParts, int kHalves>
void launch_mask(const FlashParams& p, bool causal, int mask_kind, hipStream_t s) {
    const dim3 grid(static_cast<unsigned>(static_cast<long>(p.B) * p.Hq * p.n_qblocks * (kParts ? p.n_parts : 1))), wg(256 * kHalves);
    if (causal)              hipLaunchKernelGGL((flash_fwd_kernel<T, D, true, 0, kParts, kHalves>), grid, wg, 0, s, p);
    else if (mask_kind == 1) hipLaunchKernelGGL((flash_fwd_kernel<T, D, false, 1, kParts, kHalves>), grid, wg, 0, s, p);
    else if (mask_kind == 2) hipLaunchKernelGGL((flash_fwd_kernel<T, D, false, 2, kParts, kHalves>), grid, wg, 0, s, p);
    else                     hipLaunchKernelGGL((flash_fwd_kernel<T, D, false, 0, kParts, kHalves>), grid, wg, 0, s, p);
}

template <typename T, int D>
int launch_t(FlashParams p, bool causal, int mask_kind, bool halves, hipStream_t s) {
    constexpr int kHalves = D > 128 ? 1 : 2;           // (the tiles of two halves of 256-element heads do not fit LDS)
    p.n_qblocks = (p.Lq + kBM - 1) / kBM;
    const long BH = static_cast<long>(p.B) * p.Hq;
    p.head_group = BH % 16 == 0 ? 2 : 1;
    if (causal && BH % 8 == 0) p.head_group = static_cast<int>(heads_together(BH / 8, p.n_qblocks, p.Lk, D));
    p.magic_group = magic_of(BH % 8 == 0 ? static_cast<long>(p.head_group) * p.n_qblocks : causal ? BH : p.n_qblocks);
    p.magic_heads = magic_of(p.head_group);
    p.magic_hq = magic_of(p.Hq);
    p.rep = p.Hq / p.Hkv;
    p.magic_rep = magic_of(p.rep);
    if (p.n_parts <= 1) {
        if (halves) launch_mask<T, D, false, kHalves>(p, causal, mask_kind, s);
        else        launch_mask<T, D, false, 1>(p, causal, mask_kind, s);
    } else {
        launch_mask<T, D, true, 1>(p, causal, mask_kind, s);
        PARAS_HIP_TRY(hipGetLastError());
        const dim3 grid(static_cast<unsigned>(static_cast<long>(p.B) * p.Hq * p.n_qblocks * (D / 32)));
        if (causal) hipLaunchKernelGGL((flash_combine_kernel<T, D, true>), grid, dim3(256), 0, s, p);
        else        hipLaunchKernelGGL((flash_combine_kernel<T, D, false>), grid, dim3(256), 0, s, p);
    }
    PARAS_HIP_TRY(hipGetLastError());
    return PARAS_OK;
}

bool aligned16(const void* ptr) { return (reinterpret_cast<uintptr_t>(ptr) & 15) == 0; }
bool mult8(const int64_t* strides) { return strides[0] % 8 == 0 && strides[1] % 8 == 0 && strides[2] % 8 == 0; }

}  // namespace

bool flash_supported(const paras_sdpa_args& a) {
    if (a.dtype != PARAS_BF16 && a.dtype != PARAS_F16) return false;
    if (a.D != a.Dv || (a.D != 64 && a.D != 128 && a.D != 256)) return false;
    if (a.attn != nullptr) return false;                            // the weights are never formed here
    if (a.mask_kind != 0 && (a.mask == nullptr || a.is_causal)) return false;
    if (a.mask_kind < 0 || a.mask_kind > 2) return false;
    if (a.mask_kind != 0 && a.mask_strides[3] < 0) return false;
    if (a.Lq < 1 || a.Lk < 1) return false;
    if (!(a.scale > 0.0) || !std::isfinite(a.scale)) return false;  // the running max is taken on raw scores
    if (!aligned16(a.q) || !aligned16(a.k) || !aligned16(a.v) || !aligned16(a.out)) return false;
    if (!mult8(a.q_strides) || !mult8(a.k_strides) || !mult8(a.v_strides)) return false;
    const int64_t nq = (a.Lq + kBM - 1) / kBM;
    if (a.B * a.Hq * nq > 0x7fffffffLL || a.Lq > 0x3fffffff || a.Lk > 0x3fffffff) return false;
    // K / V tiles are fetched with 32-bit byte offsets against a buffer descriptor per (batch, head)
    // that spans rows [0, Lk); offsets of rows up to one tile outside it must not wrap into it.
    for (const int64_t* st : {a.k_strides, a.v_strides}) {
        if (st[2] < 0) return false;
        if ((a.Lk + 2 * kBN) * st[2] * 2 + a.D * 2 >= 0x7fffffffLL) return false;
    }
    return true;
}

namespace {

// How the keys of a problem with few query tiles are shared out (launch_flash).  A workgroup of four waves uses a CU's arithmetic
// to the full, so nothing is gained where every CU has one; the rule trades idle CUs against the parts' way through memory.
//   Parts: up to 128 query tiles (head size 256: any number), as many parts as give every CU one (causal: 320 in all, half of which
// have keys), four tiles of keys at least (two), if the tiles a workgroup is spared, in us, are more than the second
// kernel's 4.5 us and the parts' way out and in.  In bf16 and fp16, B1 H2 S4393 D64: none 43.8 -> 24.9, causal 50.0 -> 23.4, key-padding
// mask 89 -> 34; D128 59 -> 36, 64 -> 28, 115 -> 47; D256 B1 H2 S2000 56 -> 29, 59 -> 29, 74 -> 34.  (B2 H8 S963, 128 tiles, D128 none: 18.5
// whole, 25.7 in two parts.)  Of 150 drawn problems that it shares out none is slower than whole, 1.70 times as fast in the mean; the nearest
// to the line: fp16 D128 none B1 H4 S1050 19.1 -> 18.5, D256 additive B1 H8 S824 37.3 -> 36.2, causal D64 B5 H1 S868 13.5 -> 12.6.
//   Halves within a workgroup, D <= 128: two waves per SIMD help where a wave waits or works outside the matrix cores, and under the causal
// rule they shorten the last tiles; without mask and rule they cost as much as they give.  B12 H1 S1499 D64, mask 35.3 -> 27.0; B3 H4 S2377
// D128, mask 63 -> 56; B1 H8 S8192 D128, causal 159 -> 137; B1 H32 S512 D64, mask 13.9 -> 12.7, D128, causal 13.4 -> 14.9 (eight
// tiles: whole).
struct Shares {
    int  parts = 1, part_tiles = 0;
    bool halves = false;
};
Shares plan_shares(const paras_sdpa_args& a) {
    Shares r;
    const bool causal = a.is_causal != 0, masked = a.mask_kind != 0;
    const long W = static_cast<long>(a.B * a.Hq) * ((a.Lq + kBM - 1) / kBM);
    const long tiles = ((causal && a.Lq < a.Lk ? a.Lq : a.Lk) + kBN - 1) / kBN;      // of the query tile that sees the most
    const long least = a.D > 128 ? 2 : 4;
    if (W < 1 || W > 512 || tiles <= least) return r;
    const double tile_us = a.D == 64 ? (masked ? 1.15 : causal ? 0.65 : 0.6) : a.D == 128 ? (masked ? 1.45 : 0.85) : (masked ? 2.6 : causal ? 1.55 : 1.65);
    const long parts = (causal ? 320 : 256) / W;
    if (parts > 1 && (W <= 128 || a.D > 128)) {
        const long t = (tiles + parts - 1) / parts > least ? (tiles + parts - 1) / parts : least, n = (tiles + t - 1) / t;
        if (n > 1 && tile_us * (tiles - t) > 4.5 + static_cast<double>(W * n * a.D) / (causal ? 8000 : 4000)) {
            r.parts = static_cast<int>(n);
            r.part_tiles = static_cast<int>(t);
            return r;
        }
    }
    r.halves = a.D <= 128 && ((masked && W <= 256 && tiles >= 8) || (causal && ((W <= 256 && tiles >= 12) || (W <= 512 && tiles >= 24))));
    return r;
}

}  // namespace

size_t flash_workspace(const paras_sdpa_args& a) {
    const Shares r = plan_shares(a);
    if (r.parts <= 1 || flash_uses_wide(a)) return 0;
    const size_t slots = static_cast<size_t>(a.B * a.Hq) * ((a.Lq + kBM - 1) / kBM) * r.parts;
    return slots * (kBM * a.D + 2 * kBM) * sizeof(float);
}

static int wide_group_of(const paras_sdpa_args& a) {
    return flash::wide_group(a.B, a.Hq, a.Hkv, a.Lq, a.Lk, static_cast<int>(a.D), a.mask_kind, a.is_causal != 0);
}

bool flash_uses_wide(const paras_sdpa_args& a) { return wide_group_of(a) != 0; }

int launch_flash(const paras_sdpa_args& a, Scratch scratch, hipStream_t s) {
    FlashParams p{};
    p.q = static_cast<const std::uint16_t*>(a.q);
    p.k = static_cast<const std::uint16_t*>(a.k);
    p.v = static_cast<const std::uint16_t*>(a.v);
    p.out = static_cast<std::uint16_t*>(a.out);
    p.lse = a.lse;
    p.qs_b = a.q_strides[0]; p.qs_h = a.q_strides[1]; p.qs_l = a.q_strides[2];
    p.ks_b = a.k_strides[0]; p.ks_h = a.k_strides[1]; p.ks_l = a.k_strides[2];
    p.vs_b = a.v_strides[0]; p.vs_h = a.v_strides[1]; p.vs_l = a.v_strides[2];
    p.B = static_cast<int>(a.B); p.Hq = static_cast<int>(a.Hq); p.Hkv = static_cast<int>(a.Hkv);
    p.Lq = static_cast<int>(a.Lq); p.Lk = static_cast<int>(a.Lk);
    p.n_qblocks = 0;  // set by the launcher for the workgroup size it picks
    p.scale = static_cast<float>(a.scale);
    p.scale_log2 = static_cast<float>(a.scale * 1.4426950408889634);
    p.mask = static_cast<const unsigned char*>(a.mask);
    p.ms_b = a.mask_strides[0]; p.ms_h = a.mask_strides[1]; p.ms_q = a.mask_strides[2]; p.ms_k = a.mask_strides[3];
    p.score_scale = static_cast<float>(a.scale);
    if (a.mask_kind != 0) {          // the masked variants scale the scores themselves, between two narrowings
        p.scale = 1.0f;
        p.scale_log2 = 1.4426950408889634f;
    }
    const bool causal = a.is_causal != 0;
    const int mk = a.mask_kind;
    const Shares r = plan_shares(a);
    if (r.parts > 1 && scratch.has(flash_workspace(a)) && aligned16(scratch.p)) {
        p.n_parts = r.parts;
        p.part_tiles = r.part_tiles;
        p.part_o = static_cast<float*>(scratch.p);
        p.part_ml = p.part_o + static_cast<size_t>(a.B * a.Hq) * ((a.Lq + kBM - 1) / kBM) * r.parts * kBM * a.D;
    }
    if (const int group = wide_group_of(a); group != 0) return launch_flash_wide(p, group, causal, a.dtype == PARAS_BF16, s);
    if (a.dtype == PARAS_BF16)
        return a.D == 256 ? launch_t<bf16_t, 256>(p, causal, mk, r.halves, s) : a.D == 128 ? launch_t<bf16_t, 128>(p, causal, mk, r.halves, s) : launch_t<bf16_t, 64>(p, causal, mk, r.halves, s);
    return a.D == 256 ? launch_t<f16_t, 256>(p, causal, mk, r.halves, s) : a.D == 128 ? launch_t<f16_t, 128>(p, causal, mk, r.halves, s) : launch_t<f16_t, 64>(p, causal, mk, r.halves, s);
}

}  // namespace paras
