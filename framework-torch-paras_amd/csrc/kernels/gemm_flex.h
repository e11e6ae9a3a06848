// Tile mainloop of the 16-bit products whose operands may lie either way round:
// C tile = op(A) op(B)^T with fp32 accumulation on v_mfma_f32_16x16x32.
//
// An operand is a set of `rows` (rows of C for A, columns of C for B) times the contraction.  It is
// either contiguous along the contraction ("K", what x W^T has) or contiguous along its rows ("R":
// the weight of an input gradient, both operands of a weight gradient).  A "K" tile sits in LDS as
// [row][64] and a fragment is one 16-byte read; an "R" tile sits as [64][rows], as it lies in memory,
// and a fragment is two ds_read_b64_tr_b16 (the transposing LDS read: a group of 16 lanes reads 4
// contraction steps x 16 rows and each lane receives the 4 steps of its row).  Transposing at the LDS
// read instead of in memory saves a whole pass over each such operand.
//
// A workgroup is four waves, 2 x 2, one per SIMD at the large tiles; a wave computes MI x NJ blocks of
// 16 x 16, so the tile is 32 MI x 32 NJ.  Tiles of 64 contraction steps go from memory straight to LDS
// (buffer_load ... lds), ST stages: no staging registers, no LDS stores, nothing in the loop but
// MFMAs, LDS reads and one request per few MFMAs, which is what a single wave per SIMD can issue in the
// shadow of its MFMAs.  One barrier per tile, before its last k-step: by then all of the tile's
// fragments are in registers, so its stage can be requested anew right away, for the tile ST further on, and has
// ST - 1 tiles' time to arrive, while the k-step's MFMAs run and the next tile's first fragments are read.
//
// What bounds it is the number of stages where a CU holds one or two workgroups of small tiles: a tile of 64 x 64 is 512
// cycles of MFMA and LDS work, and its operands are 1500 cycles away.  Waits are for the next tile's requests only, the later ones stay
// in flight (64 x 128 tiles, x W^T in bf16, two stages -> four: 1500 x 1024 x 4096 29.6 -> 23.1 us, 2040 x 1024 x 3584 29.5 -> 22.1,
// 232 x 7168 x 2048 25.6 -> 17.8; 192 x 128, three
// stages: 1500 x 4096 x 4096 60.8 -> 50.2; four: with the weights from HBM 53.2 -> 52.0).  256-row tiles fill LDS with two stages and are
// bound by the matrix cores' power.
//
// Direct loads fill LDS in lane order, so rows cannot be padded apart; instead the 16-byte chunks of a
// row (K) or the 32-byte units (R) are permuted by a function of the row, applied to the address a
// lane fetches from and again where fragments are read, so that the lanes of one LDS access phase hit
// distinct banks.  Loads are checked against the exact extent of the operand by the buffer unit: rows
// past its end and contraction steps past K come back as zeros without a branch.
#pragma once

#include <hip/hip_runtime.h>

#include <type_traits>

#include "core/device_math.h"
#include "kernels/gemm_tile.h"

namespace paras {
namespace flex {

using gemm::i16x8;
typedef float float4v __attribute__((ext_vector_type(4)));

// acc += b a, in place in the accumulation registers.  Written out because the compiler, given the
// builtin, moves the 256 accumulators of the large tile from register to register on their way round the
// loop (120 to 350 moves and some spills per 128 MFMAs).  Nothing here needs the wait states it would
// insert: fragments come from LDS (a wait on the counter covers them), the next MFMA on the same
// accumulator is a k-step away, and the loop ends with a pause before the accumulators are read.
template <typename T> __device__ __forceinline__ void mma(float4v& acc, i16x8 b, i16x8 a);
template <> __device__ __forceinline__ void mma<bf16_t>(float4v& acc, i16x8 b, i16x8 a) {
    asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(acc) : "v"(b), "v"(a));
}
template <> __device__ __forceinline__ void mma<f16_t>(float4v& acc, i16x8 b, i16x8 a) {
    asm volatile("v_mfma_f32_16x16x32_f16 %0, %1, %2, %0" : "+a"(acc) : "v"(b), "v"(a));
}

constexpr int kThreads = 256;
constexpr int kBK = 64;
constexpr std::uint32_t kOutOfRange = 0xF0000000u;       // a byte offset beyond any buffer extent used here
constexpr long kMaxExtent = 0xE0000000L;
constexpr long kMaxLd = 1L << 22;                        // elements: a tile's offsets stay far below kMaxExtent

__device__ __forceinline__ int wave_id() { return __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) >> 6); }

// One operand as a workgroup fetches and reads it: W requests per wave and tile.
template <int W, bool R> struct Operand {
    static constexpr int kRows = 32 * W;
    static constexpr int kElems = kRows * kBK;
    static constexpr int kBases = R ? (W >= 4 ? 4 : W) : 2;     // lane offsets of fragment reads
    const char* base;             // (first row of the tile, first contraction step of the part); uniform
    long left;                    // bytes from there to the end of the operand; uniform
    long step;                    // bytes from a tile to the next
    std::uint32_t off[W];         // this lane's chunk of each request
    int fb[kBases];

    // 32-byte unit `u` of contraction step k of an R tile sits at unit u ^ unit_swizzle(k)
    __device__ static __forceinline__ int unit_swizzle(int k) { return W >= 2 ? (k & 3) : ((k >> 1) & 1); }

    __device__ __forceinline__ void init(const std::uint16_t* p, long ld, long rows, long row0, long k_first, long k_count, int w) {
        const int lane = threadIdx.x & 63, l16 = lane & 15, kq = lane >> 4;
        if constexpr (R) {
            base = reinterpret_cast<const char*>(p + k_first * ld + row0);
            left = ((k_count - 1) * ld + (rows - row0)) * 2;
            step = kBK * ld * 2;
#pragma unroll
            for (int i = 0; i < W; ++i) {
                const int c = (i * 4 + wave_id()) * 64 + lane;
                const int k = c / (4 * W), slot = c % (4 * W);
                off[i] = static_cast<std::uint32_t>(k * ld * 2 + (slot ^ (unit_swizzle(k) << 1)) * 16);
            }
            const int k = kq * 8 + (l16 >> 2);
#pragma unroll
            for (int b = 0; b < kBases; ++b) fb[b] = k * kRows + ((w * W + b) ^ unit_swizzle(k)) * 16 + 4 * (l16 & 3);
        } else {
            base = reinterpret_cast<const char*>(p + row0 * ld + k_first);
            left = ((rows - row0 - 1) * ld + k_count) * 2;
            step = kBK * 2;
#pragma unroll
            for (int i = 0; i < W; ++i)
                off[i] = static_cast<std::uint32_t>(((i * 4 + wave_id()) * 8 + (lane >> 3)) * ld * 2 + ((lane & 7) ^ (lane >> 3)) * 16);
#pragma unroll
            for (int ks = 0; ks < 2; ++ks) fb[ks] = (w * 16 * W + l16) * kBK + ((ks * 4 + kq) ^ (l16 & 7)) * 8;
        }
    }
    // From now on only the last tile is requested: its contraction steps past the end are not to be
    // fetched (K: they are the next row's; R: the extent ends there anyway).
    __device__ __forceinline__ void last_tile(int k_in_tile) {
        if constexpr (!R) {
            const int lane = threadIdx.x & 63;
            const std::uint32_t gone = ((lane & 7) ^ (lane >> 3)) * 8 < k_in_tile ? 0u : kOutOfRange;
#pragma unroll
            for (int i = 0; i < W; ++i) off[i] |= gone;
        }
    }
    __device__ __forceinline__ __amdgpu_buffer_rsrc_t rsrc(int kt, int k_tiles) const {
        const long l = left - kt * step;
        const long n = l < 0 || kt >= k_tiles ? 0 : (l > kMaxExtent ? kMaxExtent : l);
        return __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(base + kt * step), 0, static_cast<int>(static_cast<std::uint32_t>(n)), 0x00020000);
    }
    __device__ __forceinline__ void request(__amdgpu_buffer_rsrc_t r, std::uint16_t* tile, int i) const {
        typedef __attribute__((address_space(3))) void* lds_ptr;
        __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (lds_ptr)(tile + (i * 4 + wave_id()) * 512), 16, static_cast<int>(off[i]), 0, 0, 0);
    }
    __device__ __forceinline__ i16x8 frag(const std::uint16_t* tile, int blk, int ks) const {
        if constexpr (R) {
            typedef __attribute__((address_space(3))) i16x4 lds_i16x4;
            const std::uint16_t* q = tile + fb[blk % kBases] + (blk / kBases) * kBases * 16 + ks * 32 * kRows;
            const i16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4*)(q));
            const i16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4*)(q + 4 * kRows));
            return i16x8{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
        } else {
            return *reinterpret_cast<const i16x8*>(&tile[fb[ks] + blk * 16 * kBK]);
        }
    }
};

// Waits for all but `n` of this wave's loads in flight and for its LDS reads, and meets the others.
template <int n> __device__ __forceinline__ void meet() {
    __builtin_amdgcn_s_waitcnt(0x0070 | (n & 15) | ((n >> 4) << 14));     // vmcnt(n) lgkmcnt(0)
    asm volatile("s_barrier" ::: "memory");     // (a fence of the compiler's own would wait for every direct load in flight)
}

// mainloop (below) for the largest tiles, whose two stages fill LDS.  Requests for a tile can go out once its stage is read, and with both operands
// freed together that is one k-step out of two: a request per four MFMAs there, none in the other, and what comes from HBM instead of the last-level cache is
// late.  Here B's fragments of both k-steps are read in the k-step before the tile, each into the registers that its predecessor has
// just been multiplied from, so B's stage is free a k-step earlier than A's: B is requested in the first k-step and A in the second, a
// request per eight MFMAs throughout.  It is the even pace that counts: with the same waits and distances but four MFMAs between requests it is slower than with one
// barrier.  bf16, x W^T, 256 x 256 tiles, one barrier and this: 4096 x 4096 x 4096 with its operands in HBM 103.8 and 97.8 us, 16384 x 4096 x 4096 401 and 385,
// 8192 x 4096 x 16384 805 and 738, 8192^3 753 and 733; with everything in the caches level (4096^3 94.4 and 94.0).
template <typename T, int MI, int NJ, typename OA, typename OB>
__device__ __forceinline__ void mainloop_paced(OA& oa, OB& ob, int k_count, std::uint16_t* const (&sa)[2], std::uint16_t* const (&sb)[2],
                                               float4v (&acc)[MI][NJ]) {
    constexpr int S = MI * NJ;          // MFMAs per k-step
    i16x8 af[2][MI], bf[2][NJ];
    const int k_tiles = (k_count + kBK - 1) / kBK;
    auto request_all = [&](int kt, std::uint16_t* ta, std::uint16_t* tb) {
        if (kt == k_tiles - 1) {
            oa.last_tile(k_count - kt * kBK);
            ob.last_tile(k_count - kt * kBK);
        }
        const auto ra = oa.rsrc(kt, k_tiles);
        const auto rb = ob.rsrc(kt, k_tiles);
#pragma unroll
        for (int c = 0; c < NJ; ++c) ob.request(rb, tb, c);
#pragma unroll
        for (int c = 0; c < MI; ++c) oa.request(ra, ta, c);
    };
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j) acc[i][j] = float4v{0.f, 0.f, 0.f, 0.f};
    auto pin = [&] {          // orders the accumulators' other uses against the written-out MFMAs
#pragma unroll
        for (int i = 0; i < MI; ++i)
#pragma unroll
            for (int j = 0; j < NJ; ++j) asm volatile("" : "+a"(acc[i][j]));
    };
    pin();
    constexpr int kFree = 2 * MI;       // MFMAs into a tile until its last fragment of B, asked for at its start, is there in every wave
    auto tile = [&](int kt, std::uint16_t* ca, std::uint16_t* cb, std::uint16_t* na, std::uint16_t* nb) {
        if (kt + 2 == k_tiles - 1) {
            oa.last_tile(k_count - (kt + 2) * kBK);
            ob.last_tile(k_count - (kt + 2) * kBK);
        }
        const auto ra = oa.rsrc(kt + 2, k_tiles);
        const auto rb = ob.rsrc(kt + 2, k_tiles);
#pragma unroll
        for (int j = 0; j < NJ; ++j)
#pragma unroll
            for (int i = 0; i < MI; ++i) {
                const int slot = j * MI + i;
                if (slot == kFree) {
                    __builtin_amdgcn_s_waitcnt(0xC07F);         // lgkmcnt(0): the loads stay in flight
                    asm volatile("s_barrier" ::: "memory");
                }
                mma<T>(acc[i][j], bf[0][j], af[0][i]);
                if (slot == MI / 2) bf[1][NJ - 1] = ob.frag(cb, NJ - 1, 1);
#pragma unroll
                for (int c = 0; c < MI; ++c)
                    if (kFree + (c * (S - kFree) * 7) / (8 * MI) == slot) af[1][c] = oa.frag(ca, c, 1);
#pragma unroll
                for (int c = 0; c < NJ; ++c)
                    if (kFree + 2 + (c * (S - kFree - 2)) / NJ == slot) ob.request(rb, cb, c);
                __builtin_amdgcn_sched_barrier(0);
            }
        meet<NJ>();                     // the next tile has landed, A's stage is read; B's requests are on their way
#pragma unroll
        for (int j = 0; j < NJ; ++j)
#pragma unroll
            for (int i = 0; i < MI; ++i) {
                const int slot = j * MI + i;
                mma<T>(acc[i][j], bf[1][j], af[1][i]);
#pragma unroll
                for (int c = 0; c < MI + NJ; ++c)
                    if ((c * S * 7) / (8 * (MI + NJ)) == slot) {
                        if (c < NJ) bf[0][c] = ob.frag(nb, c, 0);
                        else        af[0][c - NJ] = oa.frag(na, c - NJ, 0);
                    }
                if (i == MI / 2 && j > 0) bf[1][j - 1] = ob.frag(nb, j - 1, 1);
#pragma unroll
                for (int c = 0; c < MI; ++c)
                    if ((c * S) / MI == slot) oa.request(ra, ca, c);
                __builtin_amdgcn_sched_barrier(0);
            }
    };
    request_all(0, sa[0], sb[0]);
    request_all(1, sa[1], sb[1]);
    meet<MI + NJ>();
#pragma unroll
    for (int f = 0; f < NJ; ++f) {
        bf[0][f] = ob.frag(sb[0], f, 0);
        if (f < NJ - 1) bf[1][f] = ob.frag(sb[0], f, 1);
    }
#pragma unroll
    for (int f = 0; f < MI; ++f) af[0][f] = oa.frag(sa[0], f, 0);
    // (In whole turns of the stages, with one way out: a tile past the last one multiplies cleared stages.)
    for (int kt = 0; kt < k_tiles; kt += 2) {
        tile(kt, sa[0], sb[0], sa[1], sb[1]);
        tile(kt + 1, sa[1], sb[1], sa[0], sb[0]);
    }
    asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");      // the last products are on their way to the registers the epilogue reads
    pin();
    __builtin_amdgcn_s_waitcnt(0x0F70);         // vmcnt(0): no request may outlive the workgroup's LDS
}

// acc[i][j]: the B fragment is the instruction's first operand, so lane (l16 = lane % 16, kq = lane / 16)
// holds row i*16 + l16 of the wave's rows and columns j*16 + 4*kq .. + 3 of its columns.
// (The ST stages are separate arrays named at compile time: an LDS read waits for every direct load in flight
// that the compiler cannot prove to go elsewhere.)
// OA, OB: Operand or a type with its rsrc / request / frag / last_tile.
template <typename T, int MI, int NJ, int ST, typename OA, typename OB>
__device__ __forceinline__ void mainloop(OA& oa, OB& ob, int k_count, std::uint16_t* const (&sa)[ST], std::uint16_t* const (&sb)[ST],
                                         float4v (&acc)[MI][NJ]) {
    if constexpr (ST == 2 && MI >= 6 && NJ >= 7) {
        mainloop_paced<T, MI, NJ>(oa, ob, k_count, sa, sb, acc);
        return;
    }
    constexpr int C = MI + NJ;          // requests per wave and tile, and fragments per k-step
    constexpr int S = MI * NJ;          // MFMAs per k-step
    static_assert(ST >= 2 && (ST - 1) * C < 64, "the tiles in flight have to fit the load counter");
    i16x8 af[2][MI], bf[2][NJ];
    const int k_tiles = (k_count + kBK - 1) / kBK;
    auto request_one = [&](const auto& ra, const auto& rb, std::uint16_t* ta, std::uint16_t* tb, int c) {
        if (c < MI) oa.request(ra, ta, c);
        else        ob.request(rb, tb, c - MI);
    };
    auto request_all = [&](int kt, std::uint16_t* ta, std::uint16_t* tb) {
        if (kt == k_tiles - 1) {
            oa.last_tile(k_count - kt * kBK);
            ob.last_tile(k_count - kt * kBK);
        }
        const auto ra = oa.rsrc(kt, k_tiles);
        const auto rb = ob.rsrc(kt, k_tiles);
#pragma unroll
        for (int c = 0; c < C; ++c) request_one(ra, rb, ta, tb, c);
    };
    auto read_frag = [&](const std::uint16_t* ta, const std::uint16_t* tb, int buf, int f, int ks) {
        if (f < MI) af[buf][f] = oa.frag(ta, f, ks);
        else        bf[buf][f - MI] = ob.frag(tb, f - MI, ks);
    };
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j) acc[i][j] = float4v{0.f, 0.f, 0.f, 0.f};
    auto pin = [&] {          // orders the accumulators' other uses against the written-out MFMAs
#pragma unroll
        for (int i = 0; i < MI; ++i)
#pragma unroll
            for (int j = 0; j < NJ; ++j) asm volatile("" : "+a"(acc[i][j]));
    };
    pin();
    // The requests for the next tile that goes into this stage are spread over the whole k-step that follows the barrier: bunched into
    // its first half they come at twice the rate the CU's L1 takes them and hold up the MFMAs (8192^3 807 against
    // 774 us), spread further into the next k-step the last of them are late at the barrier (788 us).
    // Tile kt from stage (ca, cb); the next one is in (na, nb).  One body for every tile, the last ones included:
    // a copy of it for them costs the accumulators their places (hundreds of spills), so requests past the end
    // go to an empty extent, which fetches nothing and clears the stage.
    auto tile = [&](int kt, std::uint16_t* ca, std::uint16_t* cb, std::uint16_t* na, std::uint16_t* nb) {
        if (kt + ST == k_tiles - 1) {
            oa.last_tile(k_count - (kt + ST) * kBK);
            ob.last_tile(k_count - (kt + ST) * kBK);
        }
        const auto ra = oa.rsrc(kt + ST, k_tiles);
        const auto rb = ob.rsrc(kt + ST, k_tiles);
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) {
            if (ks == 1) meet<(ST - 2) * C>();         // this wave's part of the next tile has landed, its reads of this one are done
#pragma unroll
            for (int j = 0; j < NJ; ++j)
#pragma unroll
                for (int i = 0; i < MI; ++i) {
                    const int slot = j * MI + i;
                    mma<T>(acc[i][j], bf[ks][j], af[ks][i]);
#pragma unroll
                    for (int c = 0; c < C; ++c) {
                        if ((c * S * 7) / (8 * C) == slot) read_frag(ks == 0 ? ca : na, ks == 0 ? cb : nb, ks ^ 1, c, ks ^ 1);
                        if (ks == 1 && (c * S) / C == slot) request_one(ra, rb, ca, cb, c);
                    }
                    __builtin_amdgcn_sched_barrier(0);
                }
        }
    };
#pragma unroll
    for (int u = 0; u < ST; ++u) request_all(u, sa[u], sb[u]);
    meet<(ST - 1) * C>();
#pragma unroll
    for (int f = 0; f < C; ++f) read_frag(sa[0], sb[0], 0, f, 0);
    // (In whole turns of the stages, with one way out: tiles past the last one multiply cleared stages.)
    for (int kt = 0; kt < k_tiles; kt += ST) {
#pragma unroll
        for (int u = 0; u < ST; ++u) tile(kt + u, sa[u], sb[u], sa[(u + 1) % ST], sb[(u + 1) % ST]);
    }
    asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");      // the last products are on their way to the registers the epilogue reads
    pin();
    __builtin_amdgcn_s_waitcnt(0x0F70);         // vmcnt(0): no request may outlive the workgroup's LDS
}

// The results' way out.  A lane holds four columns of 16 rows apart per block: stored from there a wave's store is 16 pieces of 32 bytes, and
// a tile's stores come all at once, from every CU in the same few us, with nothing beside them on a CU that holds one workgroup.  So each wave lays its
// rows, narrowed, into one of the stages that nobody reads any more and stores them from there in whole rows, 16 bytes a lane.
// `kChunks` 16-byte pieces a row, in an order turned by the row (16 rows apart by a power of two would be one bank).
typedef __attribute__((address_space(3))) std::uint16_t lds_u16;
typedef __attribute__((address_space(3))) u32x2 lds_u32x2;
typedef __attribute__((address_space(3))) u32x4 lds_u32x4;
template <int NJ> struct RowsOut {
    static constexpr int kChunks = 2 * NJ;
    __device__ static __forceinline__ int place(int row, int chunk) { return (chunk + (row & 15)) % kChunks; }
    // columns 4*kq .. + 3 of block j of `row`
    __device__ static __forceinline__ int at(int row, int j, int kq) { return row * (16 * NJ) + place(row, 2 * j + (kq >> 1)) * 8 + (kq & 1) * 4; }
    __device__ static __forceinline__ void lay(lds_u16* out, int row, int j, int kq, u32x2 v) { *(lds_u32x2*)(out + at(row, j, kq)) = v; }
    __device__ static __forceinline__ u32x4 piece(lds_u16* out, int row, int chunk) {
        return *(lds_u32x4*)(out + row * (16 * NJ) + place(row, chunk) * 8);
    }
};

// Rows of a wave, laid out by RowsOut, to memory: `dst` is its first row and column, `rows` x `cols` of it exist (<= 0: none), in rows of `ld` elements.
// `wide`: those are whole aligned 16-byte pieces.  `nan_here`: NaNs may be among them.
template <typename T, int MI, int NJ>
__device__ __forceinline__ void store_rows(lds_u16* out, std::uint16_t* dst, long ld, long rows, long cols, bool wide, bool nan_here) {
    using Out = RowsOut<NJ>;
    constexpr int kAll = 16 * MI * Out::kChunks, kTurns = (kAll + 63) / 64;
    constexpr int kAhead = kTurns % 8 == 0 ? 8 : kTurns % 7 == 0 ? 7 : kTurns % 6 == 0 ? 6 : kTurns % 5 == 0 ? 5 : kTurns % 4 == 0 ? 4 : 1;
    const int lane = threadIdx.x & 63;
    lds_exchange_in_wave();
    if (wide && !nan_here && rows >= 16 * MI && cols >= 16 * NJ) {
#pragma unroll 1
        for (int t = 0; t < kTurns; t += kAhead) {
            u32x4 v[kAhead];
#pragma unroll
            for (int u = 0; u < kAhead; ++u) {
                const int c = (t + u) * 64 + lane;
                v[u] = Out::piece(out, c / Out::kChunks, c % Out::kChunks);
            }
#pragma unroll
            for (int u = 0; u < kAhead; ++u) {
                const int c = (t + u) * 64 + lane;
                if (kAll % 64 == 0 || c < kAll) *reinterpret_cast<u32x4*>(dst + (c / Out::kChunks) * ld + (c % Out::kChunks) * 8) = v[u];
            }
        }
        return;
    }
#pragma unroll 1
    for (int t = 0; t < kTurns; ++t) {
        const int c = t * 64 + lane, row = c / Out::kChunks, col = (c % Out::kChunks) * 8;
        if (c >= kAll || row >= rows || col >= cols) continue;
        u32x4 v = Out::piece(out, row, c % Out::kChunks);
        if (nan_here) {
#pragma unroll
            for (int u = 0; u < 4; ++u) v[u] = host_nan<T>(v[u]);
        }
        std::uint16_t* d = dst + row * ld + col;
        if (wide && col + 7 < cols) {
            *reinterpret_cast<u32x4*>(d) = v;
        } else {
#pragma unroll
            for (int e = 0; e < 8; ++e)
                if (col + e < cols) d[e] = static_cast<std::uint16_t>(v[e >> 1] >> (16 * (e & 1)));
        }
    }
}

// An accumulator, moved out of its register here and no earlier: all at once there is no room for them.  (`kWay`: the two sides of a branch
// say something different, or the compiler moves what they have in common in front of it.)
template <int kWay> __device__ __forceinline__ float4v in_turn(float4v& acc) {
    if constexpr (kWay == 0) asm volatile("; plain" : "+a"(acc) : : "memory");
    else if constexpr (kWay == 1) asm volatile("; scaled" : "+a"(acc) : : "memory");
    else                     asm volatile("; part" : "+a"(acc) : : "memory");
    return acc;
}

template <typename T> __device__ __forceinline__ u32x2 pack4(const float4v v) {
    using El = Elem<T>;
    return u32x2{El::from_f32_finite(v[0]) | (static_cast<std::uint32_t>(El::from_f32_finite(v[1])) << 16),
                 El::from_f32_finite(v[2]) | (static_cast<std::uint32_t>(El::from_f32_finite(v[3])) << 16)};
}

}  // namespace flex
}  // namespace paras
