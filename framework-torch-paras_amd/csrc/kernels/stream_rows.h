// Products of a few rows with a matrix that is read once: the mainloop that streams the weights of a
// decode-time projection (gemm.hip) and of the experts of a decode step (moe_ffn.hip).
//
// What bounds such a product is the weights' way from memory.  v_mfma_f32_16x16x32 wants a row in every
// lane of 16, and a load in that order touches 16 rows of memory with each instruction, four lanes to
// a 64-byte piece but none of them neighbours, for the weights and again for the activations.  Here every load
// instruction reads eight rows x 128 contiguous bytes, eight neighbouring lanes to a row, and the
// operand order is made on the way through 1 KB of LDS per instruction (private to the wave: no barrier; the 16-byte
// chunks of a row are permuted by its index, so that neither side has bank conflicts).
//
// The eight waves of a workgroup share out the contraction in pieces of 64 (128 bytes of a row each, dealt round
// robin).  P pieces of a wave are under way in registers at any time, 130 to 200 KB per CU where it holds two workgroups; a piece
// past the wave's last is requested with an empty extent, which fetches nothing and keeps the number of requests
// in flight known to the compiler (P is what the loop fits into 128 registers: with one more, spilled registers are
// reloaded in it through the same counter and it waits for everything: 25.9 -> 30.8 us for 8 x 14336 x 4096).
//
// Against feeding the MFMAs straight from memory, bf16: 8 x 1024 x 4096 8.4 -> 5.9 us, 8 x 14336 x 4096 30.0 -> 21.8
// (5.4 TB/s), 8 x 4096 x 14336 25.1 -> 22.0 (5.3), 13 x 2048 x 2048 6.1 -> 5.2; a mixture-of-experts layer (8 experts, top-2,
// H 4096, I 14336) of 1 / 2 / 5 / 16 tokens 160 / 250 / 470 / 557 -> 138 / 192 / 415 / 484 us (5 tokens: 6.1 TB/s).
#pragma once

#include <hip/hip_runtime.h>

#include "core/device_math.h"

namespace paras {
namespace stream {

typedef short i16x8 __attribute__((ext_vector_type(8)));

template <typename T> struct Mma16;
template <> struct Mma16<bf16_t> {
    __device__ static __forceinline__ float4_t run(u32x4 a, u32x4 b, float4_t c) {
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
    }
};
template <> struct Mma16<f16_t> {
    __device__ static __forceinline__ float4_t run(u32x4 a, u32x4 b, float4_t c) {
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
    }
};

constexpr int kWaves = 8, kThreads = kWaves * 64;
constexpr int kPiece = 64;                               // contraction elements: 128 bytes of a row
constexpr long kMaxExtent = 0xE0000000L;
constexpr long kMaxLd = 1L << 22;                        // elements between weight rows

// G matrices with the same rows and stride (gate and up), NBG blocks of 16 of their rows, up to 8 XQ activation rows.
// kLone: the only such loop of its kernel, for which the compiler then finds registers for one more piece in two of the forms.
template <int G, int NBG, int XQ, bool kLone = false> struct Shape {
    static constexpr int kBlocks = G * NBG;              // weight blocks
    static constexpr int kXBlocks = (XQ + 1) / 2;        // activation blocks of 16 rows
    static constexpr int kRequests = 2 * kBlocks + XQ;   // 1 KB each per piece
    static constexpr int kWaveElems = kRequests * 512;   // LDS per wave
    static constexpr int kP = kRequests <= 3 ? 5 : (kRequests <= 4 ? (kLone ? 5 : 4) : (kRequests <= (kLone ? 6 : 5) ? 3 : 2));
    static constexpr int kPartElems = kWaves * kBlocks * kXBlocks * 512;     // the waves' results, laid over the same LDS
    static constexpr int kLdsElems = kWaves * kWaveElems > kPartElems ? kWaves * kWaveElems : kPartElems;
};

__device__ __forceinline__ int wave_id() { return __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) >> 6); }

// The work of a workgroup: `count` >= 1 column blocks, G x NBG x 16 weight rows each.  w[g]: the first weight row of
// the first of them, `step` rows from a block to the next, `ld` elements from a row to the next, `rows` >= 1 rows from the first one
// to the end of the matrix (all uniform; rows past the end count as zeros).  x: `x_bytes` <= kMaxExtent of activations,
// x_off[q] the byte offset of this lane's row 8 q + lane / 8.  `lds`: the workgroup's kLdsElems.
// The pieces of one block follow those of the one before without a gap: while its sums meet and are stored, the
// next one's weights are on their way.  store(j, acc) is called by all waves after the block's last piece, with
// acc[b][m]: lane (r16 = lane % 16, kg = lane / 16) holds this wave's part for activation row 16 m + r16 and weight rows
// 4 kg .. + 3 of block b (blocks of w[0] first).
template <typename T, int G, int NBG, int XQ, bool kLone, typename Store>
__device__ __forceinline__ void products(const std::uint16_t* const (&w)[G], long ld, long rows, long step, int count, long K,
                                         const std::uint16_t* x, long x_bytes, const std::uint32_t (&x_off)[XQ], std::uint16_t* lds, Store&& store) {
    using S = Shape<G, NBG, XQ, kLone>;
    constexpr int P = S::kP, NB = S::kBlocks, MB = S::kXBlocks;
    const int lane = threadIdx.x & 63, wave = wave_id();
    const int r16 = lane & 15, kg = lane >> 4;
    std::uint16_t* const stage = lds + wave * S::kWaveElems;
    const int put = (lane >> 3) * 64 + ((lane & 7) ^ (lane >> 3)) * 8;
    int get[2], xget[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const int chunk = ((h * 4 + kg) ^ (r16 & 7)) * 8;
        get[h] = r16 * 64 + chunk;
        xget[h] = (XQ == 1 ? (r16 & 7) : r16) * 64 + chunk;      // (rows 8 .. 15 of a single request: copies that nobody stores)
    }
    float4_t acc[NB][MB];
    auto clear = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int b = 0; b < NB; ++b)
#pragma unroll
            for (int m = 0; m < MB; ++m) acc[b][m] = float4_t{0.f, 0.f, 0.f, 0.f};
    };
    const std::uint32_t off = static_cast<std::uint32_t>((lane >> 3) * ld * 2 + (lane & 7) * 16);
    std::uint32_t xo[XQ];
#pragma unroll
    for (int q = 0; q < XQ; ++q) xo[q] = x_off[q] + (lane & 7) * 16;
    const std::uint32_t eight_rows = static_cast<std::uint32_t>(16 * ld);

    // This wave's pieces of a block: every kWaves-th one, as many trips of P as hold them.  Every workgroup starts at
    // another one of them and wraps around, so that the workgroups do not all read the same part of their rows at once.
    const int pieces = static_cast<int>(K / kPiece);
    const int mine = pieces > wave ? (pieces - wave + kWaves - 1) / kWaves : 0;
    const int trips = ((pieces + kWaves - 1) / kWaves + P - 1) / P;
    const int first = mine > 0 ? __builtin_amdgcn_readfirstlane(static_cast<int>(blockIdx.x * 3 % static_cast<unsigned>(mine))) : 0;
    int next = first, asked = 0, ahead = 0;         // the piece and the block of the next request
    const std::uint16_t* base[G];
    int records = 0;
    auto aim = [&]() __attribute__((always_inline)) {
        const long row = ahead * step, left = ahead < count ? rows - row : 0;
        const long extent = left > 0 ? ((left - 1) * ld + K) * 2 : 0;
        records = static_cast<int>(static_cast<std::uint32_t>(extent > kMaxExtent ? kMaxExtent : extent));
#pragma unroll
        for (int g = 0; g < G; ++g) base[g] = w[g] + row * ld;
    };
    auto fetch = [&](const std::uint16_t* p, int bytes, std::uint32_t at) __attribute__((always_inline)) {
        const auto r = __builtin_amdgcn_make_buffer_rsrc(const_cast<std::uint16_t*>(p), 0, bytes, 0x00020000);
        return __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(r, static_cast<int>(at), 0, 0));
    };
    u32x4 wv[P][2 * NB], xv[P][XQ];
    auto request = [&](int u) __attribute__((always_inline)) {
        // (a piece past the wave's last, a block past the workgroup's last: an empty extent)
        const int w_bytes = asked < mine ? records : 0;
        const int a_bytes = w_bytes != 0 ? static_cast<int>(static_cast<std::uint32_t>(x_bytes)) : 0;
        const std::uint32_t at = static_cast<std::uint32_t>(wave + next * kWaves) * (kPiece * 2);
#pragma unroll
        for (int g = 0; g < G; ++g)
#pragma unroll
            for (int i = 0; i < 2 * NBG; ++i) wv[u][g * 2 * NBG + i] = fetch(base[g], w_bytes, off + (at + i * eight_rows));
#pragma unroll
        for (int q = 0; q < XQ; ++q) xv[u][q] = fetch(x, a_bytes, xo[q] + at);
        ++asked;
        next = next + 1 >= mine ? 0 : next + 1;
        __builtin_amdgcn_sched_barrier(0);
    };
    auto multiply = [&](int u) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < 2 * NB; ++i) *reinterpret_cast<u32x4*>(&stage[i * 512 + put]) = wv[u][i];
#pragma unroll
        for (int q = 0; q < XQ; ++q) *reinterpret_cast<u32x4*>(&stage[(2 * NB + q) * 512 + put]) = xv[u][q];
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            u32x4 xf[MB];
#pragma unroll
            for (int m = 0; m < MB; ++m) xf[m] = *reinterpret_cast<const u32x4*>(&stage[2 * NB * 512 + m * 1024 + xget[h]]);
#pragma unroll
            for (int b = 0; b < NB; ++b) {
                const u32x4 wf = *reinterpret_cast<const u32x4*>(&stage[b * 1024 + get[h]]);
#pragma unroll
                for (int m = 0; m < MB; ++m) acc[b][m] = Mma16<T>::run(wf, xf[m], acc[b][m]);
            }
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    };
    aim();
#pragma unroll
    for (int u = 0; u < P; ++u) request(u);
    for (int j = 0; j < count; ++j) {
        clear();
        for (int t = 0; t < trips; ++t) {
            if (t == trips - 1) {           // from here on the requests are the next block's
                ++ahead;
                asked = 0;
                next = first;
                aim();
            }
#pragma unroll
            for (int u = 0; u < P; ++u) {
                if (t * P + u < mine) multiply(u);
                request(u);
            }
        }
        store(j, acc);
    }
}

// The waves' sums meet in LDS; block (b, m) is then sum_of(...) for the wave that takes it, in wave order.
template <int NB, int MB>
__device__ __forceinline__ void share(std::uint16_t* lds, const float4_t (&acc)[NB][MB]) {
    float4_t* part = reinterpret_cast<float4_t*>(lds);
    lds_barrier();                   // the stages are done with
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
        for (int m = 0; m < MB; ++m) part[(wave_id() * (NB * MB) + b * MB + m) * 64 + (threadIdx.x & 63)] = acc[b][m];
    lds_barrier();
}
template <int NB, int MB>
__device__ __forceinline__ float4_t sum_of(const std::uint16_t* lds, int b, int m) {
    const float4_t* part = reinterpret_cast<const float4_t*>(lds) + (b * MB + m) * 64 + (threadIdx.x & 63);
    float4_t t = part[0];
#pragma unroll
    for (int v = 1; v < kWaves; ++v) {
        const float4_t o = part[v * (NB * MB) * 64];
#pragma unroll
        for (int r = 0; r < 4; ++r) t[r] += o[r];
    }
    return t;
}

}  // namespace stream
}  // namespace paras
