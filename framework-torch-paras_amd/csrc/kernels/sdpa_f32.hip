// Scaled-dot-product attention of fp32 tensors in one pass on the matrix cores: the output, the log-sum-exp and, in
// the form for large problems, the returned weights.
//
// Before, small problems ran one workgroup per query row with scalar fp64 dot products formed three
// times per score, every lane of a wavefront on a key row of its own (B1 H8 S128 D64: 44 us; B3 H64 S57
// D128: 254 us), and large ones as two batched products around a row kernel with the scores in memory (B1 H2
// S3737 D128: 740 us, of which 508 us one product with 60 workgroups).
//
// A workgroup takes 16 QB queries of one head; its four waves take the keys in turns of 16 or 32 (form_of) and meet at the end (row maximum, row sum, output: combined through LDS).  Per turn and wave:
//   S^T = K Q^T      v_mfma 16x16x4, A = 16 keys, B = 16 queries
//   online softmax   a lane holds one query and 4 keys of each 16 x 16 block
//   O^T += V^T P^T   the accumulator layout of S^T is the B operand layout of this product: step t takes
//                    register t of every lane, i.e. the keys that the instruction's row map puts there
// so nothing passes through LDS or between lanes except the row maxima.  Operands come straight from memory
// in 16-byte pieces, four MFMAs each: which contraction steps (QK) or head elements (PV) an instruction sees
// is free as long as both operands agree, and O^T then ends up with 4 adjacent elements of a row in a lane.
// K of the next turn and V of this one are requested before the turn's products.
//
// Acc = double: v_mfma_f64_16x16x4 (78 TFLOP/s published): what the general kernel computes, for the problems that it
// served.  Acc = float: v_mfma_f32_16x16x4 (157 TFLOP/s), for the large ones, which the batched products
// accumulated in fp32.  In both the softmax is fp64: exponentials and row sums unrounded, a weight rounded once, to
// the type of the product that takes it.  Scores are rounded to fp32 where the reference's
// are (the product, the scaled product, the sum with an additive mask: attention_ops.cpp:101-128).
// Against fp64, S 300 to 8192, heads of 64 to 256, scores of deviation 1 and 3: 3 to 49 % nearer than the batched products
// around an fp64 row kernel, which add up all keys in one chain where four waves add up a quarter each.
//
// NaN and infinities come out where the reference's do: a boolean mask and the causal rule select, an additive mask is
// added, and a value that nobody sees is still multiplied by its zero weights.
//
// What bounds it: small problems the chain of one turn (two memory latencies, products, merge; B1 H8 S128 D64 causal 6.9 us),
// large ones the matrix cores and the vector instructions, which do not run beside fp32 MFMAs here (weights of one query
// block interleaved with the products of the other, one MFMA to seven vector instructions: 874 -> 903 us).  B2 H16 S2048
// D128: unmasked 696-705 us = 98 TFLOP/s, causal 512-520 (every value is read, seen or not: 25 of them), 30 % padding 731, an additive
// mask 831; the batched products took 967 / 907 / 1520 / 1590.  B2 H8 S1024 D64 55 us (174), B1 H4 S2048 D256 203 (317).  (With blocks of 32 queries
// at 64 and 128 elements, turns of 32 keys and the softmax in fp64 742 / 623 / 775 / 830, 55 and 203.)  With those and the
// softmax in fp32 it took 697 / 567 / 665 / 950, 47 and 228, and single weights were 4.9e-7 off instead of 1.1e-7.
#include <hip/hip_runtime.h>

#include <cmath>

#include "core/device_math.h"
#include "core/status.h"
#include "kernels/sdpa_f32_forms.h"
#include "kernels/sdpa_internal.h"

namespace paras {
namespace {

constexpr int kWavesF = 4;
constexpr std::uint32_t kOutOfRange = 0xF0000000u;
// How far the running maximum may rise before the sums are rescaled: scores of deviation 1 to 3 rise by less after their first
// turn, and what it takes from fp32's exponent range is 8 of 87 powers of e.
constexpr double kSlack = 8.0;

struct F32Params {
    const float* q; const float* k; const float* v; float* out; float* lse;
    float* attn;          // [B, Hq, Lq, Lk] or null: takes the scaled and masked scores that were formed
    double2* row_sums;    // with attn, [B * Hq * Lq]: each row's reference point and its sum of exponentials
    const void* mask;
    int is_causal;
    int Hq, Hkv, Lq, Lk, D, Dv;
    int q_tiles;
    bool out16, attn16;   // rows of out / attn are whole 16-byte pieces
    long qs[3], ks[3], vs[3], ms[4];
    double scale;
    bool scale_is_float;
    double above;         // the exponentials' reference point lies this far above the (lagging) row maximum
};

template <typename Acc> struct Mma;
template <> struct Mma<double> {
    typedef double vec __attribute__((ext_vector_type(4)));
    __device__ static __forceinline__ vec run(float a, float b, vec c) {
        return __builtin_amdgcn_mfma_f64_16x16x4f64(static_cast<double>(a), static_cast<double>(b), c, 0, 0, 0);
    }
    __device__ static __forceinline__ vec run(float a, double b, vec c) {
        return __builtin_amdgcn_mfma_f64_16x16x4f64(static_cast<double>(a), b, c, 0, 0, 0);
    }
    __device__ static __forceinline__ int row(int g, int r) { return 4 * r + g; }       // row of register r in lane group g
};
template <> struct Mma<float> {
    typedef float vec __attribute__((ext_vector_type(4)));
    __device__ static __forceinline__ vec run(float a, float b, vec c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }
    __device__ static __forceinline__ int row(int g, int r) { return 4 * g + r; }
};

// DM: largest head size of this form (64, 128, 256); D and Dv are multiples of 4 up to it.
// A turn is KB blocks of 16 keys.  kMask: 0 = none, 1 = bool (true = attend), 2 = additive.
// (heads of up to 64 elements leave registers for two waves per SIMD)
template <typename Acc, int DM, int QB, int KB, int kMask>
__global__ __launch_bounds__(kWavesF * 64, DM == 64 || (DM == 128 && KB == 1 && sizeof(Acc) == 4) ? 2 : 1) void sdpa_f32_kernel(const F32Params p) {
    using M = Mma<Acc>;
    using vec = typename M::vec;
    constexpr int DC = DM / 16, VC = DM / 64, kTurn = 16 * KB;
    __shared__ Acc o_part[kWavesF][QB * VC * 4 * 256];
    __shared__ double m_part[kWavesF][QB][16], l_part[kWavesF][QB][16];

    // heaviest query tiles first under the causal rule
    const int qt = p.is_causal ? p.q_tiles - 1 - static_cast<int>(blockIdx.x) : static_cast<int>(blockIdx.x);
    const int h = blockIdx.y, b = blockIdx.z, hkv = h / (p.Hq / p.Hkv);
    const int lane = threadIdx.x & 63, l16 = lane & 15, g = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) >> 6);
    const int q0 = qt * 16 * QB;

    auto rsrc_of = [](const float* base, long rows, long ld, int width) {
        return __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(base), 0, static_cast<int>(((rows - 1) * ld + width) * 4), 0x00020000);
    };
    const auto kr = rsrc_of(p.k + b * p.ks[0] + hkv * p.ks[1], p.Lk, p.ks[2], p.D);      // (< 2^31 bytes: checked by f32_supported)
    const auto vr = rsrc_of(p.v + b * p.vs[0] + hkv * p.vs[1], p.Lk, p.vs[2], p.Dv);
    auto load4 = [](__amdgpu_buffer_rsrc_t r, std::uint32_t off) {
        return __builtin_bit_cast(float4_t, __builtin_amdgcn_raw_buffer_load_b128(r, static_cast<int>(off), 0, 0));
    };
    // (rows past the end come back as zeros; elements past the head size are kept out by an offset beyond the extent)
    float4_t qf[QB][DC], kf[KB][DC], vf[KB][4][VC];
    {
        const auto qr = rsrc_of(p.q + b * p.qs[0] + h * p.qs[1], p.Lq, p.qs[2], p.D);
#pragma unroll
        for (int qb = 0; qb < QB; ++qb)
#pragma unroll
            for (int c = 0; c < DC; ++c) {
                const int row = min(q0 + 16 * qb + l16, p.Lq - 1), d = 16 * c + 4 * g;
                qf[qb][c] = load4(qr, d < p.D ? static_cast<std::uint32_t>(row * p.qs[2] + d) * 4u : kOutOfRange);
            }
    }
    // (byte offsets in 32 bits: in range below 2^31 up to the last row, and a row past it is not asked for)
    const std::uint32_t kld = static_cast<std::uint32_t>(p.ks[2]) * 4u, vld = static_cast<std::uint32_t>(p.vs[2]) * 4u;
    auto load_k = [&](int j0) {
#pragma unroll
        for (int kb = 0; kb < KB; ++kb) {
            const int key = j0 + 16 * kb + l16;
            const std::uint32_t row = key < p.Lk ? static_cast<std::uint32_t>(key) * kld + 16u * g : kOutOfRange;
#pragma unroll
            for (int c = 0; c < DC; ++c) kf[kb][c] = load4(kr, (16 * c + 4 * g < p.D ? row : kOutOfRange) + 64u * c);
        }
    };
    auto load_v = [&](int j0) {
#pragma unroll
        for (int kb = 0; kb < KB; ++kb)
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                const int key = j0 + 16 * kb + M::row(g, t);
                const std::uint32_t row = key < p.Lk ? static_cast<std::uint32_t>(key) * vld + 16u * l16 : kOutOfRange;
#pragma unroll
                for (int c = 0; c < VC; ++c) vf[kb][t][c] = load4(vr, (64 * c + 4 * l16 < p.Dv ? row : kOutOfRange) + 256u * c);
            }
    };

    vec o[QB][VC][4];
    double m[QB], l[QB];                              // the maximum so far, up to kSlack behind; the sum of exponentials, unrounded
#pragma unroll
    for (int qb = 0; qb < QB; ++qb) {
        m[qb] = -INFINITY;
        l[qb] = 0;
#pragma unroll
        for (int c = 0; c < VC; ++c)
#pragma unroll
            for (int e = 0; e < 4; ++e) o[qb][c][e] = vec{0, 0, 0, 0};
    }
    const int keys = p.is_causal ? min(p.Lk, q0 + 16 * QB) : p.Lk;
    // more than 128 elements leave no registers for operands ahead of time: they are requested where they are used
    constexpr bool kAhead = DM <= 128;
    // (where a mask takes what registers these leave, places in the mask and the weights are worked out where they are used instead of being held)
    constexpr bool kTight = sizeof(Acc) == 4 && DM == 128 && QB == 2 && KB == 1 && kMask != 0;
    // The scores of a block for softmax_rows_kernel below: a lane holds 4 adjacent keys of one query.
    auto keep_scores = [&](int qb, int j, const float (&x)[4]) {
        float* at;
        if constexpr (kTight) {
            // (bytes in 32 bits past the tile's first row: there are 64 queries and 2^31 weights to a head, at least and at most)
            int query = 16 * qb + l16;
            asm volatile("" : "+v"(query));
            if (q0 + query >= p.Lq || j >= p.Lk) return;
            float* const tile = p.attn + ((static_cast<long>(b) * p.Hq + h) * p.Lq + q0) * p.Lk;
            at = reinterpret_cast<float*>(reinterpret_cast<char*>(tile) + (static_cast<std::uint32_t>(query) * static_cast<std::uint32_t>(p.Lk) + static_cast<std::uint32_t>(j)) * 4u);
        } else {
            const int i = q0 + 16 * qb + l16;
            if (i >= p.Lq || j >= p.Lk) return;
            at = p.attn + ((static_cast<long>(b) * p.Hq + h) * p.Lq + i) * p.Lk + j;
        }
        if (p.attn16) {
            *reinterpret_cast<float4_t*>(at) = float4_t{x[0], x[1], x[2], x[3]};
        } else {
#pragma unroll
            for (int r = 0; r < 4; ++r)
                if (j + r < p.Lk) at[r] = x[r];
        }
    };
    // A turn that no query of the tile sees: its weights are zeros whatever its scores are, but zero times a value that is
    // not finite is NaN, as in the reference's full product.  Each value times zero, then one product per block of the
    // output (A = those, B = zeros) that carries a NaN to its column of every query and changes nothing else.
    auto unseen_turn = [&](int j0) {
        load_v(j0);
#pragma unroll
        for (int c = 0; c < VC; ++c)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                float z = 0.0f;
#pragma unroll
                for (int kb = 0; kb < KB; ++kb)
#pragma unroll
                    for (int t = 0; t < 4; ++t) z = fmaf(vf[kb][t][c][e], 0.0f, z);
#pragma unroll
                for (int qb = 0; qb < QB; ++qb) o[qb][c][e] = M::run(z, static_cast<Acc>(0), o[qb][c][e]);
            }
    };
    // The mask of one query block's part of a turn at (kb, r).
    auto mask_at = [&](int j0, int qb, int kb, int r) {
        const long row = static_cast<long>(min(q0 + 16 * qb + l16, p.Lq - 1)), col = static_cast<long>(min(j0 + 16 * kb + M::row(g, r), p.Lk - 1));
        return b * p.ms[0] + h * p.ms[1] + row * p.ms[2] + col * p.ms[3];
    };
    // The same for all of a turn, element(qb, kb, r, place).
    auto each_mask_place = [&](int j0, auto&& element) {
        if constexpr (kTight) {
            int key = j0 + M::row(g, 0);
            asm volatile("" : "+v"(key));
            long col[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) col[r] = static_cast<long>(min(key + r, p.Lk - 1)) * p.ms[3];
#pragma unroll
            for (int qb = 0; qb < QB; ++qb) {
                int query = q0 + 16 * qb + l16;
                asm volatile("" : "+v"(query));
                const long row = b * p.ms[0] + h * p.ms[1] + static_cast<long>(min(query, p.Lq - 1)) * p.ms[2];
#pragma unroll
                for (int r = 0; r < 4; ++r) element(qb, 0, r, row + col[r]);
            }
        } else {
#pragma unroll
            for (int qb = 0; qb < QB; ++qb)
#pragma unroll
                for (int kb = 0; kb < KB; ++kb)
#pragma unroll
                    for (int r = 0; r < 4; ++r) element(qb, kb, r, mask_at(j0, qb, kb, r));
        }
    };
    // A boolean mask's part of a turn, bit 4 kb + r; false: the turn is closed to every query of the tile.
    auto open_bits = [&](int j0, unsigned (&open)[QB]) {
        unsigned any = 0;
#pragma unroll
        for (int qb = 0; qb < QB; ++qb) open[qb] = 0;
        each_mask_place(j0, [&](int qb, int kb, int r, long place) { open[qb] |= static_cast<const unsigned char*>(p.mask)[place] != 0 ? 1u << (4 * kb + r) : 0u; });
#pragma unroll
        for (int qb = 0; qb < QB; ++qb) any |= open[qb];
        return __builtin_amdgcn_ballot_w64(any != 0) != 0;
    };
    // The first turn from j0 on that this wave has scores to form for.  One that a boolean mask closes needs none (an
    // additive mask does not close anything: a NaN or +inf score plus -inf is NaN).
    bool closed = false;                              // some turn of this wave is
    auto next_open = [&](int j0, unsigned (&open)[QB]) {
        if constexpr (kMask == 1)
            for (; j0 < keys && !open_bits(j0, open); j0 += kWavesF * kTurn) {
                closed = true;
                if constexpr (sizeof(Acc) == 4)
                    if (p.attn != nullptr) {
                        const float hidden[4] = {-INFINITY, -INFINITY, -INFINITY, -INFINITY};
#pragma unroll
                        for (int qb = 0; qb < QB; ++qb)
#pragma unroll
                            for (int kb = 0; kb < KB; ++kb) keep_scores(qb, j0 + 16 * kb + M::row(g, 0), hidden);
                    }
            }
        return j0;
    };
    unsigned open[QB], open_next[QB];
    int j0 = next_open(wave * kTurn, open);
    if (kAhead && j0 < keys) load_k(j0);
    while (j0 < keys) {
        float mk[QB][KB][4];
        if constexpr (kMask == 2) each_mask_place(j0, [&](int qb, int kb, int r, long place) { mk[qb][kb][r] = static_cast<const float*>(p.mask)[place]; });
        if constexpr (kAhead) {
            load_v(j0);
        } else {
            load_k(j0);
            __builtin_amdgcn_sched_barrier(0);        // all of them on the way before the first is waited for
        }
        vec s[QB][KB];
#pragma unroll
        for (int qb = 0; qb < QB; ++qb)
#pragma unroll
            for (int kb = 0; kb < KB; ++kb) s[qb][kb] = vec{0, 0, 0, 0};
#pragma unroll
        for (int c = 0; c < DC; ++c)
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
                for (int kb = 0; kb < KB; ++kb)
#pragma unroll
                    for (int qb = 0; qb < QB; ++qb) s[qb][kb] = M::run(kf[kb][c][e], qf[qb][c][e], s[qb][kb]);
        const int j_next = next_open(j0 + kWavesF * kTurn, open_next);
        if (kAhead && j_next < keys) load_k(j_next);
        Acc pr[QB][KB][4];
#pragma unroll
        for (int qb = 0; qb < QB; ++qb) {
            const int i = q0 + 16 * qb + l16;
            float x[KB][4], mx = -INFINITY;
            // (the scale as it is given, the product rounded once; the torch ops narrow it themselves, as the reference does,
            // and the product of two floats needs no fp64)
            if (p.scale_is_float) {
                const float scale = static_cast<float>(p.scale);
#pragma unroll
                for (int kb = 0; kb < KB; ++kb)
#pragma unroll
                    for (int r = 0; r < 4; ++r) x[kb][r] = static_cast<float>(s[qb][kb][r]) * scale;
            } else {
#pragma unroll
                for (int kb = 0; kb < KB; ++kb)
#pragma unroll
                    for (int r = 0; r < 4; ++r) x[kb][r] = static_cast<float>(static_cast<double>(static_cast<float>(s[qb][kb][r])) * p.scale);
            }
            // (selected where a mask is boolean: a NaN or infinite score of a masked key is no score)
            if constexpr (kMask != 0)
#pragma unroll
                for (int kb = 0; kb < KB; ++kb)
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        if constexpr (kMask == 1) x[kb][r] = (open[qb] >> (4 * kb + r) & 1u) != 0 ? x[kb][r] : -INFINITY;
                        else                      x[kb][r] += mk[qb][kb][r];
                    }
            if (j0 + kTurn > p.Lk || (p.is_causal && j0 + kTurn - 1 > q0 + 16 * qb))          // the last keys, the diagonal
#pragma unroll
                for (int kb = 0; kb < KB; ++kb)
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        const int j = j0 + 16 * kb + M::row(g, r);
                        if (j >= p.Lk || (p.is_causal && j > i)) x[kb][r] = -INFINITY;
                    }
#pragma unroll
            for (int kb = 0; kb < KB; ++kb)
#pragma unroll
                for (int r = 0; r < 4; ++r) mx = fmaxf(mx, x[kb][r]);
            if constexpr (sizeof(Acc) == 4)
                if (p.attn != nullptr) {
#pragma unroll
                    for (int kb = 0; kb < KB; ++kb) keep_scores(qb, j0 + 16 * kb + M::row(g, 0), x[kb]);
                }
            mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
            mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
            // m follows the running maximum with some slack and in steps of whole powers of two, so that
            // the sums are rescaled seldom and exactly (a step beyond fp32's range takes them to nothing either way).
            const bool raise = static_cast<double>(mx) > m[qb] + kSlack;
            if (__builtin_amdgcn_ballot_w64(raise) != 0) {
                const double to = static_cast<double>(mx), steps = ceil((to - m[qb]) * 1.4426950408889634);
                const bool exact = steps < 128.0;
                const double f = !raise ? 1.0 : exact ? ldexp(1.0, -static_cast<int>(steps)) : 0.0;
                l[qb] *= f;
#pragma unroll
                for (int c = 0; c < VC; ++c)
#pragma unroll
                    for (int e = 0; e < 4; ++e) o[qb][c][e] *= static_cast<Acc>(f);
                m[qb] = !raise ? m[qb] : exact ? fma(steps, 0.6931471805599453, m[qb]) : to;
            }
            const double ref = m[qb] == -INFINITY ? 0.0 : m[qb] + p.above;               // no visible key yet: any reference but -inf
#pragma unroll
            for (int kb = 0; kb < KB; ++kb)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const double w = exp(static_cast<double>(x[kb][r]) - ref);
                    l[qb] += w;
                    pr[qb][kb][r] = static_cast<Acc>(w);
                }
        }
        if constexpr (!kAhead) {
            load_v(j0);
            __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int kb = 0; kb < KB; ++kb)
#pragma unroll
            for (int t = 0; t < 4; ++t)
#pragma unroll
                for (int c = 0; c < VC; ++c)
#pragma unroll
                    for (int e = 0; e < 4; ++e)
#pragma unroll
                        for (int qb = 0; qb < QB; ++qb) o[qb][c][e] = M::run(vf[kb][t][c][e], pr[qb][kb][t], o[qb][c][e]);
        j0 = j_next;
        if constexpr (kMask == 1)
#pragma unroll
            for (int qb = 0; qb < QB; ++qb) open[qb] = open_next[qb];
    }

    // what the causal rule, or a boolean mask, hides from the whole tile
    if constexpr (kMask == 0)
        for (; j0 < p.Lk; j0 += kWavesF * kTurn) unseen_turn(j0);
    if constexpr (kMask == 1)
        if (closed)
            for (j0 = wave * kTurn; j0 < keys; j0 += kWavesF * kTurn) {
                if (!open_bits(j0, open)) unseen_turn(j0);
            }

    // the waves meet
#pragma unroll
    for (int qb = 0; qb < QB; ++qb) {
        l[qb] += __shfl_xor(l[qb], 16, 64);
        l[qb] += __shfl_xor(l[qb], 32, 64);
        if (g == 0) {
            m_part[wave][qb][l16] = m[qb];
            l_part[wave][qb][l16] = l[qb];
        }
#pragma unroll
        for (int c = 0; c < VC; ++c)
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
                for (int r = 0; r < 4; ++r) o_part[wave][((qb * VC + c) * 4 + e) * 256 + r * 64 + lane] = o[qb][c][e][r];
    }
    __syncthreads();
    for (int item = wave; item < QB * VC * 4; item += kWavesF) {
        const int r = item & 3, c = (item >> 2) % VC, qb = (item >> 2) / VC;
        const int i = q0 + 16 * qb + l16, dv = 64 * c + 4 * M::row(g, r);
        double mm = m_part[0][qb][l16];
#pragma unroll
        for (int w = 1; w < kWavesF; ++w) mm = m_part[w][qb][l16] > mm ? m_part[w][qb][l16] : mm;
        const double ref = mm == -INFINITY ? 0.0 : mm;
        double sum = 0, val[4] = {0, 0, 0, 0};
#pragma unroll
        for (int w = 0; w < kWavesF; ++w) {
            const double f = exp(m_part[w][qb][l16] - ref);
            sum += f * l_part[w][qb][l16];
#pragma unroll
            for (int e = 0; e < 4; ++e) val[e] += f * static_cast<double>(o_part[w][((qb * VC + c) * 4 + e) * 256 + r * 64 + lane]);
        }
        if (i >= p.Lq) continue;
        const long row = (static_cast<long>(b) * p.Hq + h) * p.Lq + i;
        if (dv < p.Dv) {
            float4_t y;
#pragma unroll
            for (int e = 0; e < 4; ++e) y[e] = static_cast<float>(val[e] / sum);
            float* const at = p.out + row * p.Dv + dv;
            if (p.out16) {
                *reinterpret_cast<float4_t*>(at) = y;
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e) at[e] = y[e];
            }
        }
        if (c == 0 && r == 0 && g == 0) {
            if (p.lse != nullptr) p.lse[row] = static_cast<float>(mm + p.above + log(sum));
            if (p.row_sums != nullptr) p.row_sums[row] = double2{mm == -INFINITY ? 0.0 : mm + p.above, sum};
        }
    }
}

// The returned weights, in place of the scores that sdpa_f32_kernel left: exp(score - reference) / sum in fp64, rounded
// once; zeros for the keys that the causal rule hides (NaN where the row is).  A wave takes a row in pieces of W elements.
// Bound by memory (one read and one write of the weights tensor); four pieces are on the way at a time.  B2 H16 S2048 D128 with
// its 537 MB of weights 925 us, causal 714; the product, row kernel and product in their place 967 and 907; B2 H8 S1024 D64 88 (174).
template <int W>
__global__ __launch_bounds__(256) void softmax_rows_kernel(float* __restrict__ attn, const double2* __restrict__ row_sums, long rows, int Lq, int Lk, int is_causal) {
    typedef float piece __attribute__((ext_vector_type(W)));
    constexpr int kAtOnce = 4;
    const long row = static_cast<long>(blockIdx.x) * 4 + (threadIdx.x >> 6);
    if (row >= rows) return;
    const int lane = threadIdx.x & 63;
    const int seen = is_causal ? min(static_cast<int>(row % Lq) + 1, Lk) : Lk;
    const double2 of = row_sums[row];
    const double inv = 1.0 / of.y, none = 0.0 * inv;
    float* const base = attn + row * Lk;
    for (int j0 = 0; j0 < Lk; j0 += 64 * W * kAtOnce) {
        piece x[kAtOnce];
#pragma unroll
        for (int t = 0; t < kAtOnce; ++t) {
            const int j = j0 + (64 * t + lane) * W;
            if (j < seen) x[t] = *reinterpret_cast<const piece*>(base + j);
        }
#pragma unroll
        for (int t = 0; t < kAtOnce; ++t) {
            const int j = j0 + (64 * t + lane) * W;
            if (j >= Lk) continue;
            piece y;
#pragma unroll
            for (int e = 0; e < W; ++e) y[e] = static_cast<float>(none);
            if (j < seen)
#pragma unroll
                for (int e = 0; e < W; ++e)
                    if (j + e < seen) y[e] = static_cast<float>(exp(static_cast<double>(x[t][e]) - of.x) * inv);
            *reinterpret_cast<piece*>(base + j) = y;
        }
    }
}

template <typename Acc, int DM, int QB, int KB, int kMask>
void launch_masked(F32Params p, const paras_sdpa_args& a, hipStream_t s) {
    p.q_tiles = static_cast<int>((a.Lq + 16 * QB - 1) / (16 * QB));
    const dim3 g(p.q_tiles, static_cast<unsigned>(a.Hq), static_cast<unsigned>(a.B)), t(kWavesF * 64);
    hipLaunchKernelGGL((sdpa_f32_kernel<Acc, DM, QB, KB, kMask>), g, t, 0, s, p);
}
template <typename Acc, int DM, int QB, int KB>
void launch_form(const F32Params& p, const paras_sdpa_args& a, hipStream_t s) {
    if (a.mask_kind == 0)      launch_masked<Acc, DM, QB, KB, 0>(p, a, s);
    else if (a.mask_kind == 1) launch_masked<Acc, DM, QB, KB, 1>(p, a, s);
    else                       launch_masked<Acc, DM, QB, KB, 2>(p, a, s);
}

template <typename Acc, int DM>
void launch_dm(const F32Params& p, const paras_sdpa_args& a, hipStream_t s) {
    if constexpr (sizeof(Acc) == 8) {
        // up to 64 keys turns of 16 give all four waves some; at 256 elements that is also all the registers hold
        if constexpr (DM <= 128) {
            if (a.Lk > 64) return launch_form<Acc, DM, 1, 2>(p, a, s);
        }
        launch_form<Acc, DM, 1, 1>(p, a, s);
    } else {
        const Form form = form_of<DM>(a);
        if (form == Form::k16x16) return launch_form<Acc, DM, 1, 1>(p, a, s);
        if constexpr (DM == 64) {               // (no boolean mask takes 32 x 32 there)
            if (form == Form::k32x32) return a.mask_kind == 0 ? launch_masked<Acc, DM, 2, 2, 0>(p, a, s) : launch_masked<Acc, DM, 2, 2, 2>(p, a, s);
        } else if constexpr (DM == 128) {       // (only the causal rule takes 32 x 32 there)
            if (form == Form::k32x32) return launch_masked<Acc, DM, 2, 2, 0>(p, a, s);
            if (form == Form::k32x16) return launch_form<Acc, DM, 2, 1>(p, a, s);
        }
        launch_form<Acc, DM, 1, 2>(p, a, s);
    }
}

}  // namespace

// (by sizes and strides alone: paras_sdpa_workspace may be asked before the pointers are known)
bool f32_supported(const paras_sdpa_args& a) {
    if (a.dtype != PARAS_F32) return false;
    if (a.D < 4 || a.Dv < 4 || a.D > 256 || a.Dv > 256 || a.D % 4 != 0 || a.Dv % 4 != 0 || a.Lq < 1 || a.Lk < 1) return false;
    if (a.Hq > 65535 || a.B > 65535 || a.Lq >= (1L << 30) || a.Lk >= (1L << 30)) return false;
    if (a.q_strides[2] < 0 || a.k_strides[2] < 0 || a.v_strides[2] < 0) return false;
    const long lim = (1L << 29) - 1;                       // elements: byte offsets below 2^31
    return (a.Lq - 1) * a.q_strides[2] + a.D <= lim && (a.Lk - 1) * a.k_strides[2] + a.D <= lim && (a.Lk - 1) * a.v_strides[2] + a.Dv <= lim;
}

size_t f32_workspace(const paras_sdpa_args& a) { return a.attn != nullptr ? static_cast<size_t>(a.B * a.Hq * a.Lq) * sizeof(double2) : 0; }

int launch_f32(const paras_sdpa_args& a, bool accumulate_f64, void* workspace, hipStream_t s) {
    F32Params p{};
    p.q = static_cast<const float*>(a.q); p.k = static_cast<const float*>(a.k); p.v = static_cast<const float*>(a.v);
    p.out = static_cast<float*>(a.out); p.lse = a.lse; p.mask = a.mask;
    p.out16 = (reinterpret_cast<uintptr_t>(a.out) & 15) == 0;
    p.is_causal = a.is_causal;
    p.Hq = static_cast<int>(a.Hq); p.Hkv = static_cast<int>(a.Hkv);
    p.Lq = static_cast<int>(a.Lq); p.Lk = static_cast<int>(a.Lk); p.D = static_cast<int>(a.D); p.Dv = static_cast<int>(a.Dv);
    for (int i = 0; i < 3; ++i) { p.qs[i] = a.q_strides[i]; p.ks[i] = a.k_strides[i]; p.vs[i] = a.v_strides[i]; }
    for (int i = 0; i < 4; ++i) p.ms[i] = a.mask_strides[i];
    if (a.attn != nullptr) {
        PARAS_REQUIRE(!accumulate_f64, "paras sdpa: the fp64 form returns no weights");
        PARAS_REQUIRE(workspace != nullptr, "paras sdpa: workspace is null");
        PARAS_REQUIRE((reinterpret_cast<uintptr_t>(workspace) & 255) == 0, "paras sdpa: the workspace must be 256-byte aligned");
        p.attn = static_cast<float*>(a.attn);
        p.row_sums = static_cast<double2*>(workspace);
        p.attn16 = a.Lk % 4 == 0 && (reinterpret_cast<uintptr_t>(a.attn) & 15) == 0;
    }
    p.scale = a.scale;
    p.scale_is_float = static_cast<double>(static_cast<float>(a.scale)) == a.scale;
    // Lk weights of at most 1 / Lk: a weighted sum of values that fp32 holds is one that it holds
    p.above = kSlack + std::log(static_cast<double>(a.Lk));
    const long dm = a.D > a.Dv ? a.D : a.Dv;
    if (accumulate_f64) {
        if (dm <= 64)       launch_dm<double, 64>(p, a, s);
        else if (dm <= 128) launch_dm<double, 128>(p, a, s);
        else                launch_dm<double, 256>(p, a, s);
    } else {
        if (dm <= 64)       launch_dm<float, 64>(p, a, s);
        else if (dm <= 128) launch_dm<float, 128>(p, a, s);
        else                launch_dm<float, 256>(p, a, s);
    }
    PARAS_HIP_TRY(hipGetLastError());
    if (a.attn != nullptr) {
        const long rows = a.B * a.Hq * a.Lq;
        const dim3 grid(static_cast<unsigned>((rows + 3) / 4));
        if (p.attn16) hipLaunchKernelGGL((softmax_rows_kernel<4>), grid, dim3(256), 0, s, p.attn, p.row_sums, rows, p.Lq, p.Lk, a.is_causal);
        else          hipLaunchKernelGGL((softmax_rows_kernel<1>), grid, dim3(256), 0, s, p.attn, p.row_sums, rows, p.Lq, p.Lk, a.is_causal);
        PARAS_HIP_TRY(hipGetLastError());
    }
    return PARAS_OK;
}

}  // namespace paras
