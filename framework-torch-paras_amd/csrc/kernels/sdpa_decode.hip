// Split-KV decode attention for gfx950: few query rows per KV head (query
// length x GQA group <= 16), long K/V, bf16 / fp16, head dim 64 or 128.  The job is
// HBM-bound -- every K and V byte is read exactly once, K/V heads are never
// replicated for GQA (the reference copies them Hq/Hkv times:
// csrc/ops/tensor_ops.cpp:687-729) -- so the design is about keeping many
// independent 16-byte loads in flight, not about MFMA rate.
//
// grid = (splits, B*Hkv).  A workgroup owns one contiguous chunk of keys of one
// KV head; each of its 4 waves streams a quarter of the chunk in 32-key tiles:
//   S^T = K Q^T   v_mfma_f32_16x16x32: A = K rows loaded straight from HBM
//                 into registers (lane: key l%16, d = 32*step + 8*(l/16)..+7),
//                 B = the <=16 query rows (padded with zeros), in registers
//   online softmax per query (lane l%16), max shared by the 4 lane groups
//   O^T += V^T P^T  A = V^T via ds_read_b64_tr_b16 from a per-wave LDS tile
//                 (V is the one operand whose contraction index is not
//                 contiguous in memory), B = P^T from the S^T accumulators
// The 4 waves merge their (max, sum, O) in LDS; with more than one split the
// partial goes to the workspace and decode_combine_kernel merges the splits.
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdlib>
#include <type_traits>

#include "core/device_context.h"
#include "core/device_math.h"
#include "core/status.h"
#include "kernels/sdpa_internal.h"

namespace paras {
namespace {

constexpr int kThreads = 256;
constexpr int kWaves   = 4;
constexpr int kTile    = 32;        // keys per wave per step
// V row stride in LDS is D + 16 elements: 8 consecutive rows x 32 B then hit 64 distinct banks
// (288-byte rows at D = 128, 160-byte rows at D = 64).
constexpr int kMaxRows = 16;        // query rows per KV head (MFMA N)

typedef short i16x8 __attribute__((ext_vector_type(8)));
typedef __attribute__((address_space(3))) i16x4 lds_i16x4;

// (112 bytes without a mask: a launch whose arguments take more costs the host 0.7 us more, 3.4 for 2.7, and a call is two of them.)
struct DecodeParams {
    const std::uint16_t* q;
    const std::uint16_t* k;
    const std::uint16_t* v;
    std::uint16_t* out;
    float* lse;
    float* part;     // [pairs, splits]: 16 maxima, 16 sums, 16 x D outputs
    int q8_b, q8_h, q8_l, k8_b, k8_h, k8_l, v8_b, v8_h, v8_l;     // strides in eights of elements (decode_supported); between sequences 2^far eights
    int far;
    int Hkv, Lk;
    int chunk;       // keys per workgroup
    std::uint32_t shape;          // splits | Lq << 16 | G << 24
    float scale_log2, scale;
    __device__ int splits() const { return static_cast<int>(shape & 0xffff); }
    __device__ int Lq() const { return static_cast<int>(shape >> 16 & 0xff); }
    __device__ int G() const { return static_cast<int>(shape >> 24); }
};
static_assert(sizeof(DecodeParams) <= 112, "see above");
// optional mask (element strides; 0 = broadcast): bytes that are zero / non-zero, or additive values of the tensor dtype
struct DecodeMaskParams : DecodeParams {
    const unsigned char* mask;
    long ms_b, ms_h, ms_q, ms_k;
    float inv_scale;    // the scores are kept unscaled: an additive mask value m enters as m / scale
};

__host__ __device__ constexpr long slot_floats(long D) { return kMaxRows * (D + 2); }

template <typename T> struct Mma16;
template <> struct Mma16<bf16_t> {
    __device__ static __forceinline__ float4_t run(i16x8 a, i16x8 b, float4_t c) {
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
    }
    __device__ static __forceinline__ std::uint32_t pack2(float lo, float hi) {
        typedef float f32x2 __attribute__((ext_vector_type(2)));
        typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
        const f32x2 v = {lo, hi};
        return __builtin_bit_cast(std::uint32_t, __builtin_convertvector(v, bf16x2));
    }
};
template <> struct Mma16<f16_t> {
    __device__ static __forceinline__ float4_t run(i16x8 a, i16x8 b, float4_t c) {
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
    }
    __device__ static __forceinline__ std::uint32_t pack2(float lo, float hi) {
        typedef float f32x2 __attribute__((ext_vector_type(2)));
        typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
        const f32x2 v = {lo, hi};
        return __builtin_bit_cast(std::uint32_t, __builtin_convertvector(v, f16x2));
    }
};

// Combine over the 4 lane groups (lanes l, l^16, l^32, l^48) that share a query.
__device__ __forceinline__ float group_max(float x) {
    x = fmaxf(x, __shfl_xor(x, 16, kWave));
    return fmaxf(x, __shfl_xor(x, 32, kWave));
}
__device__ __forceinline__ float group_sum(float x) {
    x += __shfl_xor(x, 16, kWave);
    return x + __shfl_xor(x, 32, kWave);
}

// kMask: 0 = none, 1 = bool (true = attend), 2 = additive values of dtype T
template <typename T, int D, int kMask>
__global__ __launch_bounds__(kThreads, (D > 128 ? 1 : 2)) void decode_split_kernel(const typename std::conditional<kMask == 0, DecodeParams, DecodeMaskParams>::type p) {
    constexpr int kD = D, kVS = D + 16;
    constexpr int KS = D / 32;           // 32-wide contraction steps of q k^T
    constexpr int DB = D / 16;           // 16-wide output blocks of O^T
    constexpr int VCH = kTile * D / 8 / 64;   // 16-byte chunks of a V tile per lane
    // Per-wave V tiles (double buffered); reused as fp32 merge space at the end.
    __shared__ __attribute__((aligned(16))) std::uint16_t v_lds[kWaves][2][kTile * (D + 16)];
    __shared__ float m_lds[kWaves][kMaxRows], l_lds[kWaves][kMaxRows];

    // (One fetch for all of them: left to itself the compiler goes to memory twice in front of the first keys; 49 sequences of 187 keys 9.1 us, 8.8 so.)
    asm volatile("" ::"s"(p.q), "s"(p.k), "s"(p.v), "s"(p.q8_b), "s"(p.q8_h), "s"(p.q8_l), "s"(p.k8_b), "s"(p.k8_h), "s"(p.k8_l), "s"(p.v8_b), "s"(p.v8_h), "s"(p.v8_l),
                 "s"(p.far), "s"(p.Hkv), "s"(p.Lk), "s"(p.chunk), "s"(p.shape));
    const int split = blockIdx.x, pair = blockIdx.y, Lq = p.Lq(), G = p.G(), R = G * Lq;
    const int b = pair / p.Hkv, hkv = pair % p.Hkv;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int lq = lane & 15, lg = lane >> 4;

    // ---- the query rows of this KV head: row r = gi*Lq + i  (head hkv*G+gi, position i)
    i16x8 qreg[KS];
    {
        const bool live = lq < R;
        const int gi = live ? lq / Lq : 0, qi = live ? lq % Lq : 0;
        const std::uint16_t* qp = p.q + 8 * ((static_cast<long>(b) * p.q8_b << p.far) + static_cast<long>(hkv * G + gi) * p.q8_h + static_cast<long>(qi) * p.q8_l);
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
            i16x8 z = {0, 0, 0, 0, 0, 0, 0, 0};
            qreg[ks] = live ? *reinterpret_cast<const i16x8*>(qp + 32 * ks + 8 * lg) : z;
        }
    }

    // ---- this lane's mask row (query row lq): the 8 keys it scores per tile are 4 lg .. 4 lg + 3 of each 16-key block
    const unsigned char* mrow = nullptr;
    if constexpr (kMask != 0) {
        const bool live = lq < R;
        const int gi = live ? lq / Lq : 0, qi = live ? lq % Lq : 0;
        mrow = p.mask + (static_cast<long>(b) * p.ms_b + static_cast<long>(hkv * G + gi) * p.ms_h + static_cast<long>(qi) * p.ms_q) * (kMask == 1 ? 1 : 2);
    }

    // ---- this wave's key range
    const int chunk0 = split * p.chunk;
    const int chunk1 = min(chunk0 + p.chunk, p.Lk);
    const int wlen = (p.chunk / kWaves);  // chunk is a multiple of kWaves*kTile
    const int k_begin = chunk0 + wave * wlen;
    const int k_end = min(k_begin + wlen, chunk1);
    const int n_tiles = k_end > k_begin ? (k_end - k_begin + kTile - 1) / kTile : 0;

    const std::uint16_t* kbase = p.k + 8 * ((static_cast<long>(b) * p.k8_b << p.far) + static_cast<long>(hkv) * p.k8_h);
    const long k_row = 8L * p.k8_l, v_row = 8L * p.v8_l;
    const std::uint16_t* vbase = p.v + 8 * ((static_cast<long>(b) * p.v8_b << p.far) + static_cast<long>(hkv) * p.v8_h);

    i16x8 kcur[2][KS], knext[2][KS];
    u32x4 vst[VCH];
    auto load_k = [&](int t, i16x8 (&dst)[2][KS]) {
#pragma unroll
        for (int kb = 0; kb < 2; ++kb) {
            int key = k_begin + t * kTile + kb * 16 + lq;
            key = key < p.Lk ? key : p.Lk - 1;  // masked later; keep the load in bounds
            const std::uint16_t* kp = kbase + static_cast<long>(key) * k_row + 8 * lg;
#pragma unroll
            for (int ks = 0; ks < KS; ++ks) dst[kb][ks] = __builtin_bit_cast(i16x8, load16_nt(kp + 32 * ks));  // read once: keep it out of the caches
        }
    };
    auto load_v = [&](int t) {
#pragma unroll
        for (int i = 0; i < VCH; ++i) {
            const int c = lane + i * 64;  // 16-byte chunk of the 32 x D tile
            const int row = c / (D / 8), col = (c % (D / 8)) * 8;
            const int key = k_begin + t * kTile + row;
            vst[i] = key < k_end ? load16_nt(vbase + static_cast<long>(key) * v_row + col) : u32x4{0, 0, 0, 0};
        }
    };
    auto store_v = [&](int buf) {
#pragma unroll
        for (int i = 0; i < VCH; ++i) {
            const int c = lane + i * 64;
            const int row = c / (D / 8), col = (c % (D / 8)) * 8;
            *reinterpret_cast<u32x4*>(&v_lds[wave][buf][row * kVS + col]) = vst[i];
        }
    };

    // The mask of a tile, packed, is fetched with its keys: loads of its single bytes where they are needed wait for all the keys and
    // values requested before them (20 sequences of up to 29847 keys, 4 KV heads, D 128: 279 -> 251 us; 42 of 16260, one head: 88 -> 79).
    constexpr int MW = kMask == 2 ? 2 : 1;      // words of 4 mask values
    std::uint32_t mcur[2][MW], mnext[2][MW];
    auto load_mask = [&](int t, std::uint32_t (&dst)[2][MW]) {
        if constexpr (kMask != 0) {
            constexpr int kBytes = kMask == 1 ? 1 : 2;
            const int key0 = k_begin + t * kTile;
#pragma unroll
            for (int kb = 0; kb < 2; ++kb) {
                const int first = key0 + kb * 16 + 4 * lg;
                if (p.ms_k == 1 && key0 + kTile <= p.Lk) {
                    __builtin_memcpy(dst[kb], mrow + static_cast<long>(first) * kBytes, 4 * kBytes);      // (any alignment)
                } else {
#pragma unroll
                    for (int i = 0; i < MW; ++i) dst[kb][i] = 0;
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        const int key = first + r < p.Lk ? first + r : p.Lk - 1;                       // keys past the end are masked below anyway
                        const unsigned char* at = mrow + static_cast<long>(key) * p.ms_k * kBytes;
                        if constexpr (kMask == 1) dst[kb][0] |= static_cast<std::uint32_t>(*at) << (8 * r);
                        else                      dst[kb][r >> 1] |= static_cast<std::uint32_t>(*reinterpret_cast<const std::uint16_t*>(at)) << (16 * (r & 1));
                    }
                }
            }
        }
    };

    float4_t oacc[DB];
#pragma unroll
    for (int i = 0; i < DB; ++i) oacc[i] = float4_t{0.f, 0.f, 0.f, 0.f};
    float m_run = -INFINITY, l_run = 0.f;

    // Every wave starts at a tile of its own within its range and wraps around: the workgroups and
    // waves, which advance in step, would otherwise always be the same power of two apart in memory.
    const int rot = n_tiles > 1 ? (pair * 5 + split * 3 + wave * 7) % n_tiles : 0;
    auto tile_of = [&](int t) {
        const int tt = t + rot;
        return tt >= n_tiles ? tt - n_tiles : tt;
    };
    if (n_tiles > 0) {
        load_mask(tile_of(0), mcur);
        load_k(tile_of(0), kcur);
        load_v(tile_of(0));
        store_v(0);
    }
    // ds_read_tr lane offsets: group lg reads keys 4*lg + (m/4) (+16), 4 d's at 4*(m%4)
    const int v_off = (4 * lg + (lq >> 2)) * kVS + 4 * (lq & 3);

    for (int t = 0; t < n_tiles; ++t) {
        const int buf = t & 1;
        if (t + 1 < n_tiles) {
            load_mask(tile_of(t + 1), mnext);
            load_k(tile_of(t + 1), knext);
            load_v(tile_of(t + 1));
        }
        // S^T for two 16-key blocks
        float4_t sacc[2];
#pragma unroll
        for (int kb = 0; kb < 2; ++kb) {
            sacc[kb] = float4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int ks = 0; ks < KS; ++ks) sacc[kb] = Mma16<T>::run(kcur[kb][ks], qreg[ks], sacc[kb]);
        }
        const int key0 = k_begin + tile_of(t) * kTile;
        if constexpr (kMask != 0) {
#pragma unroll
            for (int kb = 0; kb < 2; ++kb)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    if constexpr (kMask == 1) {
                        if ((mcur[kb][0] >> (8 * r) & 0xff) == 0) sacc[kb][r] = -INFINITY;
                    } else {
                        const std::uint16_t bits = static_cast<std::uint16_t>(mcur[kb][r >> 1 & (MW - 1)] >> (16 * (r & 1)));
                        sacc[kb][r] = fmaf(Elem<T>::to_f32(bits), p.inv_scale, sacc[kb][r]);
                    }
                }
        }
        if (key0 + kTile > k_end) {
#pragma unroll
            for (int kb = 0; kb < 2; ++kb)
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    if (key0 + kb * 16 + 4 * lg + r >= k_end) sacc[kb][r] = -INFINITY;
        }
        float mloc = fmaxf(fmaxf(fmaxf(sacc[0][0], sacc[0][1]), fmaxf(sacc[0][2], sacc[0][3])),
                           fmaxf(fmaxf(sacc[1][0], sacc[1][1]), fmaxf(sacc[1][2], sacc[1][3])));
        mloc = group_max(mloc);
        const float m_new = fmaxf(m_run, mloc);
        // (with a mask every key so far may be masked out: -inf on both sides keeps the zeros, and the
        // reference point of the exponentials must not be -inf)
        const float alpha = m_run == m_new ? 1.f : __builtin_amdgcn_exp2f((m_run - m_new) * p.scale_log2);
        const float mc = m_new == -INFINITY ? 0.f : m_new * p.scale_log2;
        m_run = m_new;
        float lsum = 0.f;
#pragma unroll
        for (int kb = 0; kb < 2; ++kb)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const float e = __builtin_amdgcn_exp2f(fmaf(sacc[kb][r], p.scale_log2, -mc));
                sacc[kb][r] = e;
                lsum += e;
            }
        l_run = l_run * alpha + lsum;
#pragma unroll
        for (int i = 0; i < DB; ++i) oacc[i] *= alpha;
        // P^T operand: contraction order e<4 -> key 4*lg+e, e>=4 -> key 16+4*lg+(e-4)
        u32x4 w;
        w[0] = Mma16<T>::pack2(sacc[0][0], sacc[0][1]);
        w[1] = Mma16<T>::pack2(sacc[0][2], sacc[0][3]);
        w[2] = Mma16<T>::pack2(sacc[1][0], sacc[1][1]);
        w[3] = Mma16<T>::pack2(sacc[1][2], sacc[1][3]);
        const i16x8 pb = __builtin_bit_cast(i16x8, w);

        // Make this wave's LDS tile (written by its own lanes) visible to all of its lanes.
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
        for (int db = 0; db < DB; ++db) {
            const std::uint16_t* vp = &v_lds[wave][buf][v_off + db * 16];
            const i16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4*)(vp));
            const i16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4*)(vp + 16 * kVS));
            const i16x8 a = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
            oacc[db] = Mma16<T>::run(a, pb, oacc[db]);
        }
        if (t + 1 < n_tiles) {
            store_v(buf ^ 1);
#pragma unroll
            for (int kb = 0; kb < 2; ++kb)
#pragma unroll
                for (int ks = 0; ks < KS; ++ks) kcur[kb][ks] = knext[kb][ks];
            if constexpr (kMask != 0)
#pragma unroll
                for (int kb = 0; kb < 2; ++kb)
#pragma unroll
                    for (int i = 0; i < MW; ++i) mcur[kb][i] = mnext[kb][i];
        }
    }

    // ---- merge the 4 waves: O^T lane (query lq, group lg) holds d = 16*db + 4*lg + r
    const float l_wave = group_sum(l_run);
    __syncthreads();  // everyone is done with the V tiles
    float* o_lds = reinterpret_cast<float*>(&v_lds[0][0][0]);  // [wave][16][D] floats: 32 KB / 16 KB, inside the V tiles' space
    static_assert(sizeof(float) * kWaves * kMaxRows * D <= sizeof(std::uint16_t) * kWaves * 2 * kTile * kVS, "merge space");
    if (lq < R) {
#pragma unroll
        for (int db = 0; db < DB; ++db)
#pragma unroll
            for (int r = 0; r < 4; ++r) o_lds[(wave * kMaxRows + lq) * kD + 16 * db + 4 * lg + r] = oacc[db][r];
        if (lg == 0) {
            m_lds[wave][lq] = m_run;
            l_lds[wave][lq] = l_wave;
        }
    }
    __syncthreads();
    for (int idx = tid; idx < R * kD; idx += kThreads) {
        const int r = idx / kD, d = idx % kD;
        float M = -INFINITY;
#pragma unroll
        for (int w = 0; w < kWaves; ++w) M = fmaxf(M, m_lds[w][r]);
        float L = 0.f, O = 0.f;
#pragma unroll
        for (int w = 0; w < kWaves; ++w) {
            const float mw = m_lds[w][r];
            const float f = mw == -INFINITY ? 0.f : __builtin_amdgcn_exp2f((mw - M) * p.scale_log2);
            L += l_lds[w][r] * f;
            O += o_lds[(w * kMaxRows + r) * kD + d] * f;
        }
        if (p.splits() == 1) {
            const int gi = r / Lq, qi = r % Lq;
            const long orow = ((static_cast<long>(b) * p.Hkv + hkv) * G + gi) * Lq + qi;
            const float val = O / L;
            p.out[orow * kD + d] = static_cast<std::uint16_t>(Mma16<T>::pack2(val, 0.f) & 0xffffu);
            if (p.lse && d == 0) p.lse[orow] = M * p.scale + logf(L);
        } else {
            float* slot = p.part + (static_cast<long>(pair) * p.splits() + split) * slot_floats(kD);
            slot[2 * kMaxRows + r * kD + d] = O;
            if (d == 0) {
                slot[r] = M;
                slot[kMaxRows + r] = L;
            }
        }
    }
}

// One workgroup per (pair, query row): a lane owns 4 columns, and up to 512 / (D / 4) groups of lanes take the splits in turn, the first
// kAhead of each before the weights are known.  Bound by round trips to the L2: against D threads that go through all splits, a KV
// head of 20020 keys for each of 3 sequences (79 splits), the call: 27.0 -> 14.0 us; 2 heads of 25623 keys: 30.4 -> 14.3.
constexpr int kCombine = 512, kMaxSplits = 1024, kAhead = 4;
typedef float f32x4_any __attribute__((ext_vector_type(4), aligned(4)));

template <typename T, int D>
__global__ __launch_bounds__(kCombine) void decode_combine_kernel(const DecodeParams p) {
    constexpr int kLanes = D / 4;
    __shared__ float m_lds[kMaxSplits], l_lds[kMaxSplits];
    __shared__ float wave_m[kCombine / kWave], wave_l[kCombine / kWave];
    __shared__ float4_t o_lds[kCombine];
    const int pair = blockIdx.x, r = blockIdx.y, tid = threadIdx.x, threads = blockDim.x, waves = threads / kWave;
    const int group = tid / kLanes, groups = threads / kLanes, d0 = tid % kLanes * 4;
    const int splits = p.splits(), Lq = p.Lq(), G = p.G();
    const float* slot0 = p.part + static_cast<long>(pair) * splits * slot_floats(D);
    auto part = [&](int s) { return *reinterpret_cast<const f32x4_any*>(slot0 + s * slot_floats(D) + 2 * kMaxRows + r * D + d0); };
    float4_t ahead[kAhead];
#pragma unroll
    for (int i = 0; i < kAhead; ++i) {
        const int s = group + i * groups;
        ahead[i] = s < splits ? float4_t(part(s)) : float4_t{0.f, 0.f, 0.f, 0.f};
    }
    float M = -INFINITY;
    for (int s = tid; s < splits; s += threads) {
        const float* ml = slot0 + s * slot_floats(D) + r;
        m_lds[s] = ml[0];
        l_lds[s] = ml[kMaxRows];
        M = fmaxf(M, m_lds[s]);
    }
#pragma unroll
    for (int d = kWave / 2; d > 0; d >>= 1) M = fmaxf(M, __shfl_xor(M, d, kWave));
    if (tid % kWave == 0) wave_m[tid / kWave] = M;
    __syncthreads();
    for (int w = 0; w < waves; ++w) M = fmaxf(M, wave_m[w]);
    float L = 0.f;
    for (int s = tid; s < splits; s += threads) {
        const float f = m_lds[s] == -INFINITY ? 0.f : __builtin_amdgcn_exp2f((m_lds[s] - M) * p.scale_log2);
        m_lds[s] = f;
        L += l_lds[s] * f;
    }
#pragma unroll
    for (int d = kWave / 2; d > 0; d >>= 1) L += __shfl_xor(L, d, kWave);
    if (tid % kWave == 0) wave_l[tid / kWave] = L;
    __syncthreads();
    L = 0.f;
    for (int w = 0; w < waves; ++w) L += wave_l[w];
    float4_t O = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < kAhead; ++i) {
        const int s = group + i * groups;
        if (s < splits) O += ahead[i] * m_lds[s];
    }
#pragma unroll 4
    for (int s = group + kAhead * groups; s < splits; s += groups) O += float4_t(part(s)) * m_lds[s];
    o_lds[tid] = O;
    __syncthreads();
    if (group != 0) return;
    for (int g = 1; g < groups; ++g) O += o_lds[g * kLanes + tid];
    const int gi = r / Lq, qi = r % Lq;
    const long orow = (static_cast<long>(pair) * G + gi) * Lq + qi;
#pragma unroll
    for (int i = 0; i < 4; ++i) p.out[orow * D + d0 + i] = static_cast<std::uint16_t>(Mma16<T>::pack2(O[i] / L, 0.f) & 0xffffu);
    if (p.lse && tid == 0) p.lse[orow] = M * p.scale + logf(L);
}

// A group of lanes per split, whole waves, up to the largest workgroup
int combine_threads(int splits, long D) {
    int n = kWave;
    while (n < kCombine && n < splits * static_cast<int>(D / 4)) n *= 2;
    return n;
}

bool aligned16(const void* ptr) { return (reinterpret_cast<uintptr_t>(ptr) & 15) == 0; }
bool mult8(const int64_t* s) { return s[0] % 8 == 0 && s[1] % 8 == 0 && s[2] % 8 == 0; }

long compute_units() {
    int dev = 0;
    (void)hipGetDevice(&dev);
    auto* st = DeviceContext::instance().device(dev);
    return st ? st->compute_units : 256;
}

// Split count: whole rounds of workgroups over the CUs (a few workgroups more than that are a round of their own), one to eight of
// them, or no split at all; the one of least estimated time: that of all bytes from memory, of a CU's bytes, and of the tiles
// that follow each other in a wave, plus the merging of the splits where there are any.  Fitted to 70 problems (1 to 128 sequences, 64 to 32768
// keys, 1 to 8 KV heads, D 64 and 128): the choice is within 1 % of the best count in the mean, two workgroups per CU, rounded up,
// 5 % (42 KV heads of 16260 keys: 13 splits 79.1 us, 12 65.0; 144 heads of 298 keys: 2 splits 15.6, 1 11.1; 288 of 14555, D 64: 213 and 172).
void plan(const paras_sdpa_args& a, bool may_split, int* splits, int* chunk) {
    const long cus = compute_units(), pairs = a.B * a.Hkv, rows = pairs * (a.Hq / a.Hkv) * a.Lq;
    const long unit = kWaves * kTile;                        // 128 keys: one tile per wave
    long max_splits = (a.Lk + 2 * unit - 1) / (2 * unit);    // >= 2 tiles per wave
    if (max_splits > kMaxSplits) max_splits = kMaxSplits;
    const long per_cu = a.D <= 64 ? 3 : a.D <= 128 ? 2 : 1;
    const double key_bytes = 4.0 * a.D, memory = pairs * a.Lk * key_bytes / 9.1e6;
    auto fourth = [](double v) { return v * v * v * v; };
    double best = 1e300;
    long last = 0;
    for (long round = 0; round <= (may_split ? 8 : 0); ++round) {
        long want = round == 0 ? 1 : cus * round / pairs;
        want = want < 1 ? 1 : (want > max_splits ? max_splits : want);
        if (want == last) continue;
        last = want;
        const long steps = ((a.Lk + want - 1) / want + unit - 1) / unit, n = (a.Lk + steps * unit - 1) / (steps * unit), groups = pairs * n;
        const double cu = static_cast<double>((groups + cus - 1) / cus * steps * unit) * key_bytes / 27.5e3;
        const double chain = 1.9 * ((groups + cus * per_cu - 1) / (cus * per_cu) * steps);
        const double merge = n > 1 ? 3.6 + 1.06e-6 * rows * n * key_bytes + 0.2 * ((rows + 1023) / 1024) : 0.0;
        const double us = std::sqrt(std::sqrt(fourth(memory) + fourth(cu) + fourth(chain))) + merge;
        if (us < best) {
            best = us;
            *splits = static_cast<int>(n);
            *chunk = static_cast<int>(steps * unit);
        }
    }
}

size_t workspace_of(const paras_sdpa_args& a, int splits) {
    if (splits == 1) return 0;
    const size_t slots = static_cast<size_t>(a.B * a.Hkv) * splits;
    return slots * slot_floats(a.D) * sizeof(float);
}

// DecodeParams::far: 0 but for sequences 2^34 elements apart and more (a cache that holds all layers of a sequence together); -1: no power of two does.
int far_of(const paras_sdpa_args& a) {
    const int64_t q = a.q_strides[0] / 8, k = a.k_strides[0] / 8, v = a.v_strides[0] / 8;
    auto fits = [](int64_t n) { return n == static_cast<int>(n); };
    int far = 0;
    while (!(fits(q >> far) && fits(k >> far) && fits(v >> far))) ++far;
    return ((q | k | v) & ((int64_t{1} << far) - 1)) == 0 ? far : -1;
}

}  // namespace

bool decode_supported(const paras_sdpa_args& a) {
    if (a.dtype != PARAS_BF16 && a.dtype != PARAS_F16) return false;
    if (a.D != a.Dv || (a.D != 64 && a.D != 128 && a.D != 256)) return false;
    if (a.attn != nullptr || a.is_causal) return false;
    if (a.mask_kind != 0 && (a.mask == nullptr || a.mask_kind > 2)) return false;
    if (a.Hkv < 1 || a.Hq % a.Hkv != 0) return false;
    const int64_t rows = a.Lq * (a.Hq / a.Hkv);
    if (rows < 1 || rows > kMaxRows) return false;
    if (a.Lk < 1 || a.Lk > 0x3fffffff || a.B * a.Hkv > 65535) return false;
    if (!(a.scale > 0.0) || !std::isfinite(a.scale)) return false;
    if (!aligned16(a.q) || !aligned16(a.k) || !aligned16(a.v)) return false;
    if (!mult8(a.q_strides) || !mult8(a.k_strides) || !mult8(a.v_strides)) return false;
    for (const int64_t* st : {a.q_strides, a.k_strides, a.v_strides})
        for (int i = 1; i < 3; ++i)
            if (st[i] / 8 != static_cast<int>(st[i] / 8)) return false;          // (DecodeParams)
    return far_of(a) >= 0;
}

size_t decode_workspace(const paras_sdpa_args& a) {
    int splits = 1, chunk = 0;
    plan(a, true, &splits, &chunk);
    return workspace_of(a, splits);
}

bool decode_fills_chip(const paras_sdpa_args& a) { return a.B * a.Hkv >= 2 * compute_units(); }

int launch_decode(const paras_sdpa_args& a, Scratch scratch, hipStream_t s) {
    DecodeMaskParams p;
    p.q = static_cast<const std::uint16_t*>(a.q);
    p.k = static_cast<const std::uint16_t*>(a.k);
    p.v = static_cast<const std::uint16_t*>(a.v);
    p.out = static_cast<std::uint16_t*>(a.out);
    p.lse = a.lse;
    auto eights = [](int64_t stride) { return static_cast<int>(stride / 8); };
    p.far = far_of(a);
    auto between = [&](int64_t stride) { return static_cast<int>(stride / 8 >> p.far); };
    p.q8_b = between(a.q_strides[0]); p.q8_h = eights(a.q_strides[1]); p.q8_l = eights(a.q_strides[2]);
    p.k8_b = between(a.k_strides[0]); p.k8_h = eights(a.k_strides[1]); p.k8_l = eights(a.k_strides[2]);
    p.v8_b = between(a.v_strides[0]); p.v8_h = eights(a.v_strides[1]); p.v8_l = eights(a.v_strides[2]);
    p.Hkv = (int)a.Hkv; p.Lk = (int)a.Lk;
    const int G = (int)(a.Hq / a.Hkv), R = G * (int)a.Lq;
    int splits = 1;
    plan(a, scratch.p != nullptr && aligned16(scratch.p), &splits, &p.chunk);
    if (splits > 1 && !scratch.has(workspace_of(a, splits))) plan(a, false, &splits, &p.chunk);
    p.shape = static_cast<std::uint32_t>(splits) | static_cast<std::uint32_t>(a.Lq) << 16 | static_cast<std::uint32_t>(G) << 24;
    p.scale = static_cast<float>(a.scale);
    p.scale_log2 = static_cast<float>(a.scale * 1.4426950408889634);
    p.part = static_cast<float*>(scratch.p);
    const dim3 grid(splits, static_cast<unsigned>(a.B * a.Hkv));
    p.mask = static_cast<const unsigned char*>(a.mask);
    p.ms_b = a.mask_strides[0]; p.ms_h = a.mask_strides[1]; p.ms_q = a.mask_strides[2]; p.ms_k = a.mask_strides[3];
    p.inv_scale = static_cast<float>(1.0 / a.scale);
    const DecodeParams& plain = p;
    const bool bf = a.dtype == PARAS_BF16;
    const dim3 block(kThreads);
    const dim3 g2(static_cast<unsigned>(a.B * a.Hkv), R);
#define PARAS_DECODE_LAUNCH(T_, D_)                                                                        \
    do {                                                                                                   \
        if (a.mask_kind == 0)      hipLaunchKernelGGL((decode_split_kernel<T_, D_, 0>), grid, block, 0, s, plain); \
        else if (a.mask_kind == 1) hipLaunchKernelGGL((decode_split_kernel<T_, D_, 1>), grid, block, 0, s, p); \
        else                       hipLaunchKernelGGL((decode_split_kernel<T_, D_, 2>), grid, block, 0, s, p); \
        PARAS_HIP_TRY(hipGetLastError());                                                                  \
        if (splits > 1) {                                                                                  \
            hipLaunchKernelGGL((decode_combine_kernel<T_, D_>), g2, dim3(combine_threads(splits, D_)), 0, s, plain);                  \
            PARAS_HIP_TRY(hipGetLastError());                                                              \
        }                                                                                                  \
    } while (0)
    if (a.D == 256) {
        if (bf) PARAS_DECODE_LAUNCH(bf16_t, 256);
        else    PARAS_DECODE_LAUNCH(f16_t, 256);
    } else if (a.D == 128) {
        if (bf) PARAS_DECODE_LAUNCH(bf16_t, 128);
        else    PARAS_DECODE_LAUNCH(f16_t, 128);
    } else {
        if (bf) PARAS_DECODE_LAUNCH(bf16_t, 64);
        else    PARAS_DECODE_LAUNCH(f16_t, 64);
    }
#undef PARAS_DECODE_LAUNCH
    return PARAS_OK;
}

}  // namespace paras
