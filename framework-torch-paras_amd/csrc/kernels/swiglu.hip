// Fused SwiGLU forward/backward and rotate_half for gfx950.
//
// out = silu(gate) * up with the host engine's rounding (see
// kernels/swiglu_math.h for how the fp64 definition is met at fp32 cost).
//
// Layout: flat contiguous streams, 16 bytes per lane per access, kUnroll
// independent non-temporal accesses per stream in flight per lane, one chunk
// per workgroup (tens of thousands of short workgroups stream better here
// than a persistent grid-stride loop).
#include <hip/hip_runtime.h>

#include <type_traits>

#include "core/device_context.h"
#include "core/device_math.h"
#include "core/status.h"
#include "kernels/few_dims.h"
#include "kernels/swiglu_math.h"

namespace paras {
namespace {

constexpr int kBlock  = 256;

// One 16-byte vector of results.  fp16: every element through the fp32 tier, without a branch; the few whose value is next to a
// rounding boundary (or outside the tier's range) are redone in fp64 in a loop that runs as often as the lane with the most of
// them needs.  A wave of eight elements a lane then comes to the fp64 formula 0.7 times instead of 3.2.  bf16, where that is 0.3 for 0.5,
// branches element by element: a forward and backward of 8192 x 14336 take 301 us with the loop, 294 to 298 without.
template <typename T>
__device__ __forceinline__ u32x4 swiglu_vec(u32x4 gv, u32x4 uv) {
    using E = Elem<T>;
    using S = typename E::store_t;
    const S* ge = reinterpret_cast<const S*>(&gv);
    const S* ue = reinterpret_cast<const S*>(&uv);
    u32x4 o;
    S* oe = reinterpret_cast<S*>(&o);
    if constexpr (std::is_same_v<T, f16_t>) {
        unsigned redo = 0;
        S r[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            bool ok;
            r[j] = swiglu_fast<T>(ge[j], ue[j], ok);
            redo |= ok ? 0u : (1u << j);
        }
        while (redo != 0) {
            const int j = __builtin_ctz(redo);
            redo &= redo - 1;
            S g16 = 0, u16 = 0;
#pragma unroll
            for (int k = 0; k < 8; ++k)
                if (k == j) { g16 = ge[k]; u16 = ue[k]; }
            const S x = swiglu_exact<T>(E::to_f32(g16), E::to_f32(u16));
#pragma unroll
            for (int k = 0; k < 8; ++k)
                if (k == j) r[k] = x;
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) o[j] = r[2 * j] | (static_cast<std::uint32_t>(r[2 * j + 1]) << 16);
    } else {
#pragma unroll
        for (int j = 0; j < E::kVec; ++j) {
            if constexpr (sizeof(S) == 2) {
                bool ok;
                oe[j] = swiglu_fast<T>(ge[j], ue[j], ok);
                if (__builtin_expect(!ok, 0)) {
                    // (Left to itself the compiler forms the fp64 formula of half the elements ahead of their branches: 474 x 14336, the
                    // inputs in the caches, 15.1 us, 8.0 so.)
                    float g = E::to_f32(ge[j]);
                    asm volatile("" : "+v"(g));
                    oe[j] = swiglu_exact<T>(g, E::to_f32(ue[j]));
                }
            } else {
                oe[j] = swiglu_one<T>(ge[j], ue[j]);
            }
        }
    }
    return o;
}

// kUnroll: 16-byte vectors per stream per lane per iteration.  `tail`: elements past the last whole vector, the last workgroup's (a launch
// of their own cost 4.5 us behind 43 M elements, and as much of the host's time as the first).
template <typename T, int kUnroll>
__global__ __launch_bounds__(kBlock) void swiglu_fwd_vec(
    const typename Elem<T>::store_t* __restrict__ gate, const typename Elem<T>::store_t* __restrict__ up,
    typename Elem<T>::store_t* __restrict__ out, long nvec, int tail) {
    constexpr int V = Elem<T>::kVec;
    const long stride = static_cast<long>(gridDim.x) * kBlock * kUnroll;
    for (long base = static_cast<long>(blockIdx.x) * kBlock * kUnroll + threadIdx.x; base < nvec;
         base += stride) {
        u32x4 gv[kUnroll], uv[kUnroll];
#pragma unroll
        for (int k = 0; k < kUnroll; ++k) {
            const long i = base + static_cast<long>(k) * kBlock;
            if (i < nvec) {
                gv[k] = load16_nt(gate + i * V);
                uv[k] = load16_nt(up + i * V);
            }
        }
#pragma unroll
        for (int k = 0; k < kUnroll; ++k) {
            const long i = base + static_cast<long>(k) * kBlock;
            if (i < nvec) store16_nt(out + i * V, swiglu_vec<T>(gv[k], uv[k]));
        }
    }
    if (blockIdx.x + 1 == gridDim.x && static_cast<int>(threadIdx.x) < tail) {
        const long i = nvec * V + threadIdx.x;
        out[i] = swiglu_one<T>(gate[i], up[i]);
    }
}

template <typename T>
__global__ __launch_bounds__(kBlock) void swiglu_fwd_any(
    const typename Elem<T>::store_t* __restrict__ gate, const typename Elem<T>::store_t* __restrict__ up,
    typename Elem<T>::store_t* __restrict__ out, long n) {
    const long stride = static_cast<long>(gridDim.x) * kBlock;
    for (long i = static_cast<long>(blockIdx.x) * kBlock + threadIdx.x; i < n; i += stride)
        out[i] = swiglu_one<T>(gate[i], up[i]);
}

// Backward (csrc/ops/fused_ops.cpp:218-226), fp64 as on the host:
//   s = 1/(1+exp(-g)); dup = dy*g*s; dgate = dy*u*(s*(1+g*(1-s)))
template <typename T>
__global__ __launch_bounds__(kBlock) void swiglu_bwd_any(
    const typename Elem<T>::store_t* __restrict__ go, const typename Elem<T>::store_t* __restrict__ gate,
    const typename Elem<T>::store_t* __restrict__ up, typename Elem<T>::store_t* __restrict__ ggate,
    typename Elem<T>::store_t* __restrict__ gup, long n) {
    using E = Elem<T>;
    const long stride = static_cast<long>(gridDim.x) * kBlock;
    for (long i = static_cast<long>(blockIdx.x) * kBlock + threadIdx.x; i < n; i += stride) {
        const double dy = E::to_f64(go[i]);
        const double g  = E::to_f64(gate[i]);
        const double u  = E::to_f64(up[i]);
        const double s  = 1.0 / (1.0 + exp(-g));
        gup[i]   = E::from_f64(dy * g * s);
        ggate[i] = E::from_f64(dy * u * (s * (1.0 + g * (1.0 - s))));
    }
}

// 16-bit tensors, 16-byte aligned: eight elements per lane and access.  Every element goes through
// the fp32 fast tier; the few whose result sits next to a rounding boundary (or outside the fast
// tier's range) are collected in a bit mask and redone in fp64 in a loop that runs as often as the
// lane with the most of them needs -- usually not at all, sometimes once.
template <typename T>
__global__ __launch_bounds__(kBlock) void swiglu_bwd_vec(const std::uint16_t* __restrict__ go,
                                                         const std::uint16_t* __restrict__ gate,
                                                         const std::uint16_t* __restrict__ up,
                                                         std::uint16_t* __restrict__ ggate,
                                                         std::uint16_t* __restrict__ gup, long nvec, int tail) {
    using E = Elem<T>;
    for (long i = static_cast<long>(blockIdx.x) * kBlock + threadIdx.x; i < nvec; i += static_cast<long>(gridDim.x) * kBlock) {
        const u32x4 dv = load16_nt(go + i * 8), gv = load16_nt(gate + i * 8), uv = load16_nt(up + i * 8);
        const std::uint16_t* de = reinterpret_cast<const std::uint16_t*>(&dv);
        const std::uint16_t* ge = reinterpret_cast<const std::uint16_t*>(&gv);
        const std::uint16_t* ue = reinterpret_cast<const std::uint16_t*>(&uv);
        std::uint16_t og[8], ou[8];
        unsigned redo = 0;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            float yg, yu;
            bool ok_g, ok_u;
            swiglu_bwd_fast<T>(E::to_f32(de[j]), E::to_f32(ge[j]), E::to_f32(ue[j]), yg, yu, ok_g, ok_u);
            og[j] = E::from_f32_finite(yg);
            ou[j] = E::from_f32_finite(yu);
            redo |= (ok_g && ok_u) ? 0u : (1u << j);
        }
        while (redo != 0) {
            const int j = __builtin_ctz(redo);
            redo &= redo - 1;
            std::uint16_t d16 = 0, g16 = 0, u16 = 0;
#pragma unroll
            for (int k = 0; k < 8; ++k)
                if (k == j) { d16 = de[k]; g16 = ge[k]; u16 = ue[k]; }
            std::uint16_t xg, xu;
            swiglu_bwd_exact<T>(E::to_f32(d16), E::to_f32(g16), E::to_f32(u16), xg, xu);
#pragma unroll
            for (int k = 0; k < 8; ++k)
                if (k == j) { og[k] = xg; ou[k] = xu; }
        }
        u32x4 wg, wu;
#pragma unroll
        for (int p2 = 0; p2 < 4; ++p2) {
            wg[p2] = og[2 * p2] | (static_cast<std::uint32_t>(og[2 * p2 + 1]) << 16);
            wu[p2] = ou[2 * p2] | (static_cast<std::uint32_t>(ou[2 * p2 + 1]) << 16);
        }
        store16_nt(ggate + i * 8, wg);
        store16_nt(gup + i * 8, wu);
    }
    if (blockIdx.x + 1 == gridDim.x && static_cast<int>(threadIdx.x) < tail) {        // (past the last whole vector)
        const long i = nvec * 8 + threadIdx.x;
        swiglu_bwd_exact<T>(E::to_f32(go[i]), E::to_f32(gate[i]), E::to_f32(up[i]), ggate[i], gup[i]);
    }
}

// rotate_half (csrc/ops/fused_ops.cpp:254-263, 290-299): out[.., c] takes
// x[.., c+half] (negated for forward) when c < half, else x[.., c-half]
// (negated for backward).  Negation flips the sign bit, which is what
// -(double)v rounded back gives for every finite value and infinity; a NaN
// stays a NaN.
// A 16-bit NaN as the host writes it after its trip through double: bf16 0x7FC0, half sign | 0x7E00
// (kind 1 / 2; anything else passes through).
__device__ __forceinline__ std::uint32_t host_nan16(std::uint32_t h, int kind) {
    if (kind == 1) return (h & 0x7FFFu) > 0x7F80u ? 0x7FC0u : h;
    if (kind == 2) return (h & 0x7FFFu) > 0x7C00u ? ((h & 0x8000u) | 0x7E00u) : h;
    return h;
}
template <typename S>
__global__ __launch_bounds__(kBlock) void rotate_half_any(const S* __restrict__ x, S* __restrict__ out,
                                                          long n, long D, int backward, int nan_kind) {
    const long half = D / 2;
    const long stride = static_cast<long>(gridDim.x) * kBlock;
    constexpr S kSign = static_cast<S>(S{1} << (sizeof(S) * 8 - 1));
    for (long i = static_cast<long>(blockIdx.x) * kBlock + threadIdx.x; i < n; i += stride) {
        const long col = i % D;
        const bool first = col < half;
        const S v = x[first ? i + half : i - half];
        const bool negate = backward ? !first : first;
        S r = negate ? static_cast<S>(v ^ kSign) : v;
        // the negated half goes through double on the host and comes back as its 16-bit types
        // write a NaN; the other half is copied as it is
        if constexpr (sizeof(S) == 2) r = negate ? static_cast<S>(host_nan16(r, nan_kind)) : r;
        out[i] = r;
    }
}

// One 16-byte vector of a negated half (the other half is copied as it is).  The sign flips are one XOR per register; the
// values go through double on the host and come back as its 16-bit types write a NaN.  Rare, so behind a wave-uniform test: an
// exponent field of all ones in any of the eight elements, i.e. a NaN or an infinity.
__device__ __forceinline__ void rotate_piece(u32x4& v, bool negate, int nan_kind) {
    if (negate) {
#pragma unroll
        for (int k = 0; k < 4; ++k) v[k] ^= 0x80008000u;
    }
    const std::uint32_t exp_mask = nan_kind == 1 ? 0x7F807F80u : 0x7C007C00u;
    bool special = false;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const std::uint32_t e = v[k] & exp_mask;
        special = special || (e & 0xFFFFu) == (exp_mask & 0xFFFFu) || (e >> 16) == (exp_mask >> 16);
    }
    if (__builtin_amdgcn_ballot_w64(special && negate) != 0) {
        asm volatile("" ::: "memory");
#pragma unroll
        for (int k = 0; k < 4; ++k)
            if (negate) v[k] = host_nan16(v[k] & 0xFFFFu, nan_kind) | (host_nan16(v[k] >> 16, nan_kind) << 16);
    }
}

// 16-bit elements, D a multiple of 16, 16-byte aligned: one 16-byte vector per lane, the
// partner vector sits half a row away.
__global__ __launch_bounds__(kBlock) void rotate_half_vec16(const std::uint16_t* __restrict__ x,
                                                            std::uint16_t* __restrict__ out, long nvec,
                                                            int vec_per_row, int backward, int nan_kind) {
    const int half = vec_per_row / 2;
    const long i = static_cast<long>(blockIdx.x) * kBlock + threadIdx.x;
    if (i >= nvec) return;
    // (64-bit divisions cost a small call more than its memory accesses)
    const int col = static_cast<int>(nvec <= 0xFFFFFFFFL ? static_cast<unsigned>(i) % static_cast<unsigned>(vec_per_row) : i % vec_per_row);
    const bool first = col < half;
    u32x4 v = load16_nt(x + (first ? i + half : i - half) * 8);
    rotate_piece(v, backward ? !first : first, nan_kind);
    store16_nt(out + i * 8, v);
}

// The same for rows of D contiguous elements that lie anywhere: a projection's heads seen as [B, h, S, D], which were copied
// together first (bf16 [1, 32, 1500, 128] and [1, 8, 1500, 128], transposed views: 22.3 us, 12.6 this way).  Strides in pieces (few_dims.h).
template <int ND>
__global__ __launch_bounds__(kBlock) void rotate_half_few_dims(const std::uint16_t* __restrict__ x, std::uint16_t* __restrict__ out, unsigned nvec, int backward, int nan_kind,
                                                               unsigned s1, unsigned s2, unsigned s3, unsigned a0, unsigned a1, unsigned a2) {
    const unsigned i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= nvec) return;
    const unsigned half = s3 / 2, row = i / s3, col = i - row * s3;
    const bool first = col < half;
    std::uint64_t at, unused;
    place_of<ND>(row * s3 + (first ? col + half : col - half), s1, s2, s3, a0, a1, a2, 1, 0, 0, 0, 0, at, unused);
    u32x4 v = load16(x + at * 8);
    rotate_piece(v, backward ? !first : first, nan_kind);
    store16(out + i * 8UL, v);
}
struct RowDims {
    const std::uint16_t* x;
    std::uint16_t* out;
    unsigned nvec;
    int ndim;                    // the last dim is the row, in vectors
    int backward, nan_kind;
    unsigned sizes[8];
    long strides[8];             // elements
};
__global__ __launch_bounds__(kBlock) void rotate_half_rows_vec16(const RowDims s) {
    const unsigned i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= s.nvec) return;
    const unsigned half = s.sizes[s.ndim - 1] / 2;
    unsigned left = i / s.sizes[s.ndim - 1];
    const unsigned col = i - left * s.sizes[s.ndim - 1];
    const bool first = col < half;
    long at = static_cast<long>(first ? col + half : col - half) * 8;
    for (int d = s.ndim - 2; d >= 0; --d) {
        const unsigned q = left / s.sizes[d];
        at += static_cast<long>(left - q * s.sizes[d]) * s.strides[d];
        left = q;
    }
    u32x4 v = load16(s.x + at);
    rotate_piece(v, s.backward ? !first : first, s.nan_kind);
    store16(s.out + static_cast<long>(i) * 8, v);
}

int stream_grid(long work_items_per_block_iter, long total) {
    int dev = 0;
    (void)hipGetDevice(&dev);
    auto* st = DeviceContext::instance().device(dev);
    const long cus = st ? st->compute_units : 256;
    const long cap = cus * 8;
    const long need = (total + work_items_per_block_iter - 1) / work_items_per_block_iter;
    const long g = need < cap ? need : cap;
    return static_cast<int>(g < 1 ? 1 : g);
}

template <typename T>
int launch_swiglu_fwd(const void* gate, const void* up, void* out, long n, hipStream_t s) {
    using S = typename Elem<T>::store_t;
    constexpr int V = Elem<T>::kVec;
    const auto* g = static_cast<const S*>(gate);
    const auto* u = static_cast<const S*>(up);
    auto* o = static_cast<S*>(out);
    const bool aligned = ((reinterpret_cast<uintptr_t>(gate) | reinterpret_cast<uintptr_t>(up) |
                           reinterpret_cast<uintptr_t>(out)) % 16) == 0;
    if (aligned && n >= V) {
        // Four vectors per lane keep enough bytes under way where there are waves enough; with fewer the arithmetic of one vector
        // after the other decides, for longer where it is the two tiers of 16-bit results (bf16, four / one: 14336 vectors 5.3 / 2.9 us,
        // 131072 6.5 / 4.0, 524288 8.4 / 7.1; fp32: 14336 3.4 / 2.3, 262144 4.9 / 4.6, 672000 8.3 / 8.8).
        const long nvec = n / V;
        const int unroll = nvec <= (sizeof(S) == 2 ? 1 << 20 : 1 << 18) ? 1 : 4;
        long blocks = (nvec + kBlock * unroll - 1) / (kBlock * unroll);
        if (blocks > 0x7fffffffL) blocks = 0x7fffffffL;  // the kernel grid-strides beyond that
        const dim3 grid(static_cast<unsigned>(blocks));
        const int tail = static_cast<int>(n - nvec * V);
        if (unroll == 1) hipLaunchKernelGGL((swiglu_fwd_vec<T, 1>), grid, dim3(kBlock), 0, s, g, u, o, nvec, tail);
        else             hipLaunchKernelGGL((swiglu_fwd_vec<T, 4>), grid, dim3(kBlock), 0, s, g, u, o, nvec, tail);
    } else {
        hipLaunchKernelGGL((swiglu_fwd_any<T>), dim3(stream_grid(kBlock, n)), dim3(kBlock), 0, s, g, u, o, n);
    }
    PARAS_HIP_TRY(hipGetLastError());
    return PARAS_OK;
}

template <typename T>
int launch_swiglu_bwd(const void* go, const void* gate, const void* up, void* ggate, void* gup, long n,
                      hipStream_t s) {
    using S = typename Elem<T>::store_t;
    const auto* d = static_cast<const S*>(go);
    const auto* g = static_cast<const S*>(gate);
    const auto* u = static_cast<const S*>(up);
    auto* og = static_cast<S*>(ggate);
    auto* ou = static_cast<S*>(gup);
    if constexpr (sizeof(S) == 2) {
        const bool aligned = ((reinterpret_cast<uintptr_t>(go) | reinterpret_cast<uintptr_t>(gate) | reinterpret_cast<uintptr_t>(up) |
                               reinterpret_cast<uintptr_t>(ggate) | reinterpret_cast<uintptr_t>(gup)) % 16) == 0;
        if (aligned && n >= 8) {
            const long nvec = n / 8;
            long blocks = (nvec + kBlock - 1) / kBlock;
            if (blocks > 0x7fffffffL) blocks = 0x7fffffffL;  // the kernel grid-strides beyond that
            hipLaunchKernelGGL((swiglu_bwd_vec<T>), dim3(static_cast<unsigned>(blocks)), dim3(kBlock), 0, s, d, g, u, og, ou, nvec,
                               static_cast<int>(n - nvec * 8));
            PARAS_HIP_TRY(hipGetLastError());
            return PARAS_OK;
        }
    }
    hipLaunchKernelGGL((swiglu_bwd_any<T>), dim3(stream_grid(kBlock, n)), dim3(kBlock), 0, s, d, g, u, og, ou, n);
    PARAS_HIP_TRY(hipGetLastError());
    return PARAS_OK;
}

}  // namespace
}  // namespace paras

extern "C" {

int paras_swiglu_fwd(const void* gate, const void* up, void* out, int64_t n, int dtype, void* stream) {
    using namespace paras;
    PARAS_REQUIRE(n >= 0, "paras_swiglu_fwd: negative size");
    if (n == 0) return PARAS_OK;
    PARAS_REQUIRE(gate && up && out, "paras_swiglu_fwd: null pointer");
    hipStream_t s = nullptr;
    int rc = resolve_stream(stream, &s);
    if (rc != PARAS_OK) return rc;
    switch (dtype) {
        case PARAS_F32:  return launch_swiglu_fwd<float>(gate, up, out, n, s);
        case PARAS_F64:  return launch_swiglu_fwd<double>(gate, up, out, n, s);
        case PARAS_BF16: return launch_swiglu_fwd<bf16_t>(gate, up, out, n, s);
        case PARAS_F16:  return launch_swiglu_fwd<f16_t>(gate, up, out, n, s);
        default: return fail(PARAS_ERR_INVALID, "paras_swiglu_fwd: unknown dtype %d", dtype);
    }
}

int paras_swiglu_bwd(const void* grad_out, const void* gate, const void* up, void* grad_gate,
                     void* grad_up, int64_t n, int dtype, void* stream) {
    using namespace paras;
    PARAS_REQUIRE(n >= 0, "paras_swiglu_bwd: negative size");
    if (n == 0) return PARAS_OK;
    PARAS_REQUIRE(grad_out && gate && up && grad_gate && grad_up, "paras_swiglu_bwd: null pointer");
    hipStream_t s = nullptr;
    int rc = resolve_stream(stream, &s);
    if (rc != PARAS_OK) return rc;
    switch (dtype) {
        case PARAS_F32:  return launch_swiglu_bwd<float>(grad_out, gate, up, grad_gate, grad_up, n, s);
        case PARAS_F64:  return launch_swiglu_bwd<double>(grad_out, gate, up, grad_gate, grad_up, n, s);
        case PARAS_BF16: return launch_swiglu_bwd<bf16_t>(grad_out, gate, up, grad_gate, grad_up, n, s);
        case PARAS_F16:  return launch_swiglu_bwd<f16_t>(grad_out, gate, up, grad_gate, grad_up, n, s);
        default: return fail(PARAS_ERR_INVALID, "paras_swiglu_bwd: unknown dtype %d", dtype);
    }
}

int paras_rotate_half(const void* x, void* out, int64_t rows, int64_t D, int backward, int dtype,
                      void* stream) {
    using namespace paras;
    PARAS_REQUIRE(rows >= 0 && D >= 0, "paras_rotate_half: negative shape");
    PARAS_REQUIRE(D % 2 == 0, "paras rotate_half: last dimension must be even");
    const long n = rows * D;
    if (n == 0) return PARAS_OK;
    PARAS_REQUIRE(x && out, "paras_rotate_half: null pointer");
    hipStream_t s = nullptr;
    int rc = resolve_stream(stream, &s);
    if (rc != PARAS_OK) return rc;
    const dim3 grid(stream_grid(kBlock, n)), block(kBlock);
    switch (dtype) {
        case PARAS_F32:
            hipLaunchKernelGGL((rotate_half_any<uint32_t>), grid, block, 0, s, static_cast<const uint32_t*>(x),
                               static_cast<uint32_t*>(out), n, (long)D, backward, 0);
            break;
        case PARAS_F64:
            hipLaunchKernelGGL((rotate_half_any<uint64_t>), grid, block, 0, s, static_cast<const uint64_t*>(x),
                               static_cast<uint64_t*>(out), n, (long)D, backward, 0);
            break;
        case PARAS_BF16:
        case PARAS_F16:
            if (D % 16 == 0 && D / 8 <= 0x7fffffff && n / 8 <= 0x7fffffffL * kBlock &&
                ((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(out)) & 15) == 0) {
                const long nvec = n / 8;
                hipLaunchKernelGGL(rotate_half_vec16, dim3(static_cast<unsigned>((nvec + kBlock - 1) / kBlock)), block, 0, s,
                                   static_cast<const uint16_t*>(x), static_cast<uint16_t*>(out), nvec,
                                   static_cast<int>(D / 8), backward, dtype == PARAS_BF16 ? 1 : 2);
            } else {
                hipLaunchKernelGGL((rotate_half_any<uint16_t>), grid, block, 0, s, static_cast<const uint16_t*>(x),
                                   static_cast<uint16_t*>(out), n, (long)D, backward, dtype == PARAS_BF16 ? 1 : 2);
            }
            break;
        default: return fail(PARAS_ERR_INVALID, "paras_rotate_half: unknown dtype %d", dtype);
    }
    PARAS_HIP_TRY(hipGetLastError());
    return PARAS_OK;
}

int paras_rotate_half_strided(const void* x, void* out, int ndim, const int64_t* sizes, const int64_t* strides, int backward, int dtype,
                              void* stream) {
    using namespace paras;
    PARAS_REQUIRE(dtype == PARAS_BF16 || dtype == PARAS_F16, "paras_rotate_half_strided: 16-bit dtypes only");
    PARAS_REQUIRE(ndim >= 1 && ndim <= 8 && sizes && strides, "paras_rotate_half_strided: 1 to 8 dimensions");
    PARAS_REQUIRE(sizes[ndim - 1] % 16 == 0 && strides[ndim - 1] == 1, "paras_rotate_half_strided: rows of a multiple of 16 contiguous elements");
    RowDims d{};
    long n = 1;
    for (int k = 0; k < ndim; ++k) {
        PARAS_REQUIRE(sizes[k] >= 0 && (k == ndim - 1 || strides[k] % 8 == 0), "paras_rotate_half_strided: rows that begin on 16 bytes");
        n *= sizes[k];
        if (k + 1 < ndim && sizes[k] == 1) continue;
        if (k + 1 < ndim && d.ndim > 0 && d.strides[d.ndim - 1] == strides[k] * sizes[k]) {        // one dimension with the one before
            d.sizes[d.ndim - 1] *= static_cast<unsigned>(sizes[k]);
            d.strides[d.ndim - 1] = strides[k];
            continue;
        }
        d.sizes[d.ndim] = static_cast<unsigned>(k + 1 < ndim ? sizes[k] : sizes[k] / 8);
        d.strides[d.ndim++] = strides[k];
    }
    if (n == 0) return PARAS_OK;
    PARAS_REQUIRE(x && out, "paras_rotate_half_strided: null pointer");
    PARAS_REQUIRE(((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(out)) & 15) == 0, "paras_rotate_half_strided: operands must be 16-byte aligned");
    PARAS_REQUIRE(n / 8 < (1L << 31), "paras_rotate_half_strided: at most 2^34 elements");
    hipStream_t s = nullptr;
    int rc = resolve_stream(stream, &s);
    if (rc != PARAS_OK) return rc;
    d.x = static_cast<const uint16_t*>(x);
    d.out = static_cast<uint16_t*>(out);
    d.nvec = static_cast<unsigned>(n / 8);
    d.backward = backward;
    d.nan_kind = dtype == PARAS_BF16 ? 1 : 2;
    const dim3 grid((d.nvec + kBlock - 1) / kBlock), block(kBlock);
    Dims few;
    long row_sizes[8];
    for (int k = 0; k < d.ndim; ++k) row_sizes[k] = k + 1 < d.ndim ? static_cast<long>(d.sizes[k]) : static_cast<long>(d.sizes[k]) * 8;
    if (few_dims(d.ndim, row_sizes, d.strides, d.strides, n / 8, 8, &few)) {
        auto launch = [&](auto dims) {
            hipLaunchKernelGGL((rotate_half_few_dims<decltype(dims)::value>), grid, block, 0, s, d.x, d.out, d.nvec, backward, d.nan_kind, few.sizes[1], few.sizes[2],
                               few.sizes[3], few.a[0], few.a[1], few.a[2]);
        };
        if (d.ndim <= 2)      launch(std::integral_constant<int, 2>{});             // (a lone row: in front of it a dimension of size 1)
        else if (d.ndim == 3) launch(std::integral_constant<int, 3>{});
        else                  launch(std::integral_constant<int, 4>{});
    } else {
        hipLaunchKernelGGL(rotate_half_rows_vec16, grid, block, 0, s, d);
    }
    PARAS_HIP_TRY(hipGetLastError());
    return PARAS_OK;
}

}  // extern "C"
