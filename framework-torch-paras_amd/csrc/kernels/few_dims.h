// Elements of strided tensors of few dimensions, found without a loop over them.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace paras {

// Up to four dimensions, fewer than 2^31 elements and strides below 2^32: the number of dimensions is the kernel's, and sizes and strides are arguments of
// their own (the last dimension's at index 3), in registers when a wave starts.  A loop over dimensions fetches each one's from memory in turn, which a
// kernel of a few us has nothing to hide behind (bf16, a decode step's new keys into the cache, [8, 8, 1, 128]: 2.0 to 2.6 us, this way 1.2 to 1.5; the
// decoder block of eight sequences around it, with binary_unit8, 151.8 -> 147.2).  Strides in whatever unit the kernel moves.
struct Dims {
    unsigned sizes[4] = {1, 1, 1, 1}, a[4] = {}, b[4] = {};
};
// The place of element i in both tensors; the outermost dimension is what is left.
template <int ND>
__device__ __forceinline__ void place_of(unsigned i, unsigned s1, unsigned s2, unsigned s3, unsigned a0, unsigned a1, unsigned a2, unsigned a3, unsigned b0, unsigned b1,
                                         unsigned b2, unsigned b3, std::uint64_t& ao, std::uint64_t& bo) {
    auto times = [](unsigned c, unsigned stride) { return static_cast<std::uint64_t>(c) * stride; };
    unsigned q = i / s3, c = i - q * s3;
    ao = times(c, a3);
    bo = times(c, b3);
    if constexpr (ND >= 3) {
        const unsigned left = q;
        q = left / s2;
        c = left - q * s2;
        ao += times(c, a2);
        bo += times(c, b2);
    }
    if constexpr (ND >= 4) {
        const unsigned left = q;
        q = left / s1;
        c = left - q * s1;
        ao += times(c, a1);
        bo += times(c, b1);
    }
    ao += times(q, ND == 4 ? a0 : ND == 3 ? a1 : a2);
    bo += times(q, ND == 4 ? b0 : ND == 3 ? b1 : b2);
}
// Whether `ndim` dimensions of `sizes` and non-negative strides, in units of `unit` elements (which divides the strides of all but the last dimension, whose own
// stride is taken to be one unit if unit > 1), fit the kernels above; then also as Dims.
inline bool few_dims(int ndim, const long* sizes, const long* a, const long* b, long n, long unit, Dims* d) {
    if (ndim > 4 || n >= (1L << 31)) return false;
    *d = Dims{};
    for (int k = 0; k < ndim; ++k) {
        const bool row = k == ndim - 1 && unit > 1;
        const long as = row ? 1 : a[k] / unit, bs = row ? 1 : b[k] / unit;
        if (as < 0 || bs < 0 || as > 0xFFFFFFFFL || bs > 0xFFFFFFFFL) return false;
        d->sizes[4 - ndim + k] = static_cast<unsigned>(row ? sizes[k] / unit : sizes[k]);
        d->a[4 - ndim + k] = static_cast<unsigned>(as);
        d->b[4 - ndim + k] = static_cast<unsigned>(bs);
    }
    return true;
}

}  // namespace paras
