// Sums of a matrix's columns: the bias gradient of a linear layer (the reference's
// LinearFunction::backward sums grad_output over its rows on the host, csrc/ops/vision_ops.cpp:280-309).
//
// Bound by reading the matrix once.  A thread adds 16 bytes' worth of adjacent columns down a slab of
// rows, eight rows in flight, and stores the partial sums; a second kernel adds the slabs in order and narrows
// once.  Slabs make about two workgroups per CU whatever the shape.  Sums of a slab in fp32 for the
// 16-bit types and in fp64 for fp32 and fp64 rows, between slabs in fp64.
#include <hip/hip_runtime.h>

#include <type_traits>

#include "core/device_context.h"
#include "core/device_math.h"
#include "core/status.h"
#include "paras_hip.h"

namespace paras {
namespace {

constexpr int kBlock = 256;

template <typename T> using SlabSum = typename std::conditional<sizeof(typename Elem<T>::store_t) == 2, float, double>::type;

// V elements per thread: 16 bytes, or 1 where rows are not made of aligned 16-byte pieces
template <typename T, int V>
__global__ __launch_bounds__(kBlock) void column_sum_slab_kernel(const typename Elem<T>::store_t* __restrict__ x, double* __restrict__ partial,
                                                                 long rows, long cols, long ld, long per_slab) {
    using S = typename Elem<T>::store_t;
    using Acc = SlabSum<T>;
    const long c = (static_cast<long>(blockIdx.x) * kBlock + threadIdx.x) * V;
    if (c >= cols) return;
    const long r0 = static_cast<long>(blockIdx.y) * per_slab, r1 = r0 + per_slab < rows ? r0 + per_slab : rows;
    struct __attribute__((aligned(sizeof(S) * V))) Piece { S e[V]; };
    Acc acc[V];
#pragma unroll
    for (int v = 0; v < V; ++v) acc[v] = 0;
    auto add = [&](const Piece& p) {
#pragma unroll
        for (int v = 0; v < V; ++v) {
            if constexpr (sizeof(Acc) == 4) acc[v] += Elem<T>::to_f32(p.e[v]);
            else                            acc[v] += Elem<T>::to_f64(p.e[v]);
        }
    };
    long r = r0;
    for (; r + 8 <= r1; r += 8) {
        Piece p[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) p[u] = *reinterpret_cast<const Piece*>(x + (r + u) * ld + c);
#pragma unroll
        for (int u = 0; u < 8; ++u) add(p[u]);
    }
    for (; r < r1; ++r) add(*reinterpret_cast<const Piece*>(x + r * ld + c));
#pragma unroll
    for (int v = 0; v < V; ++v) partial[static_cast<long>(blockIdx.y) * cols + c + v] = static_cast<double>(acc[v]);
}

template <typename T>
__global__ __launch_bounds__(kBlock) void column_sum_finish_kernel(const double* __restrict__ partial, typename Elem<T>::store_t* __restrict__ out,
                                                                   long cols, long slabs) {
    const long c = static_cast<long>(blockIdx.x) * kBlock + threadIdx.x;
    if (c >= cols) return;
    double t = 0.0;
    long s = 0;
    for (; s + 8 <= slabs; s += 8) {
        double v[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) v[u] = partial[(s + u) * cols + c];
#pragma unroll
        for (int u = 0; u < 8; ++u) t += v[u];
    }
    for (; s < slabs; ++s) t += partial[s * cols + c];
    out[c] = Elem<T>::from_f64(t);
}

// rows per slab: about 512 workgroups in all, at least 8 rows each and at most 256 slabs
long slab_rows(long rows, long cols, int elem_bytes) {
    const long groups = (cols * elem_bytes / 16 + kBlock - 1) / kBlock;
    long slabs = 512 / (groups > 0 ? groups : 1);
    if (slabs > 256) slabs = 256;
    if (slabs < 1) slabs = 1;
    const long per = (rows + slabs - 1) / slabs;
    return per < 8 ? 8 : per;
}
int elem_bytes(int dtype) { return dtype == PARAS_F64 ? 8 : dtype == PARAS_F32 ? 4 : 2; }

template <typename T>
int launch(const void* x, void* out, void* ws, long rows, long cols, long ld, hipStream_t s) {
    using S = typename Elem<T>::store_t;
    constexpr int V = 16 / static_cast<int>(sizeof(S));
    const long per = slab_rows(rows, cols, sizeof(S)), slabs = (rows + per - 1) / per;
    auto* partial = static_cast<double*>(ws);
    const bool vec = cols % V == 0 && ld % V == 0 && (reinterpret_cast<uintptr_t>(x) & 15) == 0;
    const long per_wg = kBlock * (vec ? V : 1);
    const dim3 g(static_cast<unsigned>((cols + per_wg - 1) / per_wg), static_cast<unsigned>(slabs));
    if (vec) hipLaunchKernelGGL((column_sum_slab_kernel<T, V>), g, dim3(kBlock), 0, s, static_cast<const S*>(x), partial, rows, cols, ld, per);
    else     hipLaunchKernelGGL((column_sum_slab_kernel<T, 1>), g, dim3(kBlock), 0, s, static_cast<const S*>(x), partial, rows, cols, ld, per);
    PARAS_HIP_TRY(hipGetLastError());
    hipLaunchKernelGGL((column_sum_finish_kernel<T>), dim3(static_cast<unsigned>((cols + kBlock - 1) / kBlock)), dim3(kBlock), 0, s, partial,
                       static_cast<S*>(out), cols, slabs);
    PARAS_HIP_TRY(hipGetLastError());
    return PARAS_OK;
}

}  // namespace
}  // namespace paras

extern "C" {

size_t paras_column_sum_workspace(int64_t rows, int64_t cols, int dtype) {
    if (rows <= 0 || cols <= 0) return 0;
    const long per = paras::slab_rows(rows, cols, paras::elem_bytes(dtype));
    return static_cast<size_t>((rows + per - 1) / per) * static_cast<size_t>(cols) * sizeof(double);
}

int paras_column_sum(const void* x, void* out, int64_t rows, int64_t cols, int64_t ld, int dtype, void* workspace, void* stream) {
    using namespace paras;
    PARAS_REQUIRE(rows >= 0 && cols >= 0 && ld >= cols, "paras_column_sum: bad shape");
    if (cols == 0) return PARAS_OK;
    hipStream_t s = nullptr;
    int rc = resolve_stream(stream, &s);
    if (rc != PARAS_OK) return rc;
    if (rows == 0) {
        const int64_t one = 1;
        return paras_fill_strided(out, 1, &cols, &one, elem_bytes(dtype), 0, stream);
    }
    PARAS_REQUIRE(x && out && workspace, "paras_column_sum: null pointer");
    switch (dtype) {
        case PARAS_F32:  return launch<float>(x, out, workspace, rows, cols, ld, s);
        case PARAS_F64:  return launch<double>(x, out, workspace, rows, cols, ld, s);
        case PARAS_BF16: return launch<bf16_t>(x, out, workspace, rows, cols, ld, s);
        case PARAS_F16:  return launch<f16_t>(x, out, workspace, rows, cols, ld, s);
        default: return fail(PARAS_ERR_INVALID, "paras_column_sum: unknown dtype %d", dtype);
    }
}

}  // extern "C"
