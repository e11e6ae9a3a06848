// aten::linear / mm / bmm / addmm for the `paras` device (and through them nn.Linear,
// torch.matmul).  The reference copies both operands to the host, runs the
// ATen-CPU GEMM and copies the result back (csrc/ops/vision_ops.cpp:388-423,
// 248-309); here every float product runs on the device (paras_gemm: fp32
// accumulation -- fp64 for fp64 tensors -- and one rounding, as ATen-CPU does).
// Integer and mixed-dtype products are not part of this surface and raise.
#include "paras_torch.h"

#include <ATen/NativeFunctions.h>
#include <torch/csrc/autograd/custom_function.h>

#include <exception>

namespace paras_torch {
namespace {

using at::Tensor;

bool is_16bit_float(const Tensor& t) { return t.scalar_type() == c10::kBFloat16 || t.scalar_type() == c10::kHalf; }
bool is_float(const Tensor& t) {
    return is_16bit_float(t) || t.scalar_type() == c10::kFloat || t.scalar_type() == c10::kDouble;
}

void check_dtypes(const Tensor& a, const Tensor& b, const char* what) {
    require_same_device(what, a, {{"mat2", &b}});
    TORCH_CHECK(a.scalar_type() == b.scalar_type(), "paras ", what, ": operand dtypes differ");
    TORCH_CHECK(is_float(a), "paras ", what, ": only float dtypes (fp32, fp64, bf16, fp16) are supported on the device");
}

// An operand [.., rows, K] of a product as the library reads it: contiguous along the contraction, or along
// its rows (a transposed view: the weight in dy W, both operands of dy^T x).  `swap`: t is given as
// [.., K, rows].  A view that is neither, or that the 16-bit kernels cannot read (16-byte boundaries), is copied.
struct Operand {
    Tensor hold;                // owns the memory where the operand was copied
    const void* p = nullptr;
    int64_t ld = 0, batch_stride = 0;
    bool rows = false;
};
Operand operand(const Tensor& t, bool swap, bool may_be_rows) {
    const bool batched = t.dim() == 3;
    const int64_t R = t.size(swap ? -1 : -2), K = t.size(swap ? -2 : -1);
    const int64_t sr = t.stride(swap ? -1 : -2), sk = t.stride(swap ? -2 : -1);
    const auto up8 = [](int64_t n) { return (n + 7) / 8 * 8; };
    const int64_t ld_k = R > 1 ? sr : up8(K), ld_r = K > 1 ? sk : up8(R);                  // (a lone row has no stride)
    const bool along_k = (sk == 1 || K <= 1) && ld_k >= K, along_r = (sr == 1 || R <= 1) && ld_r >= R;
    const int64_t bs = batched ? t.stride(0) : 0;
    const bool wants16 = is_16bit_float(t), base_ok = !wants16 || ((reinterpret_cast<uintptr_t>(t.data_ptr()) & 15) == 0 && bs % 8 == 0);
    auto readable = [&](int64_t ld) { return base_ok && (!wants16 || ld % 8 == 0); };
    may_be_rows = may_be_rows && K > 0 && K < (1L << 30) && ld_r <= (1L << 21) && (!batched || t.size(0) <= 65535);
    if (along_k && readable(ld_k)) return {Tensor(), t.data_ptr(), ld_k, bs, false};
    if (along_r && may_be_rows && readable(ld_r)) return {Tensor(), t.data_ptr(), ld_r, bs, true};
    if (along_k && (K % 8 != 0 || t.is_contiguous())) return {Tensor(), t.data_ptr(), ld_k, bs, false};   // a dense copy would be no better aligned
    Tensor c = (swap ? t.transpose(-1, -2) : t).contiguous();
    return {c, c.data_ptr(), R > 1 ? K : up8(K), batched ? R * K : 0, false};
}

// Memory for a product's partial sums, allocated when the library says how much; what the allocator throws does not
// pass through the library.
struct Partials {
    Tensor hold;
    c10::Device device;
    std::exception_ptr failed;
    static void* allocate(void* self, size_t nbytes) noexcept {
        auto* p = static_cast<Partials*>(self);
        try {
            p->hold = workspace(nbytes, p->device);
            return p->hold.data_ptr();
        } catch (...) {
            p->failed = std::current_exception();
            return nullptr;
        }
    }
};

// out[b] = alpha * a[b] mat2[b] + beta * addend[b], a [.., M, K], into a dense tensor of `shape`.  mat2 is
// [.., K, N], or [.., N, K] with `mat2_nk`; a is [.., K, M] with `a_km`.
Tensor run_gemm(const Tensor& a_in, bool a_km, const Tensor& mat2, bool mat2_nk, const Tensor* addend, double alpha, double beta, int64_t batch,
                c10::IntArrayRef shape) {
    const int64_t M = a_in.size(a_km ? -1 : -2), K = a_in.size(a_km ? -2 : -1), N = mat2.size(mat2_nk ? -2 : -1);
    Tensor out = empty_paras(shape, a_in.scalar_type(), a_in.device());
    if (out.numel() == 0) return out;
    const int code = require_float_code(a_in, "paras gemm");
    // Rows-contiguous operands: not for fp64; A only together with B; and for 16-bit tensors with one of each the
    // contraction in whole chunks of 8.
    Operand b = operand(mat2, !mat2_nk, code != PARAS_F64);
    Operand a = operand(a_in, a_km, b.rows);
    if (b.rows && !a.rows && is_16bit_float(a_in) && K % 8 != 0) b = operand(mat2, !mat2_nk, false);
    Tensor add;
    paras_gemm_args g{};
    if (addend != nullptr && addend->defined() && beta != 0.0) {
        g.addend = addend->data_ptr();
        if (!(addend->dim() == 1 && addend->size(0) == N && addend->stride(0) == 1)) {
            add = addend->expand({M, N});                    // [1, N] -> row stride 0; full matrix -> its stride
            if (add.stride(-1) != 1 || (add.stride(-2) != 0 && add.stride(-2) < N)) add = add.contiguous();
            g.addend = add.data_ptr();
            g.ld_add = add.stride(-2);
        }
    }
    g.a = a.p; g.b = b.p; g.c = out.data_ptr();
    g.M = M; g.N = N; g.K = K;
    g.lda = a.ld; g.ldb = b.ld; g.ldc = N;
    g.batch = batch >= 0 ? batch : 1;
    g.stride_a = a.batch_stride; g.stride_b = b.batch_stride; g.stride_c = M * N;
    g.alpha = alpha; g.beta = beta; g.dtype = code;
    g.a_rows = a.rows; g.b_rows = b.rows;
    // products with few tiles run faster with a workspace for the partial sums of a split contraction
    Partials partials{Tensor(), a_in.device(), nullptr};
    const int rc = paras_gemm_scratch(&g, &Partials::allocate, &partials, stream_for(a_in));
    if (partials.failed) std::rethrow_exception(partials.failed);
    check(rc);
    return out;
}

Tensor mm(const Tensor& self, const Tensor& mat2) {
    TORCH_CHECK(self.dim() == 2 && mat2.dim() == 2, "paras mm: both arguments must be 2-D");
    TORCH_CHECK(self.size(1) == mat2.size(0), "paras mm: shapes cannot be multiplied (", self.size(0), "x", self.size(1), " and ",
                mat2.size(0), "x", mat2.size(1), ")");
    check_dtypes(self, mat2, "mm");
    return run_gemm(self, false, mat2, false, nullptr, 1.0, 0.0, -1, {self.size(0), mat2.size(1)});
}

Tensor bmm(const Tensor& self, const Tensor& mat2) {
    TORCH_CHECK(self.dim() == 3 && mat2.dim() == 3, "paras bmm: both arguments must be 3-D");
    TORCH_CHECK(self.size(0) == mat2.size(0) && self.size(2) == mat2.size(1), "paras bmm: shapes cannot be multiplied");
    check_dtypes(self, mat2, "bmm");
    return run_gemm(self, false, mat2, false, nullptr, 1.0, 0.0, self.size(0), {self.size(0), self.size(1), mat2.size(2)});
}

Tensor addmm(const Tensor& self, const Tensor& mat1, const Tensor& mat2, const at::Scalar& beta, const at::Scalar& alpha) {
    TORCH_CHECK(mat1.dim() == 2 && mat2.dim() == 2, "paras addmm: matrices must be 2-D");
    TORCH_CHECK(mat1.size(1) == mat2.size(0), "paras addmm: shapes cannot be multiplied");
    check_dtypes(mat1, mat2, "addmm");
    TORCH_CHECK(self.scalar_type() == mat1.scalar_type(), "paras addmm: operand dtypes differ");
    require_same_device("addmm", mat1, {{"self", &self}});
    return run_gemm(mat1, false, mat2, false, &self, alpha.toDouble(), beta.toDouble(), -1, {mat1.size(0), mat2.size(1)});
}

// ---- aten::linear, registered above autograd.  The composite makes a transposed view, flattens the leading
// dimensions and calls mm / addmm, and its backward is two products with transposed operands and, for a
// bias, a sum this device has no op for (the gradient crossed to the host).  Here the forward is one call and
// one autograd node holds the backward.  Operands the composite would treat otherwise go to it.
Tensor rows_of(const Tensor& x) { return x.dim() == 2 ? x : x.reshape({-1, x.size(-1)}); }

Tensor linear_forward(const Tensor& x, const Tensor& w, const Tensor& bias) {
    at::DimVector shape(x.sizes());
    shape.back() = w.size(0);
    return run_gemm(rows_of(x), false, w, true, &bias, 1.0, 1.0, -1, shape);
}

Tensor column_sum(const Tensor& t) {
    const Tensor x = t.stride(-1) == 1 && (t.size(0) <= 1 || t.stride(0) >= t.size(1)) ? t : t.contiguous();
    Tensor out = empty_paras({x.size(1)}, x.scalar_type(), x.device());
    if (out.numel() == 0) return out;
    const int code = require_float_code(x, "paras linear");
    Tensor ws = workspace(paras_column_sum_workspace(x.size(0), x.size(1), code), x.device());
    check(paras_column_sum(x.data_ptr(), out.data_ptr(), x.size(0), x.size(1), x.size(0) > 1 ? x.stride(0) : x.size(1), code, ws.data_ptr(),
                           stream_for(x)));
    return out;
}

struct LinearFunction : torch::autograd::Function<LinearFunction> {
    static Tensor forward(torch::autograd::AutogradContext* ctx, const Tensor& x, const Tensor& w, const c10::optional<Tensor>& bias) {
        ctx->save_for_backward({w.requires_grad() ? x : Tensor(), x.requires_grad() ? w : Tensor()});
        if (bias.has_value()) ctx->saved_data["bias"] = true;
        return linear_forward(x, w, bias.has_value() ? *bias : Tensor());
    }
    static torch::autograd::variable_list backward(torch::autograd::AutogradContext* ctx, const torch::autograd::variable_list& grads) {
        const auto saved = ctx->get_saved_variables();
        const Tensor &x = saved[0], &w = saved[1];
        const Tensor dy = rows_of(grads[0]);
        at::DimVector x_sizes(grads[0].sizes());
        if (w.defined()) x_sizes.back() = w.size(1);
        const bool want_x = ctx->needs_input_grad(0), want_w = ctx->needs_input_grad(1);
        const bool want_b = ctx->saved_data.count("bias") != 0 && ctx->needs_input_grad(2);
        Tensor gx, gw, gb;
        // a graph of the backward is wanted, or a gradient is a batch of gradients, a dual tensor or wrapped: dispatcher ops
        const bool composite = at::GradMode::is_enabled() || !plain(dy) || (want_x && !plain(w)) || (want_w && !plain(x));
        if (composite) {
            if (want_x) gx = at::mm(dy, w).view(x_sizes);
            if (want_w) gw = at::mm(dy.t(), rows_of(x));
            if (want_b) gb = dy.sum(0);
        } else {
            if (want_x) gx = run_gemm(dy, false, w, false, nullptr, 1.0, 0.0, -1, x_sizes);
            if (want_w) gw = run_gemm(dy, true, rows_of(x), false, nullptr, 1.0, 0.0, -1, {dy.size(1), x.size(-1)});
            if (want_b) gb = column_sum(dy);
        }
        return {gx, gw, gb};
    }
};

Tensor linear(const Tensor& x, const Tensor& w, const c10::optional<Tensor>& bias_opt) {
    const Tensor bias = bias_opt.has_value() ? *bias_opt : Tensor();
    auto alike = [&](const Tensor& t) {
        return is_paras(t) && t.device() == x.device() && t.scalar_type() == x.scalar_type() && plain(t);
    };
    const bool direct = x.dim() >= 1 && w.dim() == 2 && is_float(x) && alike(x) && alike(w) && x.size(-1) == w.size(1) && w.numel() > 0 &&
                        x.numel() > 0 && (!bias.defined() || (alike(bias) && bias.dim() == 1 && bias.size(0) == w.size(0)));
    if (!direct) return at::native::linear(x, w, bias_opt);
    return needs_grad(x, w, bias) ? LinearFunction::apply(x, w, bias.defined() ? c10::optional<Tensor>(bias) : c10::nullopt) : linear_forward(x, w, bias);
}

}  // namespace

TORCH_LIBRARY_IMPL(aten, PrivateUse1, m) {
    m.impl("mm", mm);
    m.impl("bmm", bmm);
    m.impl("addmm", addmm);
    m.impl("linear", linear);
}
TORCH_LIBRARY_IMPL(aten, AutogradPrivateUse1, m) { m.impl("linear", linear); }

}  // namespace paras_torch
