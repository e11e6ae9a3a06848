"""Dense NT GEMM (mm / bmm / addmm / linear on the device) through the C ABI.

The reference runs these on ATen-CPU with fp32 accumulation and one rounding
(csrc/ops/vision_ops.cpp:248-309,388-423); the oracle's matmul_nt accumulates
in double and rounds once.  Bar: every element within one 16-bit ulp of the
oracle (summation order is the only difference), and torch-CPU addmm / linear
as the library check for the epilogue.
"""
import ctypes as C
import math

import pytest
import torch

import capi
import oracle as O

pytestmark = pytest.mark.gpu


def ulp16(ref, dtype):
    mant = 7 if dtype == torch.bfloat16 else 10
    a = ref.double().abs().clamp_min(2.0 ** -14)
    return torch.exp2(torch.floor(torch.log2(a)) - mant)


def assert_gemm_close(out, ref, dtype):
    err = (out.double().cpu() - ref.double()).abs()
    tol = ulp16(ref, dtype) * 1.001 + 1e-6
    assert bool((err <= tol).all()), f"worst {err.max().item():.3e}, {(err > tol).sum().item()} beyond one ulp"


SHAPES = [(128, 256, 64), (1, 8, 64), (130, 257, 128), (300, 100, 192), (512, 1024, 1024), (77, 4096, 320),
          (4100, 2100, 64)]     # the last one: 256-row tiles with a single k-tile


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("shape", SHAPES)
def test_gemm_nt_matches_oracle(shape, dtype):
    M, N, K = shape
    torch.manual_seed(M * 7 + N * 3 + K)
    a, b = torch.randn(M, K).to(dtype), (0.1 * torch.randn(N, K)).to(dtype)
    out = capi.gemm_nt(a.cuda(), b.cuda())
    assert_gemm_close(out, O.matmul_nt(a, b), dtype)


def test_gemm_nt_bias_and_addmm_epilogue():
    torch.manual_seed(1)
    M, N, K = 200, 384, 256
    dt = torch.bfloat16
    a, w, bias = torch.randn(M, K).to(dt), (0.05 * torch.randn(N, K)).to(dt), torch.randn(N).to(dt)
    out = capi.gemm_nt(a.cuda(), w.cuda(), bias.cuda())
    assert_gemm_close(out, torch.nn.functional.linear(a, w, bias), dt)        # library check: x W^T + b
    self_ = torch.randn(M, N).to(dt)
    out = capi.gemm_nt(a.cuda(), w.cuda(), self_.cuda(), alpha=0.5, beta=2.0)
    exact = 0.5 * (a.double() @ w.double().t()) + 2.0 * self_.double()
    assert_gemm_close(out, exact.to(dt), dt)
    assert_gemm_close(out, torch.addmm(self_, a, w.t(), beta=2.0, alpha=0.5), dt)


def test_gemm_nt_batched_strided_and_shared_operand():
    torch.manual_seed(2)
    B, M, N, K = 3, 96, 160, 128
    dt = torch.float16
    a = torch.randn(B, M, K + 8).to(dt)
    b = (0.1 * torch.randn(B, N, K)).to(dt)
    ad, bd = a.cuda()[:, :, :K], b.cuda()                           # rows 16-byte aligned, not dense
    a = a[:, :, :K]
    assert not ad.is_contiguous()
    out = capi.gemm_nt(ad, bd)
    for i in range(B):
        assert_gemm_close(out[i], O.matmul_nt(a[i].contiguous(), b[i]), dt)
    out = capi.gemm_nt(ad, bd[0])                                   # one weight matrix for the whole batch
    for i in range(B):
        assert_gemm_close(out[i], O.matmul_nt(a[i].contiguous(), b[0]), dt)


def test_gemm_nt_errors_and_empty():
    z = lambda *s: torch.zeros(*s, dtype=torch.bfloat16, device="cuda")
    with pytest.raises(capi.ParasError, match="leading dimension"):
        a = z(8, 64)
        capi.check(capi.lib().paras_gemm_nt(a.data_ptr(), a.data_ptr(), None, a.data_ptr(), 8, 8, 64, 32, 64, 8, 0, 1, 0, 0, 0, 0,
                                            1.0, 0.0, capi.BF16, capi._stream()))
    assert capi.gemm_nt(z(0, 64), z(8, 64)).shape == (0, 8)
    assert torch.equal(capi.gemm_nt(z(4, 0), z(8, 0)), z(4, 8))          # empty contraction: zeros


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64, torch.bfloat16, torch.float16])
def test_gemm_nt_general_kernel(dtype):
    """What the MFMA kernels do not take -- fp32 / fp64 tensors, contraction sizes that are not a
    multiple of 64, rows that are not 16-byte aligned -- runs on the general device kernel."""
    torch.manual_seed(13)
    for (M, N, K) in [(1, 1, 1), (17, 9, 30), (70, 130, 65), (64, 64, 16), (129, 65, 200)]:
        a, b = torch.randn(M, K).to(dtype), (torch.randn(N, K) / math.sqrt(K)).to(dtype)
        got = capi.gemm_nt(a.cuda(), b.cuda())
        if dtype in (torch.bfloat16, torch.float16):
            assert_gemm_close(got, O.matmul_nt(a, b), dtype)
        else:
            want = a.double() @ b.double().t()
            tol = 1e-5 if dtype == torch.float32 else 1e-13
            assert torch.allclose(got.double().cpu(), want, rtol=tol, atol=tol)
        bias = torch.randn(N).to(dtype)
        got = capi.gemm_nt(a.cuda(), b.cuda(), bias.cuda(), alpha=0.5, beta=2.0)
        want = 0.5 * (a.double() @ b.double().t()) + 2.0 * bias.double()
        tol = {torch.float32: 1e-5, torch.float64: 1e-13}.get(dtype, 2e-2)
        assert torch.allclose(got.double().cpu(), want, rtol=tol, atol=tol)
    if dtype == torch.bfloat16:                                              # a multiple of 64, but rows 2 bytes off alignment
        buf = torch.randn(40 * 128 + 1).to(dtype).cuda()
        a = buf[1:].view(40, 128)
        b = (0.1 * torch.randn(24, 128)).to(dtype).cuda()
        assert_gemm_close(capi.gemm_nt(a, b), O.matmul_nt(a.cpu(), b.cpu()), dtype)


def test_gemm_nt_fp32_on_the_matrix_cores():
    """fp32 products with enough outputs for 128 x 128 tiles run on v_mfma_f32_32x32x2_f32 (full
    fp32 multiplies): ragged M, N, K, rows that are not 16-byte aligned (scalar staging), a batch
    with a shared weight, alpha / beta with a bias and with a full addend; 1e-5 against fp64."""
    torch.manual_seed(21)
    def close(got, want):
        scale = want.abs().max().item()
        assert (got.double().cpu() - want).abs().max().item() <= 1e-5 * scale
    for (M, N, K) in [(1024, 1024, 512), (1000, 777, 333), (130, 4100, 17), (4096, 640, 2048)]:
        a, b = torch.randn(M, K), torch.randn(N, K) / math.sqrt(K)
        close(capi.gemm_nt(a.cuda(), b.cuda()), a.double() @ b.double().t())
    a, b = torch.randn(700, 259), torch.randn(900, 259)                       # K odd: no 16-byte loads
    bias, full = torch.randn(900), torch.randn(700, 900)
    close(capi.gemm_nt(a.cuda(), b.cuda(), bias.cuda(), alpha=0.5, beta=2.0), 0.5 * (a.double() @ b.double().t()) + 2.0 * bias.double())
    close(capi.gemm_nt(a.cuda(), b.cuda(), full.cuda(), alpha=-1.25, beta=0.75), -1.25 * (a.double() @ b.double().t()) + 0.75 * full.double())
    buf = torch.randn(512 * 260 + 1).cuda()                                    # rows 4 bytes off 16-byte alignment
    av = buf[1:].view(512, 260)[:, :256]
    bw = torch.randn(640, 256)
    close(capi.gemm_nt(av, bw.cuda()), av.cpu().double() @ bw.double().t())
    a3, b2 = torch.randn(6, 300, 128), torch.randn(512, 128)                   # batched activations, one weight
    close(capi.gemm_nt(a3.cuda(), b2.cuda()), a3.double() @ b2.double().t())
    a3, b3 = torch.randn(5, 256, 96), torch.randn(5, 384, 96)                  # a weight per batch entry
    close(capi.gemm_nt(a3.cuda(), b3.cuda()), a3.double() @ b3.double().transpose(1, 2))


def test_gemm_nt_linearity_at_projection_size():
    """Size-independent property at a transformer projection shape: (2 a) W^T == 2 (a W^T) bit for
    bit, since scaling by a power of two commutes with every rounding; plus sampled rows vs the oracle."""
    torch.manual_seed(3)
    M, N, K = 4096, 4096, 4096
    dt = torch.bfloat16
    a1 = torch.randn(M, K, device="cuda").to(dt)
    a2 = a1 * 2                                                     # exact: a power of two
    w = (0.02 * torch.randn(N, K, device="cuda")).to(dt)
    y1, y2 = capi.gemm_nt(a1, w), capi.gemm_nt(a2, w)
    assert torch.equal(y2, y1 * 2)                                  # scaling by 2 commutes with every rounding
    rows = torch.randint(0, M, (8,))
    ref = O.matmul_nt(a1[rows].cpu(), w.cpu())
    assert_gemm_close(y1[rows], ref, dt)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_gemm_nt_many_tiles_with_ragged_edges(dtype):
    """Thousands of tiles, with M and N that are not multiples of the tile; sampled rows (first,
    last, tile boundaries) against the oracle."""
    torch.manual_seed(9)
    M, N, K = 8269, 4129, 192
    a = torch.randn(M, K, device="cuda").to(dtype)
    b = (0.1 * torch.randn(N, K, device="cuda")).to(dtype)
    bias = torch.randn(N, device="cuda").to(dtype)
    out = capi.gemm_nt(a, b)
    rows = torch.tensor([0, 1, 127, 128, 255, 256, 257, 4095, 4096, 8191, 8192, M - 2, M - 1])
    ref = O.matmul_nt(a[rows].cpu(), b.cpu())
    assert_gemm_close(out[rows], ref, dtype)
    out2 = capi.gemm_nt(a, b, bias, alpha=1.0, beta=1.0)
    assert_gemm_close(out2[rows], torch.nn.functional.linear(a[rows].cpu(), b.cpu(), bias.cpu()), dtype)
    # whole-matrix property: doubling A doubles every output bit for bit (away from f16's subnormals,
    # where 2 * round(v) and round(2 v) keep different numbers of bits)
    big = out.float().abs() > 1e-3
    assert torch.equal(capi.gemm_nt(a * 2, b)[big], (out * 2)[big])


_EIGHT_WAVES_CHILD = r"""
import hashlib, sys, torch
sys.path.insert(0, sys.argv[1])
import capi
torch.manual_seed(33)
a = torch.randn(4, 2100, 128).bfloat16().cuda()
b = (0.1 * torch.randn(4, 2100, 128)).bfloat16().cuda()
out = capi.gemm_nt(a, b)
T, E, k, H, I = 4096, 2, 2, 1024, 512
logits, x = torch.randn(T, E).bfloat16().cuda(), torch.randn(T, H).bfloat16().cuda()
wg, wu = (0.03 * torch.randn(E, I, H)).bfloat16().cuda(), (0.03 * torch.randn(E, I, H)).bfloat16().cuda()
wd = (0.03 * torch.randn(E, H, I)).bfloat16().cuda()
topi, topw, order, inv, counts, offsets = capi.moe_route(logits, k)
y = capi.moe_ffn(x, wg, wu, wd, topw, order, inv, offsets, k)
for t in (out, y):
    print(hashlib.sha256(t.cpu().view(torch.int16).numpy().tobytes()).hexdigest())
"""


def test_256_row_tiles_on_eight_waves_give_the_same_bits():
    """PARAS_GEMM_EIGHT_WAVES=1 sends the tiles of the
    expert FFN to the eight-wave kernel on 32 x 32 x 16 MFMAs.  It adds the same products in the same order as the
    four-wave kernel on 16 x 16 x 32: identical outputs, compared by digest.  (The dense product, which has no such
    form, is along as the control: the switch leaves it alone.)"""
    import os, subprocess, sys
    here = os.path.dirname(os.path.abspath(__file__))
    def run(extra):
        env = {k: v for k, v in os.environ.items() if k != "PARAS_GEMM_EIGHT_WAVES"}
        env.update(extra)
        r = subprocess.run([sys.executable, "-c", _EIGHT_WAVES_CHILD, here], env=env, capture_output=True, text=True, timeout=300)
        assert r.returncode == 0, r.stderr[-2000:]
        return r.stdout.split()
    four, eight = run({}), run({"PARAS_GEMM_EIGHT_WAVES": "1"})
    assert len(four) == 2 and four == eight


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("shape", [(4352, 4096, 256), (700, 512, 128), (64, 1024, 512), (8, 512, 256)])
def test_gemm_nt_nan_and_infinity_go_where_ieee_sends_them(shape, dtype):
    """A NaN in one row of A, an infinity in one row of B, on every tile form (256-row, 128-row, the
    split contraction of few rows, the weight-streaming kernel): NaNs exactly where fp32 arithmetic
    puts them (that row, that column; in bfloat16 with the host's NaN encoding), infinities with their signs,
    everything else as without them."""
    M, N, K = shape
    torch.manual_seed(M)
    a = torch.randn(M, K).to(dtype)
    b = (0.1 * torch.randn(N, K)).to(dtype)
    clean = capi.gemm_nt(a.cuda(), b.cuda()).cpu()
    a[M // 3, 5] = float("nan")
    b[N // 2, 7] = float("inf")
    got = capi.gemm_nt(a.cuda(), b.cuda()).cpu()
    ref = (a.float() @ b.float().T).to(dtype)
    assert torch.equal(got.isnan(), ref.isnan()) and torch.equal(got.isinf(), ref.isinf())
    assert bool(got[M // 3].isnan().all()) and bool(got[:, N // 2].isinf().sum() >= M - 2)
    assert torch.equal(got[got.isinf()], ref[ref.isinf()])
    if dtype == torch.bfloat16:
        # one NaN encoding in bfloat16, the oracle's; float16 keeps the sign of the fp32 NaN, and which sign
        # a NaN sum gets is the adder's choice (the matrix cores and a CPU differ), so only bf16 is held to bits
        want_row = O.matmul_nt(a[M // 3: M // 3 + 1], b)
        assert torch.equal(got[M // 3: M // 3 + 1].view(torch.int16), want_row.view(torch.int16))
    keep = torch.ones(M, N, dtype=torch.bool)
    keep[M // 3] = False
    keep[:, N // 2] = False
    assert torch.equal(got[keep], clean[keep])


def test_gemm_nt_256_row_tiles_agree_with_128_row_tiles():
    """A batch of four problems is big enough for the 256-row tiles, each problem alone is not:
    both forms add the same products in the same order, so they agree bit for bit (ragged M and
    N, strided batch)."""
    torch.manual_seed(21)
    Bt, M, N, K = 4, 2100, 2100, 128      # 81 tiles of 256 x 256 each (-> 128 x 128 tiles), 324 together (-> 256-row tiles)
    a = torch.randn(Bt, M, K, device="cuda").bfloat16()
    b = (0.1 * torch.randn(Bt, N, K, device="cuda")).bfloat16()
    whole = capi.gemm_nt(a, b)
    assert whole.shape == (Bt, M, N)
    for i in range(Bt):
        assert torch.equal(whole[i], capi.gemm_nt(a[i], b[i])), f"batch {i}"
    ref = O.matmul_nt(a[3, -3:].cpu(), b[3].cpu())
    assert_gemm_close(whole[3, -3:], ref, torch.bfloat16)


@pytest.mark.parametrize("shape", [(2, 1100, 2100, 64), (1, 1024, 2048, 128), (3, 2300, 4200, 64), (1, 16384, 4096, 64)])
def test_gemm_nt_tiles_dealt_to_the_dies_in_blocks_cover_every_element(shape):
    """From 4 x 8 tiles of 256 x 256 on, the workgroups take their tiles in blocks of 4 x 8 per die,
    on a grid padded to whole blocks and to eight blocks at a time: every element of every batch
    entry has to come out, none twice from a wrong tile.  Whole matrix against the oracle (which
    fits here: one k-tile or two)."""
    Bt, M, N, K = shape
    torch.manual_seed(33)
    a = torch.randn(Bt, M, K, device="cuda").bfloat16()
    b = (0.1 * torch.randn(Bt, N, K, device="cuda")).bfloat16()
    out = capi.gemm_nt(a, b)
    assert out.shape == (Bt, M, N)
    for i in range(Bt):
        assert_gemm_close(out[i], O.matmul_nt(a[i].cpu(), b[i].cpu()), torch.bfloat16)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("shape", [(1, 4096, 4096), (16, 100, 64), (17, 1027, 320), (64, 4096, 1024), (100, 515, 192),
                                   (128, 2050, 4096)])
def test_gemm_nt_few_rows(shape, dtype):
    """M <= 128 (decode-time projections) runs on the weight-streaming kernel: plain product,
    bias + scaled addend, N with and without 8-byte aligned output rows."""
    M, N, K = shape
    torch.manual_seed(M + N + K)
    a = torch.randn(M, K).to(dtype)
    b = (torch.randn(N, K) / math.sqrt(K)).to(dtype)
    assert_gemm_close(capi.gemm_nt(a.cuda(), b.cuda()), O.matmul_nt(a, b), dtype)
    bias = torch.randn(N).to(dtype)
    got = capi.gemm_nt(a.cuda(), b.cuda(), bias.cuda(), alpha=1.0, beta=1.0)
    assert_gemm_close(got, torch.nn.functional.linear(a, b, bias), dtype)
    addm = torch.randn(M, N).to(dtype)
    got = capi.gemm_nt(a.cuda(), b.cuda(), addm.cuda(), alpha=0.5, beta=2.0)
    want = torch.addmm(addm.float(), a.float(), b.float().t(), beta=2.0, alpha=0.5)
    err = (got.float().cpu() - want).abs()
    assert bool((err <= 2 * ulp16(want, dtype) + 1e-6).all())


def test_gemm_nt_few_rows_batched():
    torch.manual_seed(8)
    a = torch.randn(6, 40, 256, device="cuda").bfloat16()
    b = (0.1 * torch.randn(6, 72, 256, device="cuda")).bfloat16()
    out = capi.gemm_nt(a, b)
    for i in range(6):
        assert_gemm_close(out[i], O.matmul_nt(a[i].cpu(), b[i].cpu()), torch.bfloat16)
    shared = capi.gemm_nt(a, b[0])                      # one weight matrix for the whole batch
    for i in range(6):
        assert torch.equal(shared[i], capi.gemm_nt(a[i], b[0]))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("shape", [(32, 4096, 4096), (64, 4096, 1024), (64, 1027, 4096), (100, 1536, 2048), (128, 2050, 4096),
                                   (33, 640, 1088), (48, 4096, 2048), (49, 384, 4096), (128, 4096, 14336), (77, 130, 704)])
def test_gemm_nt_few_rows_with_workspace(shape, dtype):
    """32 to 128 rows with the workspace the library asks for: the contraction is split over
    workgroups (of the few-row kernel up to 48 rows, of the 128 x 128 tile kernel above) and the
    partial sums are added in a fixed order -- same bar as every other GEMM kernel, same result on
    every call, with bias / scaled addend and ragged N and K splits."""
    M, N, K = shape
    torch.manual_seed(M + N + K)
    a = torch.randn(M, K).to(dtype)
    b = (torch.randn(N, K) / math.sqrt(K)).to(dtype)
    assert capi.lib().paras_gemm_nt_workspace(M, N, K, 1, capi.DT[dtype]) > 0
    got = capi.gemm_nt(a.cuda(), b.cuda(), workspace=True)
    assert_gemm_close(got, O.matmul_nt(a, b), dtype)
    assert torch.equal(got, capi.gemm_nt(a.cuda(), b.cuda(), workspace=True))          # deterministic
    bias = torch.randn(N).to(dtype)
    got = capi.gemm_nt(a.cuda(), b.cuda(), bias.cuda(), alpha=1.0, beta=1.0, workspace=True)
    assert_gemm_close(got, torch.nn.functional.linear(a, b, bias), dtype)
    addm = torch.randn(M, N).to(dtype)
    got = capi.gemm_nt(a.cuda(), b.cuda(), addm.cuda(), alpha=0.5, beta=2.0, workspace=True)
    want = torch.addmm(addm.float(), a.float(), b.float().t(), beta=2.0, alpha=0.5)
    assert bool(((got.float().cpu() - want).abs() <= 2 * ulp16(want, dtype) + 1e-6).all())


def test_gemm_nt_few_rows_and_many_columns_take_the_tile_kernel():
    """33 to 128 rows against a vocabulary-sized weight matrix: enough 128 x 128 tiles to fill the
    chip, so no workspace is asked for and the result is the tile kernel's."""
    torch.manual_seed(44)
    M, N, K = 100, 24576 + 70, 256
    a = torch.randn(M, K).bfloat16()
    b = (torch.randn(N, K) / 16).bfloat16()
    assert capi.lib().paras_gemm_nt_workspace(M, N, K, 1, capi.BF16) == 0
    got = capi.gemm_nt(a.cuda(), b.cuda(), workspace=True)
    assert_gemm_close(got, O.matmul_nt(a, b), torch.bfloat16)
    bias = torch.randn(N).bfloat16()
    got = capi.gemm_nt(a.cuda(), b.cuda(), bias.cuda(), alpha=1.0, beta=1.0)
    assert_gemm_close(got, torch.nn.functional.linear(a, b, bias), torch.bfloat16)
    # batched: 3 x 64 tiles
    a3 = torch.randn(3, 60, 256, device="cuda").bfloat16()
    b3 = (torch.randn(3, 8192, 256, device="cuda") / 16).bfloat16()
    out = capi.gemm_nt(a3, b3, workspace=True)
    for i in range(3):
        assert_gemm_close(out[i], O.matmul_nt(a3[i].cpu(), b3[i].cpu()), torch.bfloat16)


def test_gemm_nt_workspace_batched_and_shapes_that_need_none():
    torch.manual_seed(6)
    a = torch.randn(3, 48, 1024, device="cuda").bfloat16()
    b = (0.05 * torch.randn(3, 768, 1024, device="cuda")).bfloat16()
    out = capi.gemm_nt(a, b, workspace=True)
    for i in range(3):
        assert_gemm_close(out[i], O.matmul_nt(a[i].cpu(), b[i].cpu()), torch.bfloat16)
    L = capi.lib()
    assert L.paras_gemm_nt_workspace(8, 4096, 4096, 1, capi.BF16) == 0        # up to 16 rows: nothing to share
    assert L.paras_gemm_nt_workspace(4096, 4096, 4096, 1, capi.BF16) == 0     # tile kernels
    assert L.paras_gemm_nt_workspace(64, 4096, 4096, 1, capi.F32) == 0        # general kernel
    x = torch.randn(8, 256, device="cuda").bfloat16()
    w = torch.randn(64, 256, device="cuda").bfloat16()
    assert torch.equal(capi.gemm_nt(x, w, workspace=True), capi.gemm_nt(x, w))


def test_mfma_rate_probe_reports_a_plausible_rate():
    """The measurement aid bench.py prints beside the attention figure: a register-only MFMA loop
    cannot beat the published peak and, on a healthy MI355X, does not fall below a fifth of it."""
    import ctypes as C
    rate = C.c_double(0.0)
    capi.check(capi.lib().paras_mfma_rate_probe(1, 0, C.byref(rate)))
    assert 500.0 < rate.value < 2600.0
    assert capi.lib().paras_mfma_rate_probe(3, 0, C.byref(rate)) != 0          # only one or two wavefronts per SIMD
    assert b"wavefronts per SIMD" in capi.lib().paras_last_error()


def test_l2_stream_probe_reports_plausible_rates():
    """The streaming probe: regions that stay in L2 come in faster than regions that do not, and
    both at a rate a CU can plausibly reach (a GEMM tile of 256 x 256 needs about 40 B/ns per CU)."""
    import ctypes as C
    rate = C.c_double(0.0)
    got = {}
    for to_lds, kib in ((1, 64), (1, 512), (0, 64)):
        capi.check(capi.lib().paras_l2_stream_probe(to_lds, kib, C.byref(rate)))
        got[(to_lds, kib)] = rate.value
    assert 40.0 < got[(1, 64)] < 400.0, got            # measured 116 - 128 B/ns per CU
    assert 5.0 < got[(1, 512)] < got[(1, 64)], got      # measured 21 - 26 B/ns per CU from the last-level cache
    assert 10.0 < got[(0, 64)] < 400.0, got             # measured 33 B/ns per CU with eight loads in flight per wavefront
    assert capi.lib().paras_l2_stream_probe(1, 48, C.byref(rate)) != 0        # not a power of two


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("shape", [(16384, 8, 4096), (5000, 1, 256), (3001, 17, 512), (2048, 32, 1024), (3001, 33, 512), (2048, 128, 1024), (700, 100, 192), (9000, 64, 4096)])
def test_gemm_nt_few_columns_and_many_rows(shape, dtype):
    """A router's logits and the like (tokens x experts): the few-row kernels with the operands in each
    other's place and the results stored transposed; plain, with a bias over the columns, with a full
    addend and a scale, and batched."""
    M, N, K = shape
    torch.manual_seed(M + N)
    a = torch.randn(M, K).to(dtype)
    b = (0.1 * torch.randn(N, K)).to(dtype)
    rows = torch.tensor([0, 1, 15, 16, 127, 128, M // 2, M - 2, M - 1])
    out = capi.gemm_nt(a.cuda(), b.cuda())
    assert out.shape == (M, N)
    assert_gemm_close(out[rows], O.matmul_nt(a[rows], b), dtype)
    # every element against an fp32 product on the device (nothing left unwritten, nothing misplaced;
    # that product sums in another order, so small results get an absolute allowance)
    ref = (a.cuda().float() @ b.cuda().float().t())
    assert bool(((out.float() - ref).abs() <= 2.0 ** -7 * ref.abs().clamp_min(0.05)).all())
    bias = torch.randn(N).to(dtype)
    out2 = capi.gemm_nt(a.cuda(), b.cuda(), bias.cuda())
    assert_gemm_close(out2[rows], torch.nn.functional.linear(a[rows], b, bias), dtype)
    full = torch.randn(M, N).to(dtype)
    out3 = capi.gemm_nt(a.cuda(), b.cuda(), full.cuda(), alpha=0.5, beta=2.0)
    want3 = (0.5 * (a[rows].double() @ b.double().t()) + 2.0 * full[rows].double())
    assert_gemm_close(out3[rows], want3, dtype)
    ab = torch.stack([a[:600], a[600:1200]]) if M >= 1200 else None
    if ab is not None:
        bb = torch.stack([b, b.flip(0)])
        ob = capi.gemm_nt(ab.cuda(), bb.cuda())
        for i in range(2):
            assert_gemm_close(ob[i, -3:], O.matmul_nt(ab[i, -3:], bb[i]), dtype)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("shape", [(1, 64, 8), (33, 72, 64), (64, 136, 200), (200, 264, 72), (130, 1000, 1000), (520, 136, 4096), (3000, 520, 512),
                                   (1000, 3000, 1032), (2048, 4096, 128)])
def test_gemm_operands_either_way_round(shape, dtype):
    """paras_gemm: both operands along the contraction, B along its rows (dy W), both along their rows
    (dy^T x) -- tiles from 32 x 128 to 256 x 256, cut short in every direction, an odd and an even number of
    contraction tiles, the contraction whole and in parts (in a fixed order: the same bits on every call)."""
    M, N, K = shape
    torch.manual_seed(M + N + K)
    a = torch.randn(M, K).to(dtype)
    b = (torch.randn(N, K) / math.sqrt(K)).to(dtype)
    bias = torch.randn(N).to(dtype)
    want = a.double() @ b.double().T
    tol = {torch.bfloat16: 4e-3, torch.float16: 6e-4, torch.float32: 3e-6}[dtype]     # (fp32: a sequential sum of 4096 products)
    rows16 = dtype != torch.float32
    ac, bc = a.cuda(), b.cuda()
    ar, br = a.T.contiguous().cuda().T, b.T.contiguous().cuda().T
    if rows16 and N % 8:
        pytest.skip("rows-contiguous 16-bit operands have leading dimensions that are multiples of 8")
    for x, y in ((ac, bc), (ac, br), (ar, br)):
        if rows16 and x is ar and M % 8:
            continue
        for ws in (False, True):
            got = capi.gemm(x, y, workspace=ws)
            assert ((got.cpu().double() - want).norm() / want.norm()).item() < tol
            assert torch.equal(got, capi.gemm(x, y, workspace=ws))
        got = capi.gemm(x, y, bias.cuda(), alpha=0.5, beta=2.0)
        ref = 0.5 * want + 2.0 * bias.double()
        assert ((got.cpu().double() - ref).norm() / ref.norm()).item() < tol


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32, torch.float64])
@pytest.mark.parametrize("shape", [(1, 1), (7, 33), (9, 64), (3000, 4096), (65, 8200), (100000, 8)])
def test_column_sum(shape, dtype):
    x = torch.randn(*shape).to(dtype)
    want = x.double().sum(0)
    got = capi.column_sum(x.cuda()).cpu().double()
    bound = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11, torch.float32: 2.0 ** -23, torch.float64: 1e-14}[dtype]
    assert bool(((got - want).abs() <= bound * want.abs() + 1e-5 * math.sqrt(shape[0]) * (1 if dtype.itemsize == 2 else 1e-2)).all())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("M", [1, 8, 9, 16, 17, 32])
def test_few_rows_streamed_through_lds(M, dtype):
    """Products of up to 32 rows: one to four requests of activations per piece; a ragged last block of weight rows; fewer
    pieces of the contraction than waves, one more than a multiple of them, several trips; workgroups with more than one
    block (N = 17000); padded strides; an infinity that only some results may see."""
    for (N, K) in [(40, 64), (23, 576), (264, 1024), (4096, 2624), (17000, 128)]:
        torch.manual_seed(M + N + K)
        a, b = torch.randn(M, K + 8).to(dtype), (torch.randn(N, K + 16) / math.sqrt(K)).to(dtype)
        bias = torch.randn(N).to(dtype)
        a[M // 2, 3] = float("inf")
        b[N // 2, 3] = 0.25
        got = capi.gemm_nt(a.cuda()[:, :K], b.cuda()[:, :K], bias.cuda()).cpu()
        want = a[:, :K].double() @ b[:, :K].double().t() + bias.double()
        special = ~torch.isfinite(want)
        assert torch.equal(got.double()[special & ~want.isnan()], want[special & ~want.isnan()])
        assert bool((got.isnan() == want.isnan()).all())
        keep = [r for r in range(M) if r != M // 2]
        if keep:            # fp32 sums of K products of size 1 / sqrt(K), then one rounding to the type: one ulp, or 1e-6 sqrt(K) where they cancel
            err = (got[keep].double() - want[keep]).abs()
            assert bool((err <= ulp16(want[keep], dtype) * 1.001 + 1e-6 * math.sqrt(K)).all())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("M", [1, 8, 16, 32])
def test_few_rows_dealt_out_evenly(M, dtype):
    """Shares of weight rows per workgroup from 8 to more than 32 rows that are no whole blocks of 16 or 32: every element,
    and nothing beside the result (rows of the output wider than it)."""
    for (N, K) in [(2052, 192), (3000, 64), (4100, 576), (7172, 128), (8192, 64), (8196, 64), (14333, 128), (21000, 64)]:
        torch.manual_seed(M + N)
        a, b = torch.randn(M, K).to(dtype).cuda(), (torch.randn(N, K) / math.sqrt(K)).to(dtype).cuda()
        out = torch.full((M + 1, N + 8), 7.0, dtype=dtype, device="cuda")
        capi.check(capi.lib().paras_gemm_nt(a.data_ptr(), b.data_ptr(), None, out.data_ptr(), M, N, K, K, K, N + 8, 0, 1, 0, 0, 0, 0, 1.0, 0.0,
                                            capi.DT[dtype], capi._stream()))
        want = a.double() @ b.double().t()
        assert bool(((out[:M, :N].double() - want).abs() <= ulp16(want, dtype) * 1.001 + 1e-6 * math.sqrt(K)).all())
        assert bool((out[M:] == 7.0).all()) and bool((out[:, N:] == 7.0).all())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_few_columns_streamed_through_lds(dtype):
    """A router's logits: many rows and few columns, the operands in each other's place."""
    for (M, N, K) in [(129, 1, 64), (300, 8, 704), (20000, 9, 128), (515, 32, 2048)]:
        torch.manual_seed(M)
        a, b = torch.randn(M, K).to(dtype), (torch.randn(N, K) / math.sqrt(K)).to(dtype)
        assert_gemm_close(capi.gemm_nt(a.cuda(), b.cuda()), (a.double() @ b.double().t()).to(dtype), dtype)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("shape", [(81, 64, 40), (105, 80, 968), (63, 968, 1768), (232, 4136, 960), (72, 752, 2880), (1056, 1016, 232), (40, 2808, 2656),
                                   (1224, 2560, 136), (1816, 2264, 552), (1816, 2264, 768), (2792, 2216, 584), (57, 112, 2632),
                                   (1500, 14336, 520), (3900, 3576, 1032), (1336, 8056, 584)])
def test_gemm_tiles_with_several_stages(shape, dtype):
    """Tiles whose operands are requested two or three tiles ahead: one tile of contraction to forty, numbers of them that do
    and do not come in whole turns of the stages, rows and columns cut short, whole and in parts, all three layouts.  Every
    element against fp64 (bar: the rounding of the result plus 4 sqrt(K) fp32 roundings of a sum of K terms near 1 / sqrt(K))."""
    M, N, K = shape
    torch.manual_seed(M + 3 * N + K)
    a = torch.randn(M, K).to(dtype).cuda()
    b = (torch.randn(N, K) / math.sqrt(K)).to(dtype).cuda()
    want = a.double() @ b.double().T
    half_ulp = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}[dtype]      # of a value just above a power of two: 8 and 11 significant bits
    bar = half_ulp * 1.01 * want.abs() + 4 * math.sqrt(K) * 2.0 ** -24 + 2.0 ** -24
    ar, br = a.T.contiguous().T, b.T.contiguous().T
    for x, y in ((a, b), (a, br), (ar, br)):
        if x is ar and M % 8:
            continue
        for ws in (False, True):
            got = capi.gemm(x, y, workspace=ws)
            assert bool(((got.double() - want).abs() <= bar).all())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("shape", [(8, 512, 1024), (33, 512, 512), (64, 4096, 512), (65, 512, 512), (64, 4104, 512), (64, 512, 576), (128, 4096, 64), (128, 4104, 64), (65, 256, 128), (128, 2048, 2048), (700, 24, 512),
                                   (96, 1000, 72), (300, 136, 14336)])
def test_scratch_is_asked_for_once_and_the_route_is_the_planned_one(shape, dtype):
    """paras_gemm_scratch: the size that paras_gemm_workspace answers, once, or no question where that is 0, and the bits of
    paras_gemm -- with that workspace, and without any where none is wanted: the route is one choice.  Either side of the rules
    for 33 to 64 rows (and for 65 to 128 with a contraction of 64), few columns, other contractions, parts.  No memory: an error before
    anything is launched."""
    M, N, K = shape
    torch.manual_seed(M + N + K)
    a, b = torch.randn(M, K).to(dtype).cuda(), (torch.randn(N, K) / math.sqrt(K)).to(dtype).cuda()
    want = a.double() @ b.double().T
    asked = []
    c, n, rc = capi.gemm_scratch(a, b, lambda size: asked.append(size) or torch.empty(size, dtype=torch.uint8, device="cuda"))
    assert rc == 0 and asked == ([n] if n else [])
    assert torch.equal(c, capi.gemm(a, b))
    if n == 0:
        assert torch.equal(c, capi.gemm(a, b, workspace=False))
    assert ((c.double() - want).norm() / want.norm()).item() < {torch.bfloat16: 4e-3, torch.float16: 6e-4, torch.float32: 3e-6}[dtype]
    if n:
        c, _, rc = capi.gemm_scratch(a, b, lambda size: None)
        assert rc == -1 and bool((c == 7).all())
    assert n > 0 or shape != (300, 136, 14336)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_addend_rows_far_apart_in_a_product_in_parts(dtype):
    """The kernel that adds the parts reads the addend: 1100 rows of 2^22 elements, the last of them beyond 2^32 elements.  Bar as in
    test_gemm_tiles_with_several_stages, with a rounding of the addend's size more."""
    M, N, K, ld = 1100, 64, 8192, 1 << 22
    g = torch.Generator(device="cuda").manual_seed(3)
    a, b = torch.randn(M, K, generator=g, device="cuda").to(dtype), (torch.randn(N, K, generator=g, device="cuda") / math.sqrt(K)).to(dtype)
    add = torch.empty(M, ld, device="cuda", dtype=dtype)[:, :N]
    add.copy_(torch.randn(M, N, generator=g, device="cuda"))
    problem = capi.GemmArgs(a.data_ptr(), b.data_ptr(), add.data_ptr(), a.data_ptr(), M, N, K, K, K, N, ld, 1, 0, 0, 0, 0, 1.0, 1.0, capi.DT[dtype], 0, 0)
    assert capi.lib().paras_gemm_workspace(C.byref(problem)) > 0
    want = a.double() @ b.double().T + add.double()
    half_ulp = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}[dtype]
    assert bool(((capi.gemm(a, b, add).double() - want).abs() <= half_ulp * 1.01 * want.abs() + (4 * math.sqrt(K) + 8) * 2.0 ** -24).all())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("K,a_rows,b_rows", [(128, 0, 0), (72, 0, 0), (8200, 0, 0), (72, 0, 1), (72, 1, 1), (8192, 1, 1)])
def test_rows_of_result_and_addend_beyond_31_bits(K, a_rows, b_rows, dtype):
    """Two rows more than 2^31 elements apart, in the result and in the addend: the few-row kernel, tiles of each layout, whole and in parts.
    Bar as in test_addend_rows_far_apart_in_a_product_in_parts."""
    M, N, ldc, ld_add = 2, 100, (1 << 31) + 8, (1 << 31) + 20
    g = torch.Generator(device="cuda").manual_seed(K)
    a, b = torch.randn(K, 8, generator=g, device="cuda").to(dtype), (torch.randn(K, 104, generator=g, device="cuda") / math.sqrt(K)).to(dtype)
    x, y = a[:, :M].T, b[:, :N].T
    a, b = a if a_rows else x.contiguous(), b if b_rows else y.contiguous()
    c, add = torch.empty(M, ldc, device="cuda", dtype=dtype)[:, :N + 4], torch.empty(M, ld_add, device="cuda", dtype=dtype)[:, :N]
    c.fill_(7)
    add.copy_(torch.randn(M, N, generator=g, device="cuda"))
    problem = capi.GemmArgs(a.data_ptr(), b.data_ptr(), add.data_ptr(), c.data_ptr(), M, N, K, a.stride(0), b.stride(0), ldc, ld_add, 1, 0, 0, 0, 0, 1.0, 1.0,
                            capi.DT[dtype], a_rows, b_rows)
    n = capi.lib().paras_gemm_workspace(C.byref(problem))
    assert (n > 0) == (K > 8000)
    ws = torch.empty(max(n, 16), dtype=torch.uint8, device="cuda")
    capi.check(capi.lib().paras_gemm(C.byref(problem), ws.data_ptr(), n, torch.cuda.current_stream().cuda_stream))
    want = x.double().contiguous() @ y.double().T + add.double()
    half_ulp = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}[dtype]
    assert bool(((c[:, :N].double() - want).abs() <= half_ulp * 1.01 * want.abs() + (4 * math.sqrt(K) + 8) * 2.0 ** -24).all())
    assert bool((c[:, N:] == 7).all())


# problems of x W^T (0), dy W (1) and dy^T x (2) that reach each tile form, whole (test_gemm_forms_cpu.py); edges cut short in both directions (N % 4 == 0; K % 64 == 8, 16 ... or few steps)
TILES = [(0, (6437, 2104, 528)), (0, (2483, 4712, 576)), (0, (7082, 792, 536)), (0, (6536, 536, 528)), (0, (7119, 392, 64)), (0, (6977, 400, 136)), (0, (683, 5488, 64)),
         (0, (5661, 144, 200)), (0, (5700, 136, 64)), (0, (33, 72, 64)), (0, (36, 72, 208)), (0, (130, 5528, 64)), (0, (2709, 4520, 520)), (0, (2389, 4344, 520)), (0, (1189, 7000, 528)),
         (1, (1645, 7336, 520)), (1, (7683, 1160, 520)), (1, (1185, 5008, 528)), (1, (6805, 520, 528)), (1, (455, 6200, 64)), (1, (470, 6232, 136)), (1, (662, 5464, 64)),
         (1, (4246, 200, 200)), (1, (34, 72, 200)), (1, (134, 5528, 72)),
         (2, (1544, 7272, 528)), (2, (4840, 1840, 528)), (2, (7192, 816, 520)), (2, (520, 6552, 536)), (2, (7016, 408, 64)), (2, (400, 7128, 144)), (2, (5576, 136, 64)), (2, (136, 5616, 64)),
         (0, (2321, 5616, 528)), (0, (4932, 2040, 560)), (0, (1180, 6544, 528)), (0, (2732, 2224, 64)), (0, (2544, 1160, 408)), (0, (1049, 1800, 64)), (0, (584, 2312, 408)),
         (0, (737, 648, 64)), (0, (694, 712, 200)), (0, (1292, 1176, 64)), (0, (33, 72, 88)), (0, (3050, 3256, 64)), (0, (2514, 776, 392)), (0, (1155, 1672, 64)),
         (0, (1220, 792, 64)), (0, (3006, 1296, 64)), (0, (5569, 2056, 528)), (0, (7152, 1168, 536)), (0, (644, 5392, 2040)),
         (1, (5466, 2128, 536)), (1, (6224, 1360, 544)), (1, (3493, 2320, 520)), (1, (519, 7256, 920)), (1, (2543, 2440, 64)), (1, (2614, 1176, 392)), (1, (1409, 1360, 64)),
         (1, (408, 4176, 400)), (1, (618, 784, 64)), (1, (898, 520, 208)), (1, (1102, 904, 64)), (1, (34, 72, 64)), (1, (2886, 3472, 64)), (1, (836, 2328, 208)),
         (1, (1228, 1616, 64)), (1, (599, 1608, 200)), (1, (2705, 1456, 64)),
         (2, (8152, 1360, 520)), (2, (1624, 5400, 520)), (2, (3656, 2224, 520)), (2, (2056, 1928, 672)), (2, (2904, 2104, 64)), (2, (2104, 984, 392)), (2, (1040, 1808, 64)),
         (2, (784, 2384, 400)), (2, (792, 648, 64)), (2, (808, 600, 208)), (2, (904, 1104, 64)), (2, (40, 72, 64)), (2, (2552, 1584, 64))]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("layout,shape", TILES)
def test_every_tile_form_stores_its_rows(layout, shape, dtype):
    """Results in rows that lie apart, with the columns and rows beside them left alone: whole 16-byte pieces, and from an address and a stride
    that are not; plain, and with an addend whose rows are and are not 8-byte pieces.  Bar: half a 16-bit ulp of the result, plus fp32 sums."""
    M, N, K = shape
    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    x, y = torch.randn(M, K, generator=g, device="cuda").to(dtype), (torch.randn(N, K, generator=g, device="cuda") / math.sqrt(K)).to(dtype)
    a, b = x.T.contiguous() if layout == 2 else x, y.T.contiguous() if layout else y
    add = torch.randn(M, N + 5, generator=g, device="cuda").to(dtype)
    prod = x.double() @ y.double().T
    half_ulp = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}[dtype]
    for off, ldc, lda_, alpha in ((8, N + 16, None, 1.0), (1, N + 9, None, 1.0), (8, N + 16, N + 5, 0.5), (3, N + 8, 0, 1.0), (8, N + 16, N + 4, 1.0)):
        buf = torch.full(((M + 1) * ldc + 16,), 7.0, device="cuda", dtype=dtype)
        used = add.reshape(-1)[:M * (N + 4)].reshape(M, N + 4) if lda_ == N + 4 else add
        problem = capi.GemmArgs(a.data_ptr(), b.data_ptr(), used.data_ptr() if lda_ is not None else None, buf.data_ptr() + 2 * off, M, N, K, a.stride(0), b.stride(0), ldc,
                                lda_ or 0, 1, 0, 0, 0, 0, alpha, 2.0, capi.DT[dtype], int(layout == 2), int(layout > 0))
        capi.check(capi.lib().paras_gemm(C.byref(problem), None, 0, torch.cuda.current_stream().cuda_stream))
        want = alpha * prod
        if lda_ is not None:
            want = want + 2.0 * (used[:1, :N] if lda_ == 0 else used[:, :N]).double()
        rows = buf[off:off + M * ldc].reshape(M, ldc)
        assert bool(((rows[:, :N].double() - want).abs() <= half_ulp * 1.01 * want.abs() + (4 * math.sqrt(K) + 16) * 2.0 ** -24).all()), (off, lda_)
        assert bool((rows[:, N:] == 7).all()) and bool((buf[:off] == 7).all()) and bool((buf[off + M * ldc:] == 7).all()), (off, lda_)


# problems whose contraction comes in parts, the last of them short, for each tile form that is split (test_gemm_forms_cpu.py); edges cut short in both directions
PARTS = [(0, (193, 6504, 10216)), (0, (139, 4464, 14440)), (0, (2050, 136, 12320)), (0, (1889, 72, 14408)), (0, (193, 2992, 10280)), (0, (1367, 72, 13496)), (0, (36, 2712, 9336)),
         (0, (34, 1232, 9640)), (0, (33, 136, 5272)), (0, (33, 176, 6760)), (0, (620, 72, 7016)), (0, (34, 72, 1048)), (0, (66, 1832, 6568)), (0, (65, 1840, 13960)),
         (0, (65, 280, 6696)), (0, (199, 2952, 11560)), (0, (131, 4112, 10912)), (1, (195, 2768, 13408)), (1, (131, 5424, 7728)), (1, (2063, 136, 12296)), (1, (2712, 72, 9496)),
         (1, (1833, 72, 6176)), (1, (34, 2712, 5432)), (1, (584, 72, 5488)), (1, (34, 272, 5032)), (1, (33, 272, 6424)), (1, (292, 72, 4872)), (1, (33, 72, 776)), (1, (898, 72, 7824)),
         (1, (1370, 72, 10488)), (1, (68, 264, 6760)), (2, (208, 5384, 7867)), (2, (72, 5552, 14555)), (2, (2744, 136, 8331)), (2, (136, 1848, 6267)), (2, (80, 5656, 10259)),
         (2, (2704, 72, 4259)), (2, (40, 2864, 7179)), (2, (72, 392, 13360)), (2, (40, 184, 5251)), (2, (40, 216, 6819)), (2, (72, 584, 4664)), (2, (40, 72, 1032)),
         (2, (152, 1840, 8211))]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("layout,shape", PARTS)
def test_every_tile_form_in_parts(layout, shape, dtype):
    """fp32 parts in a workspace (not a byte past it), added and narrowed into rows that lie apart, plain and with an addend; two products in one call.
    Bar: half a 16-bit ulp of the result, plus fp32 sums."""
    M, N, K = shape
    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    half_ulp = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}[dtype]
    for batch, ldc, alpha, ld_add in ((1, N + 16, 1.0, None), (1, N + 9, 0.5, N + 5), (2, N + 8, 1.0, 0)):
        x = torch.randn(batch, M, K, generator=g, device="cuda").to(dtype)
        y = (torch.randn(batch, N, K, generator=g, device="cuda") / math.sqrt(K)).to(dtype)
        a, b = x.transpose(1, 2).contiguous() if layout == 2 else x, y.transpose(1, 2).contiguous() if layout else y
        add = torch.randn(M, N + 5, generator=g, device="cuda").to(dtype)
        buf = torch.full((batch, M, ldc), 7.0, device="cuda", dtype=dtype)
        problem = capi.GemmArgs(a.data_ptr(), b.data_ptr(), None if ld_add is None else add.data_ptr(), buf.data_ptr(), M, N, K, a.stride(1), b.stride(1), ldc, ld_add or 0, batch,
                                a.stride(0), b.stride(0), buf.stride(0), 0, alpha, 2.0, capi.DT[dtype], int(layout == 2), int(layout > 0))
        n = capi.lib().paras_gemm_workspace(C.byref(problem))
        if batch == 1:
            assert n >= 2 * 4 * M * N and n % (4 * M * N) == 0
        ws = torch.full((n // 4 + 64,), 7.0, device="cuda")
        capi.check(capi.lib().paras_gemm(C.byref(problem), ws.data_ptr(), n, torch.cuda.current_stream().cuda_stream))
        assert bool((ws[n // 4:] == 7).all())
        for i in range(batch):
            want = alpha * (x[i].double() @ y[i].double().T)
            if ld_add is not None:
                want = want + 2.0 * (add[:1, :N] if ld_add == 0 else add[:, :N]).double()
            assert bool(((buf[i, :, :N].double() - want).abs() <= half_ulp * 1.01 * want.abs() + (4 * math.sqrt(K) + 16) * 2.0 ** -24).all()), (batch, ld_add)
        assert bool((buf[:, :, N:] == 7).all())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("M,N,K", [(16, 328, 6144), (17, 328, 6080), (17, 328, 6144), (17, 64, 9600), (24, 8, 6208), (31, 1032, 14336), (32, 4096, 6144), (32, 4104, 6144)])
def test_few_rows_of_a_long_contraction(M, N, K, dtype):
    """On both sides of where tiles in parts take over from the kernel of a few rows.  Bar: half a 16-bit ulp of the result, plus fp32 sums."""
    x, y = torch.randn(M, K, device="cuda").to(dtype), (torch.randn(N, K, device="cuda") / math.sqrt(K)).to(dtype)
    add = torch.randn(N, device="cuda").to(dtype)
    half_ulp = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}[dtype]
    for bias in (None, add):
        want = x.double() @ y.double().T + (0 if bias is None else bias.double())
        got = capi.gemm(x, y, bias).double()
        assert bool(((got - want).abs() <= half_ulp * 1.01 * want.abs() + (4 * math.sqrt(K) + 16) * 2.0 ** -24).all())
