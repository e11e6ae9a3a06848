"""The bar of the grouped expert FFN, shared by its GPU tests and by the host-only test of the bar itself."""
import torch


def ulp16(ref, dtype):
    mant = 7 if dtype == torch.bfloat16 else 10
    return 2.0 ** (torch.floor(torch.log2(ref.double().abs().clamp_min(1e-30))) - mant)


def assert_ffn_close(out, ref, dtype):
    """Per element: max(2e-2, one 16-bit ulp of the reference value).  A GEMM
    whose fp32 summation order differs from ATen's flips the last bit of a few
    intermediate y values; weighted and re-rounded they reach the output as at
    most one ulp of the top binade of the outputs, for at most 1 element in
    1000.  Measured on the layer of 8192 tokens, 8 experts, H 4096, I 14336 over all 8192 x 4096 outputs
    (max |out| 11.25): worst 0.0625, 5472 elements (1.6e-4) beyond 2e-2, 3170
    (9.4e-5) beyond max(2e-2, 1 ulp), mean error 7.8e-5.  Two evaluations of
    the same composition on the host, with ATen's GEMM and with the oracle's
    own C GEMM (another fp32 summation order), differ by as much: 64 tokens
    of that shape, 262144 outputs, worst 0.0625, 8.0e-5 of them
    beyond 2e-2 (test_parity_bars_cpu.py holds them to this same bar); ATen
    on 8 threads against ATen on one already differs by 0.031 in one of
    them."""
    err = (out.double().cpu() - ref.double()).abs()
    tol = torch.maximum(torch.full_like(err, 2e-2), ulp16(ref, dtype) * 1.001)
    frac = float((err > tol).double().mean())
    top = float(ulp16(ref.double().abs().max() * 1.999, dtype))
    assert frac <= 1e-3, f"{frac:.2e} of elements beyond max(2e-2, 1 ulp); worst {err.max().item():.3e}"
    assert err.max().item() <= max(2e-2, top) * 1.001, f"worst {err.max().item():.3e} > one ulp of the top binade {top:.3e}"
    return err
