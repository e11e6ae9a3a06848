"""What paras_sdpa_workspace and paras_sdpa_kernel_name answer (host code only: nothing is launched)."""
import ctypes as C

import pytest
import torch

import capi


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("with_attn", [False, True])
@pytest.mark.parametrize("shape", [(1, 2, 2, 40, 60, 64, 64), (1, 4, 2, 512, 512, 64, 64), (2, 4, 4, 300, 700, 128, 72), (1, 4, 4, 512, 512, 66, 66), (1, 4, 4, 512, 512, 300, 300)])
def test_workspace_of_wide_types_does_not_depend_on_the_pointers(dtype, with_attn, shape):
    """A caller may ask for the workspace before it has bound its pointers: null, aligned and odd ones give the same
    kernel and the same size."""
    B, Hq, Hkv, Lq, Lk, D, Dv = shape
    q, k, v, out = torch.zeros(B, Hq, Lq, D, dtype=dtype), torch.zeros(B, Hkv, Lk, D, dtype=dtype), torch.zeros(B, Hkv, Lk, Dv, dtype=dtype), torch.zeros(B, Hq, Lq, Dv, dtype=dtype)
    a = capi.sdpa_args(q, k, v, out)
    seen = set()
    for base in (None, 4096, 4096 + 4 * (dtype == torch.float32) + 8 * (dtype == torch.float64)):
        a.q = a.k = a.v = a.out = base
        a.attn = (base or 4096) if with_attn else None
        seen.add((capi.lib().paras_sdpa_kernel_name(C.byref(a)), capi.lib().paras_sdpa_workspace(C.byref(a))))
    assert len(seen) == 1, seen
