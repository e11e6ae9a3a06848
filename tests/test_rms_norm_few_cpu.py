"""Which RMSNorm backward passes are one launch (rms_norm_few.h, plain C++: nothing is launched)."""
import ctypes as C
import subprocess

import pytest

import capi


@pytest.fixture(scope="module")
def takes(tmp_path_factory):
    where = tmp_path_factory.mktemp("few")
    (where / "few.cpp").write_text('''#include "kernels/rms_norm_few.h"
extern "C" int takes(int elem, long go, long x, long w, long rstd, long gx, long gw, long rows, long H) {
    auto p = [](long a) { return reinterpret_cast<const void*>(a); };
    bool whole = false;
    return paras::takes_few(elem, p(go), p(x), p(w), static_cast<const float*>(p(rstd)), p(gx), p(gw), rows, H, &whole) ? 1 + whole : 0;
}
''')
    subprocess.run(["g++", "-O2", "-std=c++17", "-shared", "-fPIC", f"-I{capi.PKG / 'csrc'}", str(where / "few.cpp"), "-o", str(where / "few.so")], check=True)
    f = C.CDLL(str(where / "few.so")).takes
    f.restype, f.argtypes = C.c_int, [C.c_int] + [C.c_long] * 8
    return f


NAMES = ("go", "x", "w", "rstd", "gx", "gw")


@pytest.mark.parametrize("elem", [2, 4, 8])
@pytest.mark.parametrize("rows,H", [(1, 264), (1, 4096), (40, 264), (300, 1000), (7, 33)])
def test_results_that_share_memory_with_anything_else_are_not_one_launch(takes, elem, rows, H):
    """Its workgroups write dx and dw while others of the same launch read g, x, w and rstd.  The kernels of the other way read w in a launch
    before the one that writes dw, so dw over w is theirs to take."""
    size = {"go": rows * H * elem, "x": rows * H * elem, "w": H * elem, "rstd": rows * 4, "gx": rows * H * elem, "gw": H * elem}

    def ask(at):
        return takes(elem, *(at[n] for n in NAMES), rows, H)
    far = {n: (i + 1) << 30 for i, n in enumerate(NAMES)}
    assert ask(far) == (2 if H * elem % 16 == 0 else 1)
    for out in ("gx", "gw"):
        for other in NAMES:
            if other == out:
                continue
            # on the same byte, in its last 16 bytes, and ending in its first 16
            for at in (far[other], far[other] + (size[other] - 1) // 16 * 16, far[other] - (size[out] - 1) // 16 * 16):
                assert ask(dict(far, **{out: at})) == 0, (out, other, at - far[other])
            # next to it
            for at in (far[other] + -(-size[other] // 16) * 16, far[other] - -(-size[out] // 16) * 16):
                assert ask(dict(far, **{out: at})) != 0, (out, other, at - far[other])


@pytest.mark.parametrize("elem", [2, 4, 8])
def test_inputs_may_share_memory(takes, elem):
    assert takes(elem, 1 << 30, 1 << 30, 1 << 30, 1 << 30, 2 << 30, 3 << 30, 40, 264) == 2
