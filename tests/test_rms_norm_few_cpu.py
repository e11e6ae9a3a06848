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


# (element size, rows, columns, us of the kernels that read g and x once, us of one launch)
MEASURED = [(2, 400, 8, 5.2, 4.4), (2, 600, 8, 5.3, 5.8), (2, 700, 64, 5.3, 5.3), (2, 1000, 64, 5.4, 6.2), (2, 400, 72, 5.3, 4.2), (2, 600, 72, 5.3, 5.6), (2, 600, 136, 6.1, 5.5), (2, 700, 136, 6.2, 6.7),
            (2, 1000, 136, 6.3, 9.3), (2, 1500, 136, 6.7, 11.8), (2, 1000, 192, 6.1, 6.2), (2, 1250, 192, 6.5, 7.4), (2, 600, 200, 6.1, 5.7), (2, 750, 200, 6.2, 7.4), (2, 1000, 256, 6.5, 6.3),
            (2, 1500, 256, 6.8, 8.2), (2, 900, 264, 7.8, 7.6), (2, 1000, 264, 8.0, 8.9), (2, 1250, 384, 8.9, 7.7), (2, 1500, 360, 9.3, 10.7), (2, 1500, 488, 9.6, 10.8), (2, 1750, 584, 15.7, 14.8),
            (2, 2000, 584, 15.8, 18.5), (2, 2000, 632, 15.9, 14.1), (2, 2000, 1024, 15.4, 12.9), (2, 800, 33, 7.3, 6.6), (2, 1000, 65, 8.0, 9.4), (2, 1000, 385, 9.1, 8.1), (2, 2000, 2001, 22.4, 15.4),
            (4, 1500, 36, 8.0, 7.2), (4, 2000, 36, 8.3, 10.2), (4, 2000, 64, 8.2, 6.7), (4, 1250, 132, 8.4, 7.2), (4, 1500, 164, 9.1, 10.0), (4, 1800, 292, 11.9, 11.0), (4, 2000, 292, 12.2, 12.8),
            (4, 2000, 516, 13.6, 13.3), (4, 2000, 1000, 16.2, 14.4), (4, 5500, 8196, 236.6, 186.2), (4, 800, 33, 7.4, 7.1), (4, 1000, 33, 7.6, 8.6), (4, 1000, 129, 7.9, 7.4), (4, 1500, 777, 14.0, 12.8),
            (8, 1500, 34, 8.3, 5.6), (8, 2000, 34, 8.7, 11.0), (8, 2000, 64, 8.7, 7.0), (8, 4000, 64, 12.9, 14.5), (8, 2500, 128, 12.2, 13.2), (8, 2000, 130, 11.7, 12.6), (8, 4000, 256, 16.3, 20.4),
            (8, 3000, 448, 17.2, 15.4), (8, 5500, 512, 26.2, 30.8), (8, 2500, 642, 19.2, 19.9), (8, 5500, 672, 34.5, 29.7), (8, 5500, 1026, 53.2, 48.7), (8, 5500, 2000, 100.8, 61.9), (8, 500, 193, 7.9, 7.1),
            (8, 1000, 193, 10.0, 13.5), (8, 1000, 769, 14.5, 15.0), (8, 1000, 2001, 21.7, 17.2)]


@pytest.mark.parametrize("elem,rows,H,several,one", MEASURED)
def test_one_launch_where_that_was_measured_to_be_no_slower(takes, elem, rows, H, several, one):
    taken = takes(elem, *((i + 1) << 32 for i in range(6)), rows, H) != 0
    assert (one if taken else several) <= 1.02 * min(several, one)
