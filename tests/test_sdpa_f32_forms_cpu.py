"""Which form the one-pass fp32 attention kernel takes (sdpa_f32_forms.h, plain C++: nothing is launched)."""
import ctypes as C
import subprocess

import pytest

import capi

FORMS = ("16x16", "32x16", "16x32", "32x32")          # queries x keys of a turn
# causal, heads of 128: (heads, queries, {form: us})
CAUSAL = [(1, 6144, {"16x16": 187.6, "16x32": 147.4, "32x32": 259.7}), (1, 8192, {"16x16": 273.8, "16x32": 240.1, "32x32": 344.8}), (1, 8256, {"16x16": 273.7, "16x32": 289.1, "32x32": 349.5}),
          (1, 9216, {"16x16": 317.6, "16x32": 344.4, "32x32": 388.0}), (1, 10240, {"16x16": 359.8, "16x32": 413.8, "32x32": 431.2}), (1, 16384, {"16x16": 833.1, "16x32": 929.9, "32x32": 813.2}),
          (2, 4096, {"16x16": 175.3, "16x32": 130.6, "32x32": 177.1}), (2, 6144, {"16x16": 282.1, "16x32": 290.8, "32x32": 263.5}), (2, 7680, {"16x16": 444.3, "16x32": 431.9, "32x32": 373.8}),
          (2, 8192, {"16x16": 486.8, "16x32": 480.5, "32x32": 431.6}), (2, 9216, {"16x16": 584.7, "16x32": 631.9, "32x32": 602.9}), (2, 10240, {"16x16": 698.3, "16x32": 769.8, "32x32": 730.1}),
          (4, 4096, {"16x16": 261.5, "16x32": 259.8, "32x32": 316.3}), (4, 7168, {"16x16": 680.0, "16x32": 765.3, "32x32": 691.8}), (4, 8192, {"16x16": 885.4, "16x32": 960.6, "32x32": 861.9}),
          (8, 6144, {"16x16": 1001.6, "16x32": 1133.7, "32x32": 1046.7}), (8, 8192, {"16x16": 1697.9, "16x32": 1917.5, "32x32": 1727.0})]
# unmasked, heads of 256: (sequences, heads, queries, {form: us})
WIDE = [(7, 8, 66, {"16x16": 23.9, "16x32": 23.3}), (7, 8, 86, {"16x16": 26.0, "16x32": 25.5}), (7, 8, 112, {"16x16": 27.3, "16x32": 29.4}), (7, 8, 192, {"16x16": 49.0, "16x32": 59.1}),
        (1, 16, 128, {"16x16": 14.1, "16x32": 14.7})]


@pytest.fixture(scope="module")
def form(tmp_path_factory):
    where = tmp_path_factory.mktemp("forms")
    (where / "forms.cpp").write_text('''#include "kernels/sdpa_f32_forms.h"
extern "C" int form(long B, long H, long S, int D, int causal) {
    paras_sdpa_args a{};
    a.B = B; a.Hq = a.Hkv = H; a.Lq = a.Lk = S; a.D = D; a.is_causal = causal;
    return static_cast<int>(D == 64 ? paras::form_of<64>(a) : D == 128 ? paras::form_of<128>(a) : paras::form_of<256>(a));
}
''')
    subprocess.run(["g++", "-O2", "-std=c++17", "-shared", "-fPIC", f"-I{capi.PKG / 'csrc'}", f"-I{capi.PKG.parent / 'include'}", str(where / "forms.cpp"), "-o", str(where / "forms.so")], check=True)
    f = C.CDLL(str(where / "forms.so")).form
    f.restype, f.argtypes = C.c_int, [C.c_long] * 3 + [C.c_int] * 2
    return f


@pytest.mark.parametrize("H,S,us", CAUSAL)
def test_causal_forms_by_measured_problems(form, H, S, us):
    assert us[FORMS[form(1, H, S, 128, 1)]] <= 1.015 * min(us.values())


@pytest.mark.parametrize("B,H,S,us", WIDE)
def test_forms_of_256_elements_by_measured_problems(form, B, H, S, us):
    assert us[FORMS[form(B, H, S, 256, 0)]] <= 1.015 * min(us.values())
