"""Which tiles a 16-bit product runs on (gemm_flex_plan.h, plain C++: nothing is launched)."""
import ctypes as C
import math
import random
import subprocess

import pytest

import capi

FORMS = (19, 17, 13)          # of x W^T, dy W, dy^T x


@pytest.fixture(scope="module")
def planner(tmp_path_factory):
    where = tmp_path_factory.mktemp("plan")
    (where / "plan.cpp").write_text('''#include <chrono>
#include "kernels/gemm_flex_plan.h"
using namespace paras::flex;
extern "C" long plan(int layout, long M, long N, long K, long batch, int may_split) {          // tile + 64 parts
    const Plan p = plan_of(M, N, K, batch, layout == 2, layout > 0, may_split != 0);
    return p.tile + 64L * p.splits;
}
extern "C" double host_us(int layout, long M, long N, long K) {
    double best = 1e9;
    for (int r = 0; r < 60; ++r) {
        const auto t0 = std::chrono::steady_clock::now();
        for (int i = 0; i < 200; ++i) {
            volatile long m = M;
            volatile long k = plan_of(m, N, K, 1, layout == 2, layout > 0, true).k_per_split;
            (void)k;
        }
        const double us = std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count() * 1e6 / 200;
        if (us < best) best = us;
    }
    return best;
}
extern "C" int forms(int layout) { return layout == 2 ? kFirstOddRows : layout == 1 ? kAlongContraction : kTileCount; }
''')
    subprocess.run(["g++", "-O2", "-std=c++17", "-shared", "-fPIC", f"-I{capi.PKG / 'csrc'}", str(where / "plan.cpp"), "-o", str(where / "plan.so")], check=True)
    lib = C.CDLL(str(where / "plan.so"))
    lib.plan.restype, lib.plan.argtypes = C.c_long, [C.c_int] + [C.c_long] * 4 + [C.c_int]
    lib.host_us.restype, lib.host_us.argtypes = C.c_double, [C.c_int] + [C.c_long] * 3
    return lib


@pytest.mark.parametrize("layout", [0, 1, 2])
def test_every_form_and_every_form_in_parts_is_run_by_a_shape_of_the_gpu_tests(planner, layout):
    from test_gpu_gemm import PARTS, TILES
    assert planner.forms(layout) == FORMS[layout]

    def tile(shape, may_split):
        p = planner.plan(layout, *shape, 1, may_split)
        return p % 64, p // 64
    # (of x W^T with whole tiles of contraction, up to 128 rows are another kernel's)
    whole = {tile(s, 0)[0] for l, s in TILES if l == layout and (layout or s[0] > 128 or s[2] % 64)}
    assert whole == set(range(FORMS[layout]))
    chosen = {tile(s, 1) for l, s in PARTS if l == layout}
    assert all(parts > 1 for _, parts in chosen)
    split = {t for t, _ in chosen}
    rng = random.Random(7)

    def size(lo, hi):
        return int(math.exp(rng.uniform(math.log(lo), math.log(hi))))
    for _ in range(200000):
        M, N, K = 8 * size(3, 2048), 8 * size(1, 2048), 8 * size(1, 2048)
        t, parts = tile((M, N, K), 1)
        assert t in whole and (parts == 1 or t in split), (M, N, K, t, parts)


def test_forms_that_few_rows_cannot_fill_are_not_looked_at(planner):
    """Host time against that of a product whose first form ends the search: 2.3 to 2.6 times as long, 5 times with all of them."""
    long, short = (min(planner.host_us(0, *s) for _ in range(3)) for s in ((48, 1024, 1024), (8192, 8192, 8192)))
    assert long <= 3.6 * short
