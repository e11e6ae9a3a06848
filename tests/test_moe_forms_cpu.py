"""Which tiles the products of an expert layer run on (moe_forms.h, plain C++: nothing is launched)."""
import ctypes as C
import subprocess

import pytest

import capi

ONE_BY_ONE, SUPER_TILES = 6, 5
# (gate-up, experts, routed rows, columns, contraction steps, us of the layer with 256 x 256 tiles one by one less that of the best other form)
MEASURED = [
    (1, 8, 10342, 1152, 1408, 14), (1, 32, 15856, 704, 1152, 14), (0, 32, 6628, 2112, 2688, 22), (0, 64, 20142, 1216, 2048, 17), (0, 8, 11832, 3264, 12736, 61),
    (0, 4, 8008, 3392, 704, 2), (0, 16, 10436, 640, 5824, 22), (1, 32, 7800, 1792, 1664, 11), (1, 4, 3968, 1152, 1024, 10), (1, 4, 3702, 5312, 512, 12),
    (1, 8, 12290, 1152, 3648, -80), (1, 4, 8008, 704, 3392, -14), (1, 4, 6109, 3648, 3904, -66), (1, 8, 9584, 2304, 3072, -69), (1, 8, 1526, 2752, 1856, -11), (1, 4, 1668, 3264, 832, -15),
    (1, 4, 587, 6016, 1664, -13), (0, 8, 11190, 2112, 5760, -92), (0, 64, 25116, 1088, 5312, -63), (0, 16, 8586, 1216, 1280, -14), (0, 8, 7878, 3328, 1280, -13), (0, 32, 6184, 2368, 6976, -31), (0, 64, 29106, 1472, 3008, -35), (0, 8, 13786, 2112, 4800, -57),
]


@pytest.fixture(scope="module")
def form(tmp_path_factory):
    where = tmp_path_factory.mktemp("forms")
    (where / "forms.cpp").write_text('#include "kernels/moe_forms.h"\nextern "C" int form(int swiglu, long E, long R, long N, long K) { return paras::grouped_form(swiglu != 0, E, R, N, K); }\n')
    subprocess.run(["g++", "-O2", "-std=c++17", "-shared", "-fPIC", f"-I{capi.PKG / 'csrc'}", str(where / "forms.cpp"), "-o", str(where / "forms.so")], check=True)
    f = C.CDLL(str(where / "forms.so")).form
    f.restype, f.argtypes = C.c_int, [C.c_int] + [C.c_long] * 4
    return f


@pytest.mark.parametrize("case", MEASURED)
def test_tiles_are_dealt_one_by_one_where_that_was_measured_to_be_faster(form, case):
    assert (form(*case[:5]) == ONE_BY_ONE) == (case[5] < 0)


def test_every_form_is_chosen_by_a_shape_of_the_gpu_tests(form):
    """TILE_SHAPES of test_gpu_moe.py reaches both products' tile forms, super-tiles and tiles one by one among them."""
    from test_gpu_moe import TILE_SHAPES
    chosen = [(form(1, E, T * k, I, H), form(0, E, T * k, H, I)) for T, E, k, H, I in TILE_SHAPES]
    assert {f for pair in chosen for f in pair} == set(range(7)), chosen
    assert ONE_BY_ONE in {g for g, _ in chosen} and ONE_BY_ONE in {d for _, d in chosen}, chosen


def test_every_tile_of_both_products_is_chosen_by_a_shape_of_the_gpu_tests(tmp_path):
    """TILE_SHAPES and FURTHER_TILE_SHAPES of test_gpu_moe.py reach all that grouped_tiles chooses among, and sizes from one row to the largest get a form that the product has."""
    from test_gpu_moe import FURTHER_TILE_SHAPES, TILE_SHAPES
    (tmp_path / "tiles.cpp").write_text('#include "kernels/moe_forms.h"\n'
                                        'extern "C" int tiles(int swiglu, long E, long R, long N, long K) { return paras::grouped_tiles(swiglu != 0, E, R, N, K); }\n'
                                        'extern "C" int has(int swiglu, int form) { return form >= 0 && form < paras::kAllFormCount && paras::kAllForms[form].step[swiglu ? 0 : 1] > 0; }\n')
    subprocess.run(["g++", "-O2", "-std=c++17", "-shared", "-fPIC", f"-I{capi.PKG / 'csrc'}", str(tmp_path / "tiles.cpp"), "-o", str(tmp_path / "tiles.so")], check=True)
    lib = C.CDLL(str(tmp_path / "tiles.so"))
    lib.tiles.argtypes = [C.c_int] + [C.c_long] * 4
    shapes = TILE_SHAPES + FURTHER_TILE_SHAPES
    assert {lib.tiles(1, E, T * k, I, H) for T, E, k, H, I in shapes} >= {f for f in range(15) if lib.has(1, f)}
    assert {lib.tiles(0, E, T * k, H, I) for T, E, k, H, I in shapes} >= {f for f in range(15) if lib.has(0, f)}
    for E in (1, 3, 64, 4096):
        for R in (1, 31, 32, 33, 1000, 16384, 1 << 24):
            for N, K in ((64, 64), (64, 14336), (14336, 64), (4096, 4096), (1 << 20, 1 << 20)):
                for swiglu in (0, 1):
                    assert lib.has(swiglu, lib.tiles(swiglu, E, R, N, K)), (swiglu, E, R, N, K)
