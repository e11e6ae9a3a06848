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


# (gate-up, experts, routed rows, columns, contraction steps, grouped_form's choice, {form: us of the layer with it}): what either choice and the best form took
LAYERS = [(1, 4, 677, 3712, 2944, 0, {0: 99.0, 2: 106.7, 14: 96.2}), (1, 8, 1204, 3264, 3328, 5, {5: 150.7, 6: 149.8, 11: 162.0}),
          (1, 8, 7316, 9920, 1536, 5, {5: 683.0, 6: 673.7, 11: 730.3}), (1, 16, 14480, 1024, 1152, 5, {5: 147.0, 6: 146.3, 11: 154.4}),
          (1, 8, 644, 1344, 640, 4, {4: 26.2, 9: 27.6}), (1, 8, 3666, 3840, 640, 5, {5: 110.2, 6: 109.9, 12: 109.7}), (1, 8, 16384, 14336, 4096, 5, {5: 4552.6}),
          (0, 8, 16384, 4096, 14336, 5, {5: 4568.8}), (0, 32, 3920, 768, 2112, 2, {1: 127.8, 2: 113.7, 9: 113.6}), (0, 8, 132, 2240, 9728, 4, {4: 202.1, 7: 214.5}),
          (0, 8, 136, 2432, 8576, 4, {4: 197.5, 7: 209.4}), (0, 8, 168, 2240, 5696, 4, {4: 126.0, 7: 133.5}), (0, 16, 62, 1152, 1664, 4, {4: 46.0, 7: 48.0}),
          (0, 8, 102, 2496, 1664, 4, {4: 47.5, 7: 49.5}), (0, 8, 460, 640, 4096, 4, {4: 58.1, 7: 50.9}), (1, 8, 460, 4096, 640, 2, {2: 57.8, 10: 54.9}),
          (1, 32, 8668, 1280, 1856, 5, {5: 254.3, 12: 215.4}), (1, 8, 4374, 1408, 1088, 6, {0: 73.0, 6: 101.5, 12: 71.0}), (1, 16, 3484, 1024, 1024, 5, {5: 66.7, 12: 53.5}),
          (1, 32, 8676, 5440, 2240, 5, {5: 1114.9, 12: 954.7}), (0, 8, 1160, 1408, 576, 3, {1: 30.2, 3: 35.5}), (0, 16, 4646, 3968, 2624, 5, {5: 495.6, 11: 466.3, 13: 451.3}),
          (1, 64, 28776, 1280, 3072, 5, {5: 724.0, 6: 721.3}), (1, 16, 7032, 5760, 2496, 5, {5: 651.1, 6: 654.6}), (0, 64, 3330, 2496, 1664, 2, {2: 334.8}),
          (1, 4, 720, 10944, 1856, 2, {2: 208.7, 11: 190.4}), (0, 4, 720, 1856, 10944, 3, {3: 208.1}), (1, 8, 1916, 1728, 640, 5, {0: 37.3, 5: 50.5}),
          (1, 8, 7644, 1152, 832, 5, {5: 96.0, 12: 70.4}), (1, 8, 5282, 1728, 576, 5, {5: 84.3, 11: 62.4}), (1, 8, 2144, 768, 1344, 1, {1: 50.0, 2: 37.0}),
          (0, 4, 163, 1024, 7936, 4, {4: 80.6, 7: 64.6}), (0, 4, 76, 832, 12928, 4, {4: 118.7, 7: 93.2}), (0, 4, 70, 1152, 12096, 4, {4: 115.9, 7: 92.7}),
          (0, 4, 241, 768, 10240, 4, {4: 105.7, 7: 83.8}), (0, 4, 537, 576, 11968, 4, {4: 122.8, 7: 98.2})]


@pytest.fixture(scope="module")
def tiles(tmp_path_factory):
    where = tmp_path_factory.mktemp("tiles")
    (where / "tiles.cpp").write_text('''#include "kernels/moe_forms.h"
using namespace paras;
extern "C" int tiles(int swiglu, long E, long R, long N, long K) { return grouped_tiles(swiglu != 0, E, R, N, K); }
extern "C" double rate(int form, int w) {          // of the chip, in 1e15 operations per second
    const GroupedForm& t = kAllForms[form];
    return t.step[w] > 0 ? 2.0 * t.m * t.n * kFormStep * t.per_cu * 256 / t.step[w] * 1e6 / 1e15 : 0.0;
}
extern "C" double bytes_per_us(int cached, int swiglu) {
    return cached ? (swiglu ? TileChoice<true>::from_caches : TileChoice<false>::from_caches) : (swiglu ? TileChoice<true>::from_memory : TileChoice<false>::from_memory);
}
''')
    subprocess.run(["g++", "-O2", "-std=c++17", "-shared", "-fPIC", f"-I{capi.PKG / 'csrc'}", str(where / "tiles.cpp"), "-o", str(where / "tiles.so")], check=True)
    lib = C.CDLL(str(where / "tiles.so"))
    lib.tiles.argtypes = [C.c_int] + [C.c_long] * 4
    lib.rate.restype = lib.bytes_per_us.restype = C.c_double
    return lib


@pytest.mark.parametrize("case", LAYERS)
def test_tiles_by_measured_layers(tiles, form, case):
    """Against grouped_form's choice and against the best form.  (One routing of each layer; the host knows the expected number of tiles only.)"""
    us = case[6]
    assert form(*case[:5]) == case[5]
    assert us[tiles.tiles(*case[:5])] <= 1.06 * min(us.values())


@pytest.mark.parametrize("case", [c for c in MEASURED if c[5] < 0 or c[0] == 0])
def test_tiles_dealt_one_by_one_and_what_stands_for_them(tiles, case):
    """Where they were faster, they or a further form; of down products nowhere else."""
    chosen = tiles.tiles(*case[:5])
    assert chosen >= ONE_BY_ONE if case[5] < 0 else chosen != ONE_BY_ONE


def test_estimates_keep_to_what_the_chip_can_do(tiles):
    assert max(tiles.rate(f, w) for f in range(15) for w in range(2)) <= 2.5
    assert all(tiles.bytes_per_us(0, s) <= 8e6 and tiles.bytes_per_us(1, s) <= 40e6 for s in (0, 1))
