"""The choice of a product's route and what it costs on the host (host code only: nothing is launched)."""
import ctypes as C
import time

import pytest

import capi


def args(M, N, K, dtype=capi.BF16, a_rows=0, b_rows=0):
    return capi.GemmArgs(4096, 4096, None, 4096, M, N, K, M if a_rows else K, N if b_rows else K, N, 0, 1, 0, 0, 0, 0, 1.0, 0.0, dtype, a_rows, b_rows)


def host_us(*problems):
    """Per problem, the quickest of many short stretches of calls, taken in turn: the time without other work on the machine."""
    ask, best = capi.lib().paras_gemm_workspace, [1e9] * len(problems)
    for _ in range(100):
        for i, g in enumerate(problems):
            ref, t = C.byref(g), time.perf_counter()
            for _ in range(100):
                ask(ref)
            best[i] = min(best[i], (time.perf_counter() - t) / 100)
    return [b * 1e6 for b in best]


@pytest.mark.parametrize("shape", [(48, 1024, 2048), (128, 2048, 2048), (1024, 1024, 4096), (512, 4096, 4096)])
def test_the_search_for_a_tile_is_short(shape):
    """Against a call that needs no search (8 rows, 0.3 us here, nearly all of it ctypes): looking at every form and number of parts
    took 6 to 6.5 times as long as that, the search that leaves out what cannot win 2 to 2.8 times."""
    none, search = host_us(args(8, *shape[1:]), args(*shape))
    assert search <= 4.2 * none


@pytest.mark.parametrize("a_rows,b_rows", [(0, 0), (0, 1), (1, 1)])
def test_parts_of_the_contraction_by_size(a_rows, b_rows):
    """The workspace is whole copies of the result in fp32, and only where there are too few tiles for the chip."""
    for M, N, K, split in [(128, 2048, 8192, True), (256, 512, 14336, True), (64, 256, 16384, True), (4096, 4096, 4096, False), (8192, 14336, 512, False), (200, 200, 64, False),
                           (1 << 20, 64, 64, False), (64, 1 << 20, 64, False)]:
        n = capi.lib().paras_gemm_workspace(C.byref(args(M, N, K, a_rows=a_rows, b_rows=b_rows)))
        assert n % (4 * M * N) == 0 and (n > 0) == split and n != 4 * M * N, (M, N, K, n)


@pytest.mark.parametrize("a_rows,b_rows", [(0, 0), (0, 1), (1, 1)])
def test_the_route_does_not_depend_on_how_far_apart_the_rows_of_the_result_are(a_rows, b_rows):
    for ld in (512, 1 << 22, (1 << 31) - 1, 1 << 31, 1 << 33):
        g = args(256, 512, 14336, a_rows=a_rows, b_rows=b_rows)
        g.addend, g.ldc, g.ld_add = 4096, ld, ld
        assert capi.lib().paras_gemm_workspace(C.byref(g)) == capi.lib().paras_gemm_workspace(C.byref(args(256, 512, 14336, a_rows=a_rows, b_rows=b_rows))) > 0, ld
