"""What paras_sdpa_workspace and paras_sdpa_kernel_name answer (host code only: nothing is launched)."""
import ctypes as C
import random
import subprocess

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


@pytest.mark.parametrize("apart", [1 << 20, (1 << 34) - 8, 1 << 34, 80 * 2 * 8 * 131072 * 128, (1 << 40) + 4096])
def test_one_token_attention_does_not_depend_on_how_far_apart_sequences_are(apart):
    """The one-token kernel takes caches that hold all layers of a sequence together, whose sequences are 2^34 elements apart and more."""
    q, k, out = torch.zeros(2, 32, 1, 128, dtype=torch.bfloat16), torch.zeros(2, 8, 1000, 128, dtype=torch.bfloat16), torch.zeros(2, 32, 1, 128, dtype=torch.bfloat16)
    a = capi.sdpa_args(q, k, k, out)
    want = capi.lib().paras_sdpa_workspace(C.byref(a))
    a.k_strides[0] = a.v_strides[0] = apart
    assert capi.lib().paras_sdpa_kernel_name(C.byref(a)) == b"decode_split" and capi.lib().paras_sdpa_workspace(C.byref(a)) == want


@pytest.fixture(scope="module")
def deal(tmp_path_factory):
    """sdpa_flash_deal.h as a library of its own (plain C++, no HIP)."""
    where = tmp_path_factory.mktemp("deal")
    (where / "deal.cpp").write_text('''#include "kernels/sdpa_flash_deal.h"
#include <chrono>
using namespace paras::flash;
extern "C" long by_runs(long heads, long nq, long wgs, long G) { return most_by_runs(heads, nq, wgs, G); }
extern "C" long by_places(long heads, long nq, long wgs, long G) { return most_by_places(heads, nq, wgs, G); }
extern "C" double seconds(long BH, long nq, long blocks, double bytes, int times) {
    const auto start = std::chrono::steady_clock::now();
    volatile double sink = 0;
    for (int i = 0; i < times; ++i) sink = sink + deal_of(BH, nq, blocks, bytes).cost;
    return std::chrono::duration<double>(std::chrono::steady_clock::now() - start).count();
}
extern "C" int group(long BH, long nq, long blocks, double bytes) { return deal_of(BH, nq, blocks, bytes).group; }
extern "C" long together(long heads, long nq, long Lk, long D) { return heads_together(heads, nq, Lk, D); }
extern "C" double cost(long BH, long nq, long blocks, double bytes) { return deal_of(BH, nq, blocks, bytes).cost; }
''')
    subprocess.run(["g++", "-O2", "-std=c++17", "-shared", "-fPIC", f"-I{capi.PKG / 'csrc'}", str(where / "deal.cpp"), "-o", str(where / "deal.so")], check=True)
    lib = C.CDLL(str(where / "deal.so"))
    for f in (lib.by_runs, lib.by_places, lib.together):
        f.restype, f.argtypes = C.c_long, [C.c_long] * 4
    lib.seconds.restype, lib.seconds.argtypes = C.c_double, [C.c_long] * 3 + [C.c_double, C.c_int]
    lib.group.restype, lib.cost.restype = C.c_int, C.c_double
    lib.group.argtypes = lib.cost.argtypes = [C.c_long] * 3 + [C.c_double]
    return lib


def most_one_by_one(heads, nq, wgs, G):
    """The kernel's numbering of items, item by item: what the workgroup with the most gets, in tiles of keys."""
    load = [0] * wgs
    for i in range(heads * nq):
        turn, x = divmod(i, wgs)
        load[wgs - 1 - x if turn % 2 else x] += nq - i % (G * nq) // G
    return max(load)


def test_the_most_a_workgroup_gets_is_what_dealing_item_by_item_gives(deal):
    rng = random.Random(5)
    cases = [(1, 1, 1, 1), (8, 6, 32, 8), (252, 10, 256, 1), (7, 33, 32, 7), (3, 2, 300, 1), (64, 16, 256, 64), (5, 25, 32, 5)]
    for n in range(400):
        G = rng.randint(1, 12)
        cases.append((G * rng.randint(1, 20), rng.randint(1, 40), rng.randint(1, 40 if n % 2 else 300), G))
    for c in cases:
        want = most_one_by_one(*c)
        assert deal.by_runs(*c) == want and deal.by_places(*c) == want, c


@pytest.mark.parametrize("B,H,S", [(3, 36, 2560), (9, 12, 2560), (3, 28, 3584), (15, 4, 5120), (5, 28, 2048), (9, 4, 8192), (1, 36, 8192), (7, 12, 3840), (5, 14, 3840), (13, 12, 1792),
                                   (3, 28, 1500), (3, 28, 4096), (5, 8, 6175), (6, 8, 5376), (4, 32, 4096)])
def test_causal_query_tiles_are_dealt_evenly(deal, B, H, S):
    """No workgroup has over a tenth more than its share (one head at a time it is 1.3 to 2 times for most of these), whether the heads are dealt to the
    XCDs or not and however many items there are; and the cost that is reported is that of the deal."""
    nq, BH = -(-S // 256), B * H
    blocks = min(256, BH * nq)
    blocks -= blocks % 8 if BH % 8 == 0 else 0
    heads, wgs = (BH // 8, blocks // 8) if BH % 8 == 0 else (BH, blocks)
    G = deal.group(BH, nq, blocks, 512.0 * S)
    assert heads % G == 0
    uneven = most_one_by_one(heads, nq, wgs, G) / (heads * nq * (nq + 1) / 2 / wgs)
    assert uneven <= 1.1, (G, uneven)
    fits = G * S * 512 * (8 if BH % 8 == 0 else 1) <= 128e6
    assert deal.cost(BH, nq, blocks, 512.0 * S) >= 0.45 + 0.55 * uneven - 1e-9 and (not fits or deal.cost(BH, nq, blocks, 512.0 * S) <= 0.45 + 0.55 * uneven + 1e-9)


@pytest.mark.parametrize("B,H,S", [(3, 28, 1500), (7, 12, 1500), (5, 28, 1500), (5, 12, 2048), (1, 36, 4096), (15, 4, 1500), (5, 16, 1500), (4, 32, 4096), (1, 97, 8192)])
def test_a_deal_is_worked_out_in_a_microsecond(deal, B, H, S):
    """0.2 to 1.2 us, once per call; a walk over every item of every group took 10 to 60, twice."""
    nq, BH = -(-S // 256), B * H
    blocks = min(256, BH * nq) // 8 * 8 if BH % 8 == 0 else min(256, BH * nq)
    assert min(deal.seconds(BH, nq, blocks, 512.0 * S, 100) for _ in range(200)) / 100 <= 4e-6


# (sequences, heads, queries, head size, {heads together: us})
TOGETHER = [(29, 24, 308, 128, {1: 53.0, 3: 53.9, 29: 61.1, 87: 63.1}), (18, 40, 550, 128, {2: 110.7, 3: 111.7, 9: 113.9, 15: 119.1, 18: 117.0, 30: 130.1, 90: 133.0}),
            (6, 64, 194, 128, {2: 20.5, 4: 20.5, 8: 20.4, 16: 20.2, 24: 22.6, 48: 23.7}), (10, 64, 276, 128, {2: 47.1, 4: 47.0, 8: 46.1, 16: 49.3, 40: 53.9, 80: 53.0}),
            (7, 64, 602, 128, {2: 75.0, 4: 74.4, 8: 77.2, 14: 81.3, 28: 84.9, 56: 92.5}), (28, 64, 321, 64, {2: 67.4, 4: 67.4, 8: 68.9, 16: 68.4, 32: 81.5, 56: 74.6, 224: 74.8}),
            (10, 40, 263, 256, {2: 86.1, 5: 86.0, 10: 86.7, 25: 93.2, 50: 92.3}), (2, 32, 1334, 256, {2: 98.0, 4: 102.5, 8: 101.8}), (4, 16, 2048, 64, {2: 54.4, 4: 50.9, 8: 45.7}),
            (8, 8, 1024, 64, {2: 21.9, 4: 22.0, 8: 17.4}), (12, 2, 4143, 64, {1: 95.4, 3: 69.7}), (2, 32, 700, 128, {2: 22.3, 4: 20.4, 8: 20.1}), (19, 8, 1749, 64, {1: 90.3, 19: 81.0}),
            (37, 8, 261, 64, {1: 15.7, 37: 14.4}), (7, 32, 610, 64, {2: 29.6, 4: 27.3, 7: 25.6, 14: 25.0, 28: 24.3}), (20, 64, 134, 128, {2: 51.9, 4: 42.9, 8: 42.9, 16: 43.3, 32: 48.0, 80: 48.2}),
            (2, 32, 934, 256, {2: 70.2, 4: 59.9, 8: 61.2}), (2, 32, 4326, 64, {2: 188.4, 4: 171.6, 8: 172.6})]


@pytest.mark.parametrize("B,H,S,D,us", TOGETHER)
def test_heads_whose_longest_tiles_are_taken_first(deal, B, H, S, D, us):
    """Of the numbers measured, the chosen one (or the next, where it was not measured) is within 4 % of the best."""
    group = deal.together(B * H // 8, -(-S // 128), S, D)
    assert (B * H // 8) % group == 0
    assert us[min(us, key=lambda g: abs(g - group))] <= 1.04 * min(us.values()), group


def test_heads_together_divide_the_heads_of_an_xcd(deal):
    for heads in range(1, 300):
        for nq, Lk, D in ((1, 128, 64), (2, 200, 128), (3, 300, 256), (9, 1100, 64), (40, 5000, 128), (1 << 20, 1 << 27, 256)):
            g = deal.together(heads, nq, Lk, D)
            assert 1 <= g <= heads and heads % g == 0 and (g > 1 or heads % 2 or heads == 1)
