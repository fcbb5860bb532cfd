"""The kernel, tile and K split linear() picks (tlhip_linear_plan, host only):
measured pairs of plans that are a fifth or more apart, the bounds every plan
keeps to, and the shapes that are refused."""
import ctypes as C
import random

import pytest

from tensorlogic_amd import F16, F32, Q4_0, Q6_K, Q8_0
from tensorlogic_amd import _lib as L

GEMV, SKINNY, TILED, BASIC, PLAIN, STAGED = range(6)


def plan(M, N, K, wt):
    """(kernel, tile rows, tile columns, K slices, bytes of partials, RoPE in the epilogue)"""
    p = (C.c_int64 * 6)()
    L.check(L.lib().tlhip_linear_plan(M, N, K, wt, p))
    return tuple(p)


# us, weights in the caches and out of HBM averaged; the other number is the
# skinny kernel's (want TILED) or the tiled kernel's best plan (want SKINNY)
@pytest.mark.parametrize("wt,M,N,K,want,us,other", [
    (F16, 7, 113, 10112, SKINNY, 7.3, 10.2), (F16, 17, 73, 4864, SKINNY, 6.8, 9.4), (F16, 44, 97, 9984, SKINNY, 7.9, 10.5),
    (Q8_0, 10, 91, 10240, SKINNY, 8.1, 11.0), (Q8_0, 13, 347, 8448, SKINNY, 8.3, 11.0), (Q4_0, 12, 230, 6528, SKINNY, 8.3, 11.0),
    (F16, 60, 26331, 256, TILED, 7.5, 24.0), (F16, 35, 14853, 2048, TILED, 15.2, 32.6), (Q8_0, 61, 27631, 384, TILED, 8.3, 18.4),
    (Q8_0, 56, 18368, 8128, TILED, 49.5, 110.5), (Q4_0, 59, 10868, 3008, TILED, 12.5, 26.2), (Q4_0, 56, 27157, 960, TILED, 10.8, 23.2),
])
def test_up_to_64_rows_take_the_faster_kernel(wt, M, N, K, want, us, other):
    assert plan(M, N, K, wt)[0] == want


# us of the tile and split named, and of those an earlier fit of the costs picked
@pytest.mark.parametrize("wt,M,N,K,tile,us,other", [
    (Q8_0, 396, 466, 4288, (64, 32, 1), 10.4, 15.2), (Q4_0, 978, 292, 5760, (64, 32, 1), 12.7, 17.5),
    (Q4_0, 652, 9307, 480, (128, 128, 1), 21.8, 30.3), (Q4_0, 374, 2579, 576, (64, 64, 1), 6.7, 9.1),
    (Q4_0, 130, 15689, 384, (128, 128, 1), 11.3, 14.8), (F16, 995, 108, 8320, (64, 32, 4), 11.5, 14.9),
    (Q8_0, 40, 2048, 5632, (64, 32, 4), 10.4, 11.9), (F16, 100, 7680, 2560, (64, 64, 1), 16.0, 18.7),
])
def test_tile_and_split(wt, M, N, K, tile, us, other):
    kernel, rows, cols, splits, _, _ = plan(M, N, K, wt)
    assert kernel == TILED and (rows, cols, splits) == tile


# us of the staged and of the tiled kernel's planned launch
@pytest.mark.parametrize("wt,M,N,K,staged,tiled", [
    (Q4_0, 2000, 23565, 256, 68.9, 98.2), (Q4_0, 1720, 11632, 448, 41.6, 55.6), (Q8_0, 916, 14250, 320, 27.7, 38.7),
    (Q8_0, 916, 17175, 512, 42.3, 55.1), (Q8_0, 883, 15011, 768, 44.8, 53.2), (Q4_0, 1078, 8700, 448, 22.4, 29.0),
    (Q8_0, 1024, 9583, 2048, 85.0, 74.0), (Q4_0, 855, 4827, 3456, 67.4, 53.2), (F16, 223, 8369, 1024, 28.2, 14.2),
    (Q8_0, 738, 5483, 4928, 88.7, 75.8), (Q4_0, 129, 10240, 256, 9.8, 7.0),
])
def test_many_tiles_of_a_short_k_are_staged(wt, M, N, K, staged, tiled):
    assert plan(M, N, K, wt)[0] == (STAGED if staged < tiled else TILED)


def test_every_plan_keeps_to_its_bounds():
    """Partials of a split within the fixed workspace of the no-allocation entry
    point, none without a split, tiles of the kernels' shapes; up to 4 rows a
    GEMV wherever it is built for the row length."""
    rng = random.Random(3)
    for _ in range(4000):
        wt = rng.choice([F16, Q4_0, Q8_0])
        M, N, K = rng.randrange(1, 2100), int(2 ** rng.uniform(0, 16)), 32 * int(2 ** rng.uniform(0, 9))
        kernel, rows, cols, splits, ws, rope = plan(M, N, K, wt)
        assert ws <= 20 << 20 and (ws > 0) == (splits > 1)
        if M <= 4:
            assert kernel == GEMV or (wt != F16 and K > 4096)
        elif kernel == SKINNY:
            assert M <= 64 and K % 64 == 0 and rows in (16, 32, 48, 64) and cols in (32, 64)
        elif kernel == STAGED:
            assert M > 64 and K % 64 == 0 and K <= 1024 and (rows, cols, splits) == (128, 128, 1)
        else:
            assert (kernel, rows, cols) in [(TILED, a, b) for a, b in ((128, 128), (128, 64), (64, 128), (64, 64), (64, 32))]
        if kernel == TILED and splits > 1:
            assert ws >= splits * M * N * 4


def test_other_forms():
    assert plan(70, 50, 0, Q8_0)[0] == PLAIN and plan(3, 50, 0, Q4_0)[0] == PLAIN
    assert plan(5, 122, 50, F16)[0] == PLAIN and plan(3, 122, 50, F16)[0] == GEMV
    assert plan(5, 64, (1 << 22) + 32, Q4_0)[0] == BASIC
    assert plan(1, 32000, 2048, Q6_K)[0] == GEMV and plan(300, 4096, 2048, Q6_K) == (*plan(300, 4096, 2048, F16)[:5], 0)
    for args, kind in (((5, 64, 48, Q4_0), "InvalidDimension"), ((0, 64, 64, F16), "InvalidDimension"),
                       ((5, 64, 64, F32), "DtypeError")):
        with pytest.raises(L.TLHipError) as e:
            plan(*args)
        assert e.value.kind == kind
