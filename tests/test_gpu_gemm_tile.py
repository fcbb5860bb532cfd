"""The tiled MFMA GEMM (csrc/gemm_tile.hpp) against the CPU oracle where it can
go wrong: every tile shape, rows and columns one past and one short of a tile,
K of one block, K that ends inside a step (an odd number of 32-element blocks:
the scale words then start on odd elements), more tiles than compute units,
and K splits with ragged columns.  The bars are test_gpu_ops.assert_close's:
both sides sum in fp32 (a bias adds one f16 rounding, hence inputs that keep
outputs below 8)."""
import numpy as np
import pytest

from tensorlogic_amd import F16, Q4_0, Q8_0
from tensorlogic_amd import synth as S

from test_gpu_ops import assert_close
from test_linear_plan import BASIC, TILED, plan

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("qt", [Q4_0, Q8_0, F16])
@pytest.mark.parametrize("M,N,K", [
    (65, 130, 32),      # one block of K
    (129, 1000, 96),    # partial step, one row past two tiles
    (70, 3001, 160),    # N odd: scalar epilogue
    (130, 2050, 2080),  # 65 blocks per row
    (96, 4100, 1056),
    (129, 8200, 1056),
    (513, 4099, 288),   # N odd
    (1025, 2049, 544),  # one past a tile each way
    (255, 8191, 1056),  # one short each way
    (66, 61, 4128),     # K split, N not a multiple of 8
    (260, 515, 8224),   # K split with a partial last step
])
def test_gemm_tile(dev, oracle, qt, M, N, K):
    x = S.normal_f16(11, f"tx{M}x{K}", (M, K), 0.0, 0.25)
    b = S.normal_f16(11, f"tb{N}", (N,))
    if qt == F16:
        wh = S.normal_f16(11, f"tW{N}x{K}", (N, K), 0.0, 0.02)
        w, ref = dev.tensor(wh), oracle.linear(x, wh, b)
    else:
        gen = {Q4_0: S.q4_0_blocks, Q8_0: S.q8_0_blocks}[qt]
        d = {Q4_0: (1e-4, 1e-3), Q8_0: (2e-5, 2e-4)}[qt]
        blocks = gen(11, f"tW{N}x{K}", N, K, *d)
        w, ref = dev.quantized(blocks, (N, K), qt), oracle.linear_q(x, blocks, 2 if qt == Q4_0 else 8, N, b)
    y = dev.tensor(x).linear(w, dev.tensor(b)).numpy()
    assert_close(y, ref, what=f"tiled gemm {qt} {M}x{N}x{K}")


# a shape for every tile and weight type, with K long enough that the ring of
# scales (two groups of four steps) wraps: 10 steps of 128 or 5 of 256, the last
# one partial; rows and columns one past or short of a tile
EVERY_TILE = [(qt, tile, M, N, K) for tile, shapes in {
    (128, 128): {F16: (193, 10241, 1184), Q4_0: (193, 10241, 1184), Q8_0: (193, 10241, 1184)},
    (128, 64): {F16: (129, 8191, 1312), Q4_0: (1793, 1032, 1184), Q8_0: (1793, 1032, 1184)},
    (64, 128): {F16: (129, 10241, 1184), Q4_0: (65, 10241, 1184), Q8_0: (65, 10241, 1184)},
    (64, 64): {F16: (65, 4099, 1184), Q4_0: (65, 4099, 1184), Q8_0: (65, 4099, 1184)},
    (64, 32): {F16: (65, 2049, 1184), Q4_0: (65, 2049, 1184), Q8_0: (65, 2049, 1184)},
}.items() for qt, (M, N, K) in shapes.items()]


@pytest.mark.parametrize("qt,tile,M,N,K", EVERY_TILE)
def test_every_tile(dev, oracle, qt, tile, M, N, K):
    assert plan(M, N, K, qt)[:4] == (TILED, *tile, 1)
    test_gemm_tile(dev, oracle, qt, M, N, K)


@pytest.mark.parametrize("qt,M,N,K,slices", [(Q4_0, 512, 2560, 10240, 3), (Q8_0, 260, 515, 8224, 3), (Q4_0, 130, 256, 8192, 8),
                                             (F16, 66, 2560, 10240, 6), (F16, 130, 515, 8224, 4)])
def test_split_is_deterministic(dev, oracle, qt, M, N, K, slices):
    """The slices of a K split are summed in slice order: repeated calls give the
    same bits, and the oracle's result."""
    kernel, _, _, splits, ws, _ = plan(M, N, K, qt)
    assert (kernel, splits) == (TILED, slices) and ws > 0
    x = S.normal_f16(15, f"dx{M}x{K}", (M, K), 0.0, 0.25)
    if qt == F16:
        wh = S.normal_f16(15, f"dW{N}x{K}", (N, K), 0.0, 0.02)
        w, ref = dev.tensor(wh), oracle.linear(x, wh)
    else:
        blocks = (S.q4_0_blocks if qt == Q4_0 else S.q8_0_blocks)(15, f"dW{N}x{K}", N, K, 1e-4, 1e-3)
        w, ref = dev.quantized(blocks, (N, K), qt), oracle.linear_q(x, blocks, 2 if qt == Q4_0 else 8, N)
    tx = dev.tensor(x)
    first = tx.linear(w).numpy()
    for _ in range(4):
        assert np.array_equal(tx.linear(w).numpy().view(np.uint16), first.view(np.uint16))
    assert_close(first, ref, what=f"split {qt} {M}x{N}x{K}")


@pytest.mark.parametrize("qt", [Q4_0, Q8_0, F16])
def test_rows_past_the_tiled_ranges(dev, qt):
    """Rows of 2^22 + 32 elements take the basic kernel: few nonzero
    activations, small integers times a power of two, so that every sum is
    exact."""
    M, N, K = 6, 70, (1 << 22) + 32
    assert plan(M, N, K, qt)[0] == BASIC
    rng = np.random.default_rng(16)
    at = np.unique(np.concatenate([[0, 31, 32, K - 33, K - 32, K - 1], rng.integers(0, K, 200)]))
    x = np.zeros((M, K), np.float16)
    x[:, at] = rng.integers(-2, 3, (M, at.size))
    if qt == F16:
        cols = rng.integers(-8, 8, (N, at.size)).astype(np.float16)
        wh = np.zeros((N, K), np.float16)
        wh[:, at] = cols
        w = dev.tensor(wh)
    else:
        size, off = (18, 8) if qt == Q4_0 else (34, 0)
        blocks = rng.integers(0, 256, (N, K // 32, size), dtype=np.uint8)
        blocks[:, :, :2] = np.array([0.0625], np.float16).view(np.uint8)
        e, b = at % 32, blocks[:, at // 32]
        if qt == Q4_0:
            q = b[:, np.arange(at.size), 2 + e % 16] >> np.where(e < 16, 0, 4) & 15
        else:
            q = b[:, np.arange(at.size), 2 + e].view(np.int8)
        cols = (q.astype(np.float32) - off) * 0.0625
        w = dev.quantized(blocks, (N, K), qt)
    want = x[:, at].astype(np.float64) @ cols.astype(np.float64).T
    assert np.array_equal(dev.tensor(x).linear(w).numpy(), want.astype(np.float16))


def test_gemm_tile_keeps_rows_apart(dev):
    """A row of infinities and NaN weights stay in their own outputs: rows and
    columns past the tile's edge and blocks past K add nothing."""
    M, N, K = 67, 131, 1056
    x = S.normal_f16(12, "nx", (M, K))
    x[5] = np.inf
    w = S.normal_f16(12, "nw", (N, K), 0.0, 0.05)
    w[77, K - 1] = np.nan
    y = dev.tensor(x).linear(dev.tensor(w)).numpy()
    bad = ~np.isfinite(y)
    want = np.zeros((M, N), bool)
    want[5] = True
    want[:, 77] = True
    assert np.array_equal(bad, want)


@pytest.mark.parametrize("qt", [Q4_0, Q8_0, F16])
@pytest.mark.parametrize("M", [3, 17, 70])
def test_empty_sum(dev, qt, M):
    """K = 0: every output is the empty sum, or the bias."""
    N = 50
    b = S.normal_f16(13, "eb", (N,))
    x = dev.tensor(np.zeros((M, 0), np.float16))
    w = dev.tensor(np.zeros((N, 0), np.float16)) if qt == F16 else dev.quantized(np.zeros(0, np.uint8), (N, 0), qt)
    keep = dev.tensor(np.full((M, N), np.nan, np.float16))   # (freed: the outputs' blocks are not zero to begin with)
    del keep
    assert not x.linear(w).numpy().any()
    assert np.array_equal(x.linear(w, dev.tensor(b)).numpy(), np.broadcast_to(b, (M, N)))
