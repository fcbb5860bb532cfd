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

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("qt", [Q4_0, Q8_0, F16])
@pytest.mark.parametrize("M,N,K", [
    (65, 130, 32),      # 64 x 32 tiles, one block of K
    (129, 1000, 96),    # partial step, one row past two tiles
    (70, 3001, 160),    # N odd: scalar epilogue
    (130, 2050, 2080),  # 65 blocks per row
    (96, 4100, 1056),   # 64 x 64 tiles
    (129, 8200, 1056),  # 64 x 128 tiles
    (513, 4099, 288),   # 128 x 64 tiles, N odd, over 256 workgroups
    (1025, 2049, 544),  # 128 x 128 tiles, one past each way
    (255, 8191, 1056),  # 128 x 128 tiles, one short each way
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
