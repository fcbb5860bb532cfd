"""The staged MFMA GEMM (csrc/kernels_gemm_staged.hip) against the CPU oracle:
many tiles of a short K, with rows and columns one past and short of a tile, K
of one to sixteen steps (fewer and more than the LDS stages, which are three
and, up to 256 tiles, four), and the epilogues a model's prompt pass gives it.
The bars are test_gpu_ops.assert_close's (inputs as in test_gpu_gemm_tile)."""
import pytest

from tensorlogic_amd import F16, Q4_0, Q8_0
from tensorlogic_amd import synth as S

from test_gpu_model import _compare
from test_gpu_ops import assert_close
from test_linear_plan import STAGED, plan

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("qt,M,N,K", [(qt, *s) for qt in (Q4_0, Q8_0) for s in [
    (1100, 3700, 64), (513, 8193, 320), (65, 32900, 192), (2047, 2180, 448), (1290, 3330, 1024)]] + [
    # up to 256 tiles: four stages, two, three and five steps
    (qt, *s) for qt in (Q4_0, Q8_0, F16) for s in [(300, 7000, 128), (300, 9500, 192)]] + [
    (Q8_0, 257, 8190, 320), (F16, 257, 8190, 320)])
def test_gemm_staged(dev, oracle, qt, M, N, K):
    assert plan(M, N, K, qt)[0] == STAGED
    x = S.normal_f16(14, f"sx{M}x{K}", (M, K), 0.0, 0.25)
    b = S.normal_f16(14, f"sb{N}", (N,))
    if qt == F16:
        wh = S.normal_f16(14, f"sW{N}x{K}", (N, K), 0.0, 0.02)
        w, ref = dev.tensor(wh), oracle.linear(x, wh, b)
    else:
        gen = {Q4_0: S.q4_0_blocks, Q8_0: S.q8_0_blocks}[qt]
        d = {Q4_0: (1e-4, 1e-3), Q8_0: (2e-5, 2e-4)}[qt]
        blocks = gen(14, f"sW{N}x{K}", N, K, *d)
        w, ref = dev.quantized(blocks, (N, K), qt), oracle.linear_q(x, blocks, 2 if qt == Q4_0 else 8, N, b)
    y = dev.tensor(x).linear(w, dev.tensor(b)).numpy()
    assert_close(y, ref, what=f"staged gemm {qt} {M}x{N}x{K}")


def test_llama_wide_ffn_prompt(dev, oracle, tmp_path):
    """SwiGLU pairs in the staged epilogue: 450 rows of a 256 -> 2 x 4352 gate/up."""
    dims = dict(n_layers=1, hidden=256, inter=4352, n_heads=4, n_kv=2, vocab=1000)
    assert plan(450, 2 * dims["inter"], dims["hidden"], Q4_0)[0] == STAGED
    path = str(tmp_path / "wide_ffn.gguf")
    S.write_llama_gguf(path, seed=33, **dims)
    _compare(dev, oracle, path, 0, S.token_ids(33, "prompt", 450, dims["vocab"]), 2, max_ctx=500)


def test_phi2_wide_ffn_prompt(dev, oracle, tmp_path):
    """Bias and GELU in the staged epilogue: 500 rows of a 320 -> 9600 fc1."""
    dims = dict(n_layers=1, hidden=320, inter=9600, n_heads=4, vocab=1000, rot=32)
    assert plan(500, dims["inter"], dims["hidden"], Q8_0)[0] == STAGED
    path = str(tmp_path / "wide_fc1.gguf")
    S.write_phi2_gguf(path, seed=34, **dims)
    _compare(dev, oracle, path, 1, S.token_ids(34, "prompt", 500, dims["vocab"]), 2, max_ctx=550)
