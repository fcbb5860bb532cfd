"""The many-row forms of the TL program's builtins where they can go wrong:
the matrix-core einsums at tile edges and odd key counts, and the 16-byte
elementwise, mask, broadcast and one-wave-per-row softmax kernels on both
sides of the rules that choose them."""
import numpy as np
import pytest

from tensorlogic_amd import F32
from tensorlogic_amd import synth as S
from tensorlogic_amd.tensor import attention, einsum

from test_einsum_rule import einsum_rule  # noqa: F401 (fixture "rule")
from test_gpu_ops import assert_close, ulp_diff

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("I,J,H,Hkv,D", [(16, 16, 4, 2, 64), (15, 40, 4, 2, 64), (33, 65, 8, 2, 80), (64, 128, 4, 4, 128),
                                         (65, 129, 6, 3, 64), (130, 31, 2, 1, 80), (31, 257, 4, 1, 128)])
def test_einsums_many_rows(dev, oracle, I, J, H, Hkv, D):
    q = S.normal_f16(21, f"mq{I}{D}", (I, H, D))
    k = S.normal_f16(21, f"mk{J}{D}", (J, Hkv, D))
    v = S.normal_f16(21, f"mv{J}{D}", (J, Hkv, D))
    sc = einsum("ihd,jhd->ihj", dev.tensor(q), dev.tensor(k)).numpy()
    assert_close(sc, oracle.einsum_scores(q, k), what=f"scores {I}x{J} H{H}/{Hkv} D{D}")
    p = np.random.default_rng(I + J).random((I, H, J)).astype(np.float32)
    p = (p / p.sum(-1, keepdims=True)).astype(np.float16)
    out = einsum("ihj,jhd->ihd", dev.tensor(p), dev.tensor(v)).numpy()
    assert_close(out, oracle.einsum_context(p, v), what=f"context {I}x{J} H{H}/{Hkv} D{D}")


@pytest.mark.parametrize("I,J,H,Hkv,D", [(65, 129, 32, 8, 64), (33, 257, 64, 2, 64), (17, 1000, 32, 32, 80), (100, 16, 48, 4, 80),
                                         (129, 31, 32, 8, 80), (48, 65, 64, 64, 128), (130, 128, 16, 2, 128), (66, 17, 60, 4, 128)])
def test_einsums_on_the_matrix_cores(dev, oracle, rule, I, J, H, Hkv, D):
    """The same past the sizes from which the matrix-core kernels are taken:
    rows and keys on, one past and short of their tiles."""
    assert rule.scores(I, H, J) and rule.context(I, H, J, D)
    test_einsums_many_rows(dev, oracle, I, J, H, Hkv, D)


def test_context_on_the_matrix_cores_keeps_non_finite_values_apart(dev, rule):
    I, J, H, D = 37, 71, 64, 64
    assert rule.scores(I, H, J) and rule.context(I, H, J, D)
    q, k, v = (S.normal_f16(22, n, s) for n, s in (("q", (I, H, D)), ("k", (J, H, D)), ("v", (J, H, D))))
    q[36, 0, 3], k[70, 1, 0], v[70, 0, 5] = np.inf, np.nan, np.inf
    sc = einsum("ihd,jhd->ihj", dev.tensor(q), dev.tensor(k)).numpy()
    want = np.zeros((I, H, J), bool)
    want[36, 0], want[:, 1, 70] = True, True
    assert np.array_equal(~np.isfinite(sc), want)
    p = np.full((I, H, J), 1.0 / J, np.float16)
    out = einsum("ihj,jhd->ihd", dev.tensor(p), dev.tensor(v)).numpy()
    assert np.array_equal(np.isposinf(out), np.broadcast_to(np.arange(D) == 5, (I, H, D)) & (np.arange(H) == 0)[None, :, None])


def test_einsums_keep_non_finite_values_apart(dev):
    """An infinite query row, key or value shows up only where it takes part:
    padding rows and keys of the tiles add nothing."""
    I, J, H, D = 37, 71, 2, 64
    q, k, v = (S.normal_f16(22, n, s) for n, s in (("q", (I, H, D)), ("k", (J, H, D)), ("v", (J, H, D))))
    q[36, 0, 3] = np.inf
    k[70, 1, 0] = np.nan
    sc = einsum("ihd,jhd->ihj", dev.tensor(q), dev.tensor(k)).numpy()
    want = np.zeros((I, H, J), bool)
    want[36, 0] = True
    want[:, 1, 70] = True
    assert np.array_equal(~np.isfinite(sc), want)
    v[70, 0, 5] = np.inf
    p = np.full((I, H, J), 1.0 / J, np.float16)
    out = einsum("ihj,jhd->ihd", dev.tensor(p), dev.tensor(v)).numpy()
    assert np.array_equal(np.isposinf(out), np.broadcast_to(np.arange(D) == 5, (I, H, D)) & (np.arange(H) == 0)[None, :, None])


@pytest.mark.parametrize("rows,n", [(70000 // 8, 8), (33, 2048), (65, 1025), (31, 2113)])
def test_elementwise_wide(dev, oracle, rows, n):
    x = S.normal_f16(23, f"x{n}", (rows, n), 0.0, 4.0)
    u = S.normal_f16(23, f"u{n}", (rows, n))
    b = S.normal_f16(23, f"b{n}", (n,))
    tx, tu, tb = dev.tensor(x), dev.tensor(u), dev.tensor(b)
    for got, ref in ((tx.sigmoid(), oracle.sigmoid(x)), (tx.silu(), oracle.silu(x)), (tx.gelu(), oracle.gelu(x)),
                     (tx.silu_mul(tu), oracle.swiglu(x, u))):
        assert ulp_diff(got.numpy(), ref).max() <= 1
    f = np.float32
    for got, ref in ((tx + tu, x.astype(f) + u), (tx * tu, x.astype(f) * u), (tx * 0.125, x.astype(f) * f(0.125)),
                     (tx + tb, x.astype(f) + b), (tx * tb, x.astype(f) * b)):
        assert np.array_equal(got.numpy().view(np.uint16), ref.astype(np.float16).view(np.uint16))


@pytest.mark.parametrize("fn", ["gelu", "sigmoid", "silu"])
def test_activations_over_all_f16(dev, oracle, fn):
    x = np.arange(65536, dtype=np.uint16).view(np.float16)
    got, ref = getattr(dev.tensor(x), fn)().numpy(), getattr(oracle, fn)(x)
    assert np.array_equal(np.isnan(got), np.isnan(ref))
    ok = ~np.isnan(ref)
    # one f16 rounding of an f32 value within a few f32 ulps of the oracle's
    assert ulp_diff(got[ok], ref[ok]).max() <= 1


def test_activation_errors_against_64_bits(dev):
    """sigmoid and gelu over all f16 inputs against 64-bit arithmetic, in f16
    ulps of the result.  The bars are what expf with a full divide, and tanhf,
    give on the device (largest and mean error; sigmoid 0.5001209 / 0.1374203,
    gelu 1.6957698 / 0.1430744): the hardware's exp and reciprocal may not be
    further off."""
    x = np.arange(65536, dtype=np.uint16).view(np.float16)
    x = x[np.isfinite(x)]
    f = x.astype(np.float64)
    with np.errstate(over="ignore"):
        refs = {"sigmoid": (1 / (1 + np.exp(-f)), 0.500121, 0.13742034),
                "gelu": (0.5 * f * (1 + np.tanh(np.sqrt(2 / np.pi) * (f + 0.044715 * f**3))), 1.695770, 0.14307442)}
    for fn, (ref, most, mean) in refs.items():
        got = getattr(dev.tensor(x), fn)().numpy().astype(np.float64)
        err = np.abs(got - ref) / 2.0 ** (np.floor(np.log2(np.maximum(np.abs(ref), 2.0**-14))) - 10)
        assert err.max() <= most and err.mean() <= mean, (fn, err.max(), err.mean())


@pytest.mark.parametrize("I,H,J", [(48, 32, 48), (40, 32, 61), (130, 4, 136)])
def test_mask_wide(dev, I, H, J):
    sc = S.normal_f16(24, f"s{I}{J}", (I, H, J))
    m = (np.random.default_rng(J).random((I, J)) < 0.5).astype(np.float16)
    m[0, 0] = -0.0
    full = np.broadcast_to(m[:, None, :], (I, H, J))
    want = np.where(full == 0, np.float16(-10000), sc)
    for mask in (m, np.ascontiguousarray(full)):
        got = dev.tensor(sc).apply_attention_mask(dev.tensor(mask)).numpy()
        assert np.array_equal(got.view(np.uint16), want.view(np.uint16))


@pytest.mark.parametrize("dtype", [np.float16, np.float32])
@pytest.mark.parametrize("src,dst", [((70, 4, 1, 64), (70, 4, 8, 64)), ((80, 1, 80), (80, 32, 80)), ((81, 1, 81), (81, 9, 81)),
                                     ((1, 1, 1), (1, 32, 300)), ((700, 1), (700, 16)), ((1, 24), (300, 24)), ((5, 1, 3), (5, 40, 3)),
                                     ((64, 1, 8, 1), (64, 3, 8, 16)), ((1,), (4100,))])
def test_broadcast_wide(dev, dtype, src, dst):
    x = np.random.default_rng(3).standard_normal(src).astype(dtype)
    got = dev.tensor(x, F32 if dtype == np.float32 else 0).broadcast_to(dst).numpy()
    assert np.array_equal(got, np.broadcast_to(x, dst))


@pytest.mark.parametrize("rows,n", [(5, 1), (7, 9), (6, 64), (5, 127), (6, 130), (9, 401), (3, 512), (4, 1024), (2, 1025)])
def test_softmax_one_wave_rows(dev, oracle, rows, n):
    x = S.normal_f16(25, f"x{n}", (rows, n), 0.0, 3.0)
    x[1] = -10000.0        # a fully masked row, and infinities among values
    if n > 8:
        x[0, n - 1], x[0, 3] = np.inf, -np.inf
    got = dev.tensor(x).softmax().numpy()
    assert ulp_diff(got, oracle.softmax(x)).max() <= 1


@pytest.mark.parametrize("D,H,Hkv", [(64, 8, 2), (80, 4, 4), (128, 8, 2)])
@pytest.mark.parametrize("J", [2049, 2177, 4000, 8191, 16500])
def test_one_row_over_many_key_chunks(dev, oracle, D, H, Hkv, J):
    """17 chunks of 128 keys and more: groups of chunks that end inside, at and
    past the last one, and more chunks than one batch of loads."""
    q, k, v = (S.normal_f16(29, f"{n}{D}{J}", (r, hh, D)) for n, r, hh in (("q", 1, H), ("k", J, Hkv), ("v", J, Hkv)))
    got = attention(dev.tensor(q), dev.tensor(k), dev.tensor(v), J - 1, 1 / np.sqrt(D)).numpy()
    assert_close(got, oracle.attention(q, k, v, J - 1, 1 / np.sqrt(D), True), what=f"one row, {J} keys of {D}")
    if J == 2177:   # keys without a finite score in most chunks, then in all: uniform over every key
        k[:, :, 0], q[:, :, 0] = np.inf, 1.0
        k[-1, :, 0] = 0.0
        got = attention(dev.tensor(q), dev.tensor(k), dev.tensor(v), J - 1, 1 / np.sqrt(D)).numpy()
        assert_close(got, np.repeat(v[-1:], H // Hkv, axis=1), what="one finite score")
        k[-1, :, 0] = np.inf
        got = attention(dev.tensor(q), dev.tensor(k), dev.tensor(v), J - 1, 1 / np.sqrt(D)).numpy()
        assert_close(got, oracle.attention(q, k, v, J - 1, 1 / np.sqrt(D), True), what="no finite score")
