"""The dtype and shape a Tensor keeps are those the library has for its handle."""
import numpy as np
import pytest

import tensorlogic_amd as tl

pytestmark = pytest.mark.gpu


def _asked(t):
    probe = tl.Tensor(t.dev, t.h)
    info = probe._info()
    probe.h = None  # the handle stays t's to free
    return info


@pytest.mark.parametrize("dtype", [tl.F16, tl.F32, tl.I32])
def test_kept_metadata_is_the_library_s(dev, dtype):
    made = [dev.empty(np.array([3, 5]), dtype), dev.empty([0, 4], dtype), dev.tensor(np.float32(2.0), dtype),
            dev.tensor(np.ones((2, 3, 4)), dtype)]
    made.append(made[-1].reshape([np.int64(6), 4]))
    made.append(made[-1].slice_last() if dtype != tl.I32 else made[-1])
    if dtype != tl.I32:
        cache = tl.KVCache(dev, 1, 8, 1, 64, dtype)
        kv = dev.empty((2, 1, 64), dtype)
        cache.set(0, kv, kv)
        made += [cache.get_k(0), made[3].softmax(), made[3].reshape((6, 4)).linear(made[3].reshape((6, 4)))]
    for t in made:
        assert (t.dtype, t.shape) == _asked(t)


def test_a_refused_reshape_leaves_the_tensor(dev):
    t = dev.empty((2, 6))
    with pytest.raises(tl.TLHipError):
        t.reshape((5, 2))
    assert t.shape == (2, 6)
