"""broadcast_to's dim merging, kernel choice and index arithmetic
(csrc/broadcast_plan.hpp, compiled here as host code) against the coordinates
the target shape gives, over shapes of every form and past 2^32 elements,
where a count held in 32 bits would wrap."""
import ctypes as C
import os
import random
import subprocess

import numpy as np
import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "tensorlogic_amd", "csrc")
DRIVER = """
#include "broadcast_plan.hpp"
using namespace tlhip;
// target shape s[n] and input strides t[n] -> is the wide kernel taken, and
// for each of `count` target elements g (rounded down to a vector) the input
// element by the kernel's arithmetic and by the one-per-thread kernel's
extern "C" int run(int n, const int64_t* s, const int64_t* t, int V, int count, const int64_t* g, int64_t* wide, int64_t* one) {
    BcastDims full;
    full.nd = n;
    int64_t total = 1;
    for (int i = 0; i < n; i++) total *= full.shape[i] = s[i], full.xstride[i] = t[i];
    const BcastDims b = bcast_merge(full);
    const bool ok = bcast_wide_ok(b, total, V);
    for (int i = 0; i < count; i++) {
        one[i] = bcast_src(b, g[i]);
        if (ok) wide[i] = (int64_t)bcast_wide_src(b, (uint32_t)(g[i] / V), V) + (b.xstride[b.nd - 1] ? g[i] % V : 0);
    }
    return ok;
}
"""


@pytest.fixture(scope="module")
def run(tmp_path_factory):
    d = tmp_path_factory.mktemp("bcast")
    (d / "driver.cpp").write_text(DRIVER)
    subprocess.run(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", "-I", CSRC, str(d / "driver.cpp"), "-o", str(d / "driver.so")],
                   check=True)
    f = C.CDLL(str(d / "driver.so")).run

    def call(src, dst, V, g):
        """(wide kernel taken, its input elements, the general kernel's)"""
        src = (1,) * (len(dst) - len(src)) + tuple(src)
        strides, st = [0] * len(dst), 1
        for i in reversed(range(len(dst))):
            strides[i] = 0 if src[i] == 1 else st
            st *= src[i]
        a = [np.ascontiguousarray(v, np.int64) for v in (dst, strides, g)]
        wide, one = np.full(len(g), -1, np.int64), np.full(len(g), -1, np.int64)
        p = [C.c_void_p(v.ctypes.data) for v in (*a, wide, one)]
        ok = f(len(dst), p[0], p[1], V, len(g), p[2], p[3], p[4])
        return bool(ok), wide, one, strides

    return call


def _want(dst, strides, g):
    """Input elements by the target's coordinates, in Python integers."""
    out = []
    for x in map(int, g):
        e = 0
        for n, st in zip(reversed(dst), reversed(strides)):
            e += x % n * st
            x //= n
        out.append(e)
    return np.array(out, np.int64)


def _check(run, src, dst, V, g):
    ok, wide, one, strides = run(src, dst, V, g)
    want = _want(dst, strides, g)
    assert np.array_equal(one, want), (src, dst)
    if ok:
        assert np.array_equal(wide, want), (src, dst, V)
    return ok


@pytest.mark.parametrize("V", [8, 4])
@pytest.mark.parametrize("src,dst", [
    ((65536, 65544), (65536, 65544)),            # merged to one run past 2^32 elements
    ((65536, 65544), (2, 65536, 65544)),
    ((65536, 65536), (65536, 65536)),            # exactly 2^32
    ((1,), (65536, 65536)),                      # a scalar repeated
    ((3, 1, 1), (3, 65536, 32768)),              # a repeated run below 2^32, the whole beyond
    ((1, 65536, 65544), (1, 65536, 65544)),
    ((40000, 1, 24), (40000, 9000, 24)),
])
def test_past_32_bits(run, V, src, dst):
    total = int(np.prod(dst, dtype=object))
    rng = random.Random(V)
    edges = [0, 1, V, 2**19, 2**31, 2**32 - 1, 2**32, 2**32 + 8 * 4099 + 3, total - 1]
    g = sorted({x for x in edges + [rng.randrange(total) for _ in range(300)] if x < total})
    took = _check(run, src, dst, V, g)
    assert took == (total // V <= 0xffffff00)


def test_all_forms(run):
    """Random ranks, sizes, repeated dims and vector widths: both kernels."""
    rng, taken = random.Random(0), 0
    for _ in range(400):
        n = rng.randrange(1, 7)
        dst = tuple(rng.choice([1, 2, 3, 4, 5, 7, 8, 16, 24, 33]) for _ in range(n))
        src = tuple(1 if rng.random() < 0.4 else d for d in dst)[rng.randrange(n):]
        total = int(np.prod(dst))
        g = range(total) if total <= 4096 else [rng.randrange(total) for _ in range(500)] + [total - 1]
        taken += _check(run, src, dst, rng.choice([4, 8]), list(g))
    assert taken > 20
