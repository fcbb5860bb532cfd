"""The sizes at which the attention einsums take the matrix cores
(csrc/einsum_rule.hpp, compiled here as host code): measured pairs of both
kernels that are at least a tenth apart, at the two ends and the middle of the
ranges of rows, heads and keys."""
import ctypes as C
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "tensorlogic_amd", "csrc")


@pytest.fixture(scope="module", name="rule")
def einsum_rule(tmp_path_factory):
    d = tmp_path_factory.mktemp("einsum")
    (d / "r.cpp").write_text('#include "einsum_rule.hpp"\n'
                             'extern "C" int scores(int I, int H, int J) { return tlhip::scores_mfma_wins(I, H, J); }\n'
                             'extern "C" int context(int I, int H, int J, int D) { return tlhip::context_mfma_wins(I, H, J, D); }\n')
    subprocess.run(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", "-I", CSRC, str(d / "r.cpp"), "-o", str(d / "r.so")], check=True)
    return C.CDLL(str(d / "r.so"))


# (I, H, J, D, 8-lane us, matrix-core us)
@pytest.mark.parametrize("I,H,J,D,lanes,mfma", [
    (16, 2, 8000, 128, 55.4, 116.8), (128, 2, 1000, 128, 10.1, 19.9), (400, 2, 129, 128, 5.9, 8.8), (16, 32, 400, 128, 7.1, 11.7),
    (16, 32, 1000, 128, 12.1, 19.9), (65, 2, 33, 128, 4.1, 6.2), (64, 32, 400, 128, 16.3, 12.0), (400, 32, 16, 128, 26.7, 8.7),
    (17, 1, 129, 64, 3.2, 4.8), (128, 1, 1000, 64, 6.4, 8.1), (128, 4, 400, 64, 4.7, 6.2), (16, 32, 400, 64, 4.7, 6.0),
    (400, 4, 1000, 64, 16.0, 8.5), (64, 32, 400, 64, 9.3, 6.4), (400, 32, 400, 64, 40.3, 8.9),
    (16, 32, 129, 80, 4.3, 5.6), (48, 32, 400, 80, 13.0, 7.8), (17, 32, 8000, 80, 96.2, 59.1), (128, 32, 16, 80, 7.0, 4.5),
])
def test_context_takes_the_faster_kernel(rule, I, H, J, D, lanes, mfma):
    assert bool(rule.context(I, H, J, D)) == (mfma < lanes)


@pytest.mark.parametrize("I,H,J,lanes,mfma", [
    (16, 1, 33, 3.4, 3.6), (65, 4, 100, 3.3, 4.4), (65, 2, 129, 4.0, 5.3), (64, 2, 400, 4.0, 5.3),
    (128, 4, 400, 7.9, 4.2), (17, 32, 400, 8.4, 3.7), (16, 4, 2048, 5.9, 3.9), (400, 32, 400, 137.2, 10.5),
])
def test_scores_take_the_faster_kernel(rule, I, H, J, lanes, mfma):
    assert bool(rule.scores(I, H, J)) == (mfma < lanes)


def test_few_rows_or_keys_stay_on_the_lanes(rule):
    """A decode row, and fewer keys than half a tile, whatever the other sizes."""
    for few, many in ((1, 10**6), (15, 10**6)):
        assert not rule.scores(few, 32, many) and not rule.scores(many, 32, few)
        for D in (64, 80, 128):
            assert not rule.context(few, 32, many, D) and not rule.context(many, 32, few, D)
