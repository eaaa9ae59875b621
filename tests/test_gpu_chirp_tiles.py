"""Tiles of the one-launch Bluestein pass (lines with a prime factor above 7 and at
most 2048 points), forward and back, against numpy.  Bound 1e-12, the FP64 parity bound of
every transform here."""
import numpy as np
import pytest

import topefft
from conftest import rel_l2

pytestmark = pytest.mark.gpu


def _check(dims):
    rng = np.random.default_rng(sum(dims))
    x = rng.standard_normal(dims[::-1]) + 1j * rng.standard_normal(dims[::-1])
    fw = topefft.Framework()
    p = topefft.Plan(fw, dims, x)
    names = p.pass_names()
    X = p.exec(topefft.FORWARD).reshape(x.shape)
    back = p.exec(topefft.INVERSE).reshape(x.shape)
    p.destroy()
    fw.destroy()
    want = np.fft.fftn(x)
    assert "chirp_pre" in names, names
    assert rel_l2(X, want) < 1e-12 and rel_l2(back, x) < 1e-12, dims
    last = (-1,) * x.ndim  # the last element's tile is the partial one
    assert abs(X[last] - want[last]) < 1e-12 * np.linalg.norm(x) * np.sqrt(x.size), dims


@pytest.mark.parametrize("dims", [(1, 11, 70), (1, 13, 32), (1, 127, 33), (1, 509, 5), (1, 2039, 3), (1, 11, 1)],
                         ids=lambda d: "x".join(map(str, d)))
def test_planes_of_one_column(dims):
    """The middle axis lies along contiguous memory; the planes' lines share blocks of
    32 (11 and 13 points), 8 (127), 2 (509) and 1 (2039)."""
    _check(dims)


# 16-line tiles for 32 < 2n - 1 <= 256 points of convolution, 8-line ones up to
# 512, from 512 tiles on: 515 tiles, the last one half full; one width above:
# full tiles and a partial one of 4 lines (509 points) or 2 (1021, 2039)
@pytest.mark.parametrize("dims", [(8232, 31), (8232, 61), (8232, 127), (4116, 251), (35, 509), (2058, 509),
                                  (35, 1021), (1029, 1021), (35, 2039), (1029, 2039), (12, 61, 25)],
                         ids=lambda d: "x".join(map(str, d)))
def test_column_tiles(dims):
    _check(dims)
