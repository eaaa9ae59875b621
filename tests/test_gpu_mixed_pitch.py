"""Strided mixed-radix lines whose widest tile fits the LDS only with the lines
packed: complex128 lines of 2049 to 2560 points in tiles of four and of more
than 3413 in tiles of two, with and without a remainder in the last tile,
beside the spread tiles of the lengths around them, against numpy's FP64
transform (rel-L2 <= 1e-12)."""
import numpy as np
import pytest

import topefft
from conftest import rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims", [(1000, 2100), (1029, 2187), (1030, 2560), (625, 2592), (625, 3375), (625, 3456),
                                  (1000, 3600), (625, 4050)], ids=lambda d: "x".join(map(str, d)))
def test_packed_tiles(dims):
    n = dims[0] * dims[1]
    rng = np.random.default_rng(n)
    x = rng.uniform(-1, 1, n) + 1j * rng.uniform(-1, 1, n)
    fw = topefft.Framework()
    p = topefft.Plan(fw, dims, x)
    assert "mixed_radix_f64" in p.pass_names()
    fwd = p.exec(topefft.FORWARD)
    back = p.exec(topefft.INVERSE)
    p.destroy()
    fw.destroy()
    assert rel_l2(fwd, np.fft.fftn(x.reshape(dims[::-1])).reshape(-1)) < 1e-12
    assert rel_l2(back, x) < 1e-12
