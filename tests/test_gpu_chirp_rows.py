"""Contiguous lines with a prime factor above 7 and more than 2048 points: every
split of the padded row (8192 to 2^24 points), the shortest and longest length of
a row, one and several lines, against numpy's FP64 transform (rel-L2 <= 1e-12)."""
import numpy as np
import pytest

import topefft
from conftest import rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims", [(2049,), (4093,), (4097,), (8191,), (8195,), (16381,), (32749,), (65521,), (131071,),
                                  (262139,), (524287,), (1048573,), (2097143,), (4194301,), (8388593,), (2053, 3),
                                  (4092, 33), (10007, 4), (2057, 3, 2), (66011, 5), (33, 4099)],
                         ids=lambda d: "x".join(map(str, d)))
def test_chirp_rows(dims):
    n = int(np.prod(dims))
    rng = np.random.default_rng(n)
    x = rng.uniform(-1, 1, n) + 1j * rng.uniform(-1, 1, n)
    a = x.reshape(dims[::-1])
    fw = topefft.Framework()
    p = topefft.Plan(fw, dims, x)
    names = p.pass_names()
    fwd = p.exec(topefft.FORWARD)
    back = p.exec(topefft.INVERSE)
    inv = p.exec(topefft.INVERSE)
    p.destroy()
    fw.destroy()
    assert names[0] == "chirp_pre" and "chirp_mul" in names, names
    if dims[0] > 2048:
        assert names[:3] == ["chirp_pre", "chirp_mul", "chirp_post"], names
    assert rel_l2(fwd, np.fft.fftn(a).reshape(-1)) < 1e-12
    assert rel_l2(back, x) < 1e-12
    assert rel_l2(inv, np.fft.ifftn(a).reshape(-1)) < 1e-12
