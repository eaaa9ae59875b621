"""Real rows of 7-smooth length in one pass (transform and half spectrum): odd
and even half lengths, the shortest and longest rows, one to five radices'
tiles, row counts that leave the last tile short, both precisions, packed and
unpacked DC and Nyquist columns, against numpy's FP64 rfftn (complex128 rel-L2
<= 1e-12, complex64 <= 1e-6); lengths outside the range keep the step on its
own."""
import numpy as np
import pytest

import topefft
from conftest import rel_l2

pytestmark = pytest.mark.gpu

HALF = [18, 20, 21, 25, 27, 35, 49, 60, 75, 105, 135, 189, 240, 343, 500, 675, 1000, 1029, 1500, 2187, 2401, 3000, 3584,
        4050]


def seeded(dims, dtype):
    n = int(np.prod(dims))
    return np.random.default_rng(n).uniform(-1, 1, n).astype(dtype)


@pytest.mark.parametrize("m", HALF)
@pytest.mark.parametrize("prec", ["f64", "f32"])
def test_real_mixed_rows(m, prec):
    dtype, kw, tol = (np.float64, {}, 1e-12) if prec == "f64" else (np.float32, {"precision": topefft.PREC_F32}, 1e-6)
    for dims in [(2 * m,), (2 * m, 3), (2 * m, 70), (2 * m, 5, 6)]:
        x = seeded(dims, dtype)
        fw = topefft.Framework()
        p = topefft.RealPlan(fw, dims, x, **kw)
        names = p.pass_names()
        X = p.forward()
        back = p.inverse()
        p.destroy()
        fw.destroy()
        assert names[0] == "real_rows_mixed" and "real_half_spectrum" not in names, names
        want = np.fft.rfftn(x.astype(np.float64).reshape(dims[::-1])).reshape(-1)
        assert rel_l2(X.astype(np.complex128), want) < tol, dims
        assert rel_l2(back.astype(np.float64), x.astype(np.float64)) < tol, dims


@pytest.mark.parametrize("nx", [10, 30, 32, 8400])
def test_step_on_its_own(nx):
    x = seeded((nx, 4), np.float64)
    fw = topefft.Framework()
    p = topefft.RealPlan(fw, (nx, 4), x)
    names = p.pass_names()
    X = p.forward()
    back = p.inverse()
    p.destroy()
    fw.destroy()
    assert "real_half_spectrum" in names, names
    assert rel_l2(X, np.fft.rfftn(x.reshape(4, nx)).reshape(-1)) < 1e-12
    assert rel_l2(back, x) < 1e-12
