"""Contiguous rows of up to 15 points (the lengths of one mixed radix) at the edges
of their 64-row blocks, forward and back, against numpy.  FP64 bound 1e-14: a row is
one butterfly of at most two factors, a few rounding errors of 1.1e-16 each;
complex64 2e-6 by the ratio of the types' rounding errors."""
import numpy as np
import pytest

import topefft
from conftest import rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec,bound", [("f64", 1e-14), ("f32", 2e-6)])
@pytest.mark.parametrize("n", [3, 5, 6, 7, 9, 10, 12, 14, 15])
def test_mixed_rows(n, prec, bound):
    for count in (1, 63, 64, 65, 1000):
        rng = np.random.default_rng(1000 * n + count)
        x = rng.standard_normal((count, n)) + 1j * rng.standard_normal((count, n))
        if prec == "f32":
            x = x.astype(np.complex64)
        fw = topefft.Framework()
        p = topefft.BatchPlan(fw, n, count, x, topefft.PREC_F64 if prec == "f64" else topefft.PREC_F32)
        assert p.pass_names() == ["mixed_radix_" + prec]
        X = p.exec(topefft.FORWARD).reshape(count, n)
        back = p.exec(topefft.INVERSE).reshape(count, n)
        p.destroy()
        fw.destroy()
        want = np.fft.fft(x.astype(complex), axis=1)
        for k in {0, count // 2, count - 1}:  # every row of its own: a stray one would vanish in the whole
            assert rel_l2(X[k], want[k]) < bound, (n, count, k)
        assert rel_l2(X, want) < bound and rel_l2(back, x) < bound, (n, count)


def test_mixed_rows_in_planes():
    """Rows of a 3D array (one packed run) and an axis of length 12 along contiguous
    memory in planes of one column."""
    for dims in ((15, 20, 9), (1, 12, 70)):
        rng = np.random.default_rng(sum(dims))
        x = rng.standard_normal(dims[::-1]) + 1j * rng.standard_normal(dims[::-1])
        fw = topefft.Framework()
        p = topefft.Plan(fw, dims, x)
        X = p.exec(topefft.FORWARD).reshape(x.shape)
        back = p.exec(topefft.INVERSE).reshape(x.shape)
        p.destroy()
        fw.destroy()
        assert rel_l2(X, np.fft.fftn(x)) < 1e-13 and rel_l2(back, x) < 1e-13, dims
