"""Fused power-of-two real rows at every length, with row counts that fill no
block, one block and a remainder, both precisions, against numpy's FP64 rfftn
(complex128 rel-L2 <= 1e-12, complex64 <= 1e-6)."""
import numpy as np
import pytest

import topefft
from conftest import rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx", [128, 256, 512, 1024, 2048, 4096, 8192])
@pytest.mark.parametrize("prec", ["f64", "f32"])
def test_real_rows(nx, prec):
    dtype, kw, tol = (np.float64, {}, 1e-12) if prec == "f64" else (np.float32, {"precision": topefft.PREC_F32}, 1e-6)
    for dims in [(nx,), (nx, 2), (nx, 8), (nx, 15), (nx, 3, 7)]:
        n = int(np.prod(dims))
        x = np.random.default_rng(n).uniform(-1, 1, n).astype(dtype)
        fw = topefft.Framework()
        p = topefft.RealPlan(fw, dims, x, **kw)
        names = p.pass_names()
        X = p.forward()
        back = p.inverse()
        p.destroy()
        fw.destroy()
        assert names[0] == "real_rows_fused", names
        want = np.fft.rfftn(x.astype(np.float64).reshape(dims[::-1])).reshape(-1)
        assert rel_l2(X.astype(np.complex128), want) < tol, dims
        assert rel_l2(back.astype(np.float64), x.astype(np.float64)) < tol, dims
