"""Column passes of 7-smooth length around 2048 elements, up to which one block takes
every line, forward and back, against numpy; bounds 1e-12 and 1e-6, the parity bounds of
every FP64 and complex64 transform here."""
import numpy as np
import pytest

import topefft
from conftest import rel_l2

pytestmark = pytest.mark.gpu


# 2034, 2052, 2040, 2048 + 8, 2000 elements a column pass; one and two lines; planes whose
# lines carry over; 64 lines and more than a tile holds
@pytest.mark.parametrize("prec,bound", [("f64", 1e-12), ("f32", 1e-6)])
@pytest.mark.parametrize("dims", [(113, 18), (114, 18), (17, 120), (257, 8, 3), (2, 1000), (1, 2000), (5, 24, 7),
                                  (64, 28), (64, 30), (66, 30), (3, 60, 10), (7, 21, 2), (16, 20)],
                         ids=lambda d: "x".join(map(str, d)))
def test_small_column_passes(dims, prec, bound):
    if prec == "f32":  # complex64 plans take 7-smooth axes only
        dims = {113: (112, 18), 114: (120, 18), 17: (16, 125), 257: (256, 8, 3), 66: (70, 30)}.get(dims[0], dims)
    rng = np.random.default_rng(sum(dims))
    x = rng.standard_normal(dims[::-1]) + 1j * rng.standard_normal(dims[::-1])
    fw = topefft.Framework()
    if prec == "f32":
        x = x.astype(np.complex64)
        p = topefft.Plan(fw, dims, x, precision=topefft.PREC_F32)
    else:
        p = topefft.Plan(fw, dims, x)
    assert "mixed_radix_" + prec in p.pass_names()
    X = p.exec(topefft.FORWARD).reshape(x.shape)
    back = p.exec(topefft.INVERSE).reshape(x.shape)
    p.destroy()
    fw.destroy()
    assert rel_l2(X, np.fft.fftn(x.astype(complex))) < bound and rel_l2(back, x) < bound
