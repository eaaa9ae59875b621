"""Complex64 columns whose threads hold 32 elements: lengths of every radix list
that takes them, with 1024 lines and more and remainders in the last tile, beside
fewer lines and lengths that stay at 16, against numpy's FP64 transform (rel-L2 <=
1e-6, complex64)."""
import numpy as np
import pytest

import topefft
from conftest import rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims", [(1024, 2430), (1029, 2646), (1050, 3087), (1024, 3240), (1029, 3402), (1029, 3500),
                                  (1029, 3645), (1024, 3750), (1134, 3920), (1024, 4032), (1029, 4050), (1008, 4000),
                                  (1024, 3600), (200, 4000)], ids=lambda d: "x".join(map(str, d)))
def test_wide_columns(dims):
    n = dims[0] * dims[1]
    rng = np.random.default_rng(n)
    x = rng.uniform(-1, 1, n) + 1j * rng.uniform(-1, 1, n)
    x = x.astype(np.complex64).astype(np.complex128)
    fw = topefft.Framework()
    p = topefft.Plan(fw, dims, x, precision=topefft.PREC_F32)
    assert "mixed_radix_f32" in p.pass_names()
    fwd = p.exec(topefft.FORWARD)
    back = p.exec(topefft.INVERSE)
    p.destroy()
    fw.destroy()
    assert rel_l2(fwd, np.fft.fftn(x.reshape(dims[::-1])).reshape(-1)) < 1e-6
    assert rel_l2(back, x) < 1e-6
