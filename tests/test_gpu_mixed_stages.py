"""The mixed-radix pass at the sizes where its schedule changes: every radix
alone (n <= 16, one thread per line), lists of two to five radices, block
sizes of 256, 512 and 1024 threads, tiles of strided lines that end in a
remainder or run over the end of a plane, both precisions and directions,
against the FP64 oracle (complex128 rel-L2 <= 1e-12, complex64 <= 1e-6)."""
import numpy as np
import pytest

import topefft
from conftest import rel_l2

pytestmark = pytest.mark.gpu

LENGTHS = [3, 5, 6, 7, 9, 10, 12, 14, 15, 18, 20, 21, 24, 30, 36, 45, 48, 63, 75, 84, 98, 125, 126, 144, 196, 210, 225,
           240, 343, 375, 480, 500, 640, 686, 729, 960, 1029, 1280, 1500, 2187, 2401, 2560, 2592, 3125, 3360, 3584,
           3840, 4050, 4032]


def seeded(dims, salt):
    n = int(np.prod(dims))
    rng = np.random.default_rng(salt + n)
    return rng.uniform(-1, 1, n) + 1j * rng.uniform(-1, 1, n)


@pytest.mark.parametrize("n", LENGTHS)
@pytest.mark.parametrize("prec", ["f64", "f32"])
def test_mixed_stages(oracle, n, prec):
    kw, tol = ({}, 1e-12) if prec == "f64" else ({"precision": topefft.PREC_F32}, 1e-6)
    for dims in [(n, 3), (5, n), (3, n, 2)]:
        x = seeded(dims, 3)
        fw = topefft.Framework()
        p = topefft.Plan(fw, dims, x, **kw)
        assert "mixed_radix_" + prec in p.pass_names()
        fwd = p.exec(topefft.FORWARD)
        back = p.exec(topefft.INVERSE)
        inv = p.exec(topefft.INVERSE)
        p.destroy()
        fw.destroy()
        x = x.astype(np.complex64).astype(np.complex128) if prec == "f32" else x
        assert rel_l2(fwd, oracle.dft(x, dims, topefft.FORWARD)) < tol, dims
        assert rel_l2(back, x) < tol, dims
        assert rel_l2(inv, oracle.dft(x, dims, topefft.INVERSE)) < tol, dims


@pytest.mark.parametrize("dims", [(1200, 700), (100, 100, 100), (45, 50, 84), (3000, 130), (130, 3000), (515, 96)],
                         ids=lambda d: "x".join(map(str, d)))
def test_mixed_full_tiles(dims):
    # enough lines for full tiles in every block, with remainders (515 = 5 x 103
    # puts strided 96-point lines beside a Bluestein axis)
    x = seeded(dims, 8)
    want = np.fft.fftn(x.reshape(dims[::-1])).reshape(-1)
    fw = topefft.Framework()
    p = topefft.Plan(fw, dims, x)
    fwd = p.exec(topefft.FORWARD)
    back = p.exec(topefft.INVERSE)
    p.destroy()
    fw.destroy()
    assert rel_l2(fwd, want) < 1e-12
    assert rel_l2(back, x) < 1e-12
