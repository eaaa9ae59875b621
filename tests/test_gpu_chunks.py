"""3D arrays of at least 512 MiB, whose X and Y passes run in turn over chunks of
planes: the transform of a product field against the product of its factors'
spectra (rel-L2 <= 1e-12 for complex128, <= 1e-6 for complex64), the round trip, and
the same through a caller's array and for real input.  The plane counts give
two, four and an odd number of chunks."""
import numpy as np
import pytest

import topefft
from conftest import rel_l2

pytestmark = pytest.mark.gpu


def separable(dims, rng):
    """A product field a(x) b(y) c(z) and its spectrum's factors."""
    f = [rng.uniform(-1, 1, n) + 1j * rng.uniform(-1, 1, n) for n in dims]
    x = np.einsum("k,j,i->kji", f[2], f[1], f[0]).reshape(-1)
    return x, [np.fft.fft(v) for v in f]


# 512 x 512 x 128 complex128: two chunks of 64 planes; 300 x 300 x 375
# (mixed radix): three of 125; complex64 512 x 512 x 256 on the vector ALUs and
# on the matrix cores
@pytest.mark.parametrize("dims,prec,mode", [((512, 512, 128), None, None), ((300, 300, 375), None, None),
                                            ((512, 512, 256), topefft.PREC_F32, topefft.MODE_VALU),
                                            ((512, 512, 256), topefft.PREC_F32, topefft.MODE_MFMA_FP16X3)],
                         ids=["f64", "mixed", "f32", "mfma"])
def test_chunked_planes(dims, prec, mode):
    rng = np.random.default_rng(7)
    x, f = separable(dims, rng)
    tol = 1e-12 if prec is None else 1e-6
    want = np.einsum("k,j,i->kji", f[2], f[1], f[0]).reshape(-1)
    fw = topefft.Framework()
    p = topefft.Plan(fw, dims, x, precision=prec, mode=mode)
    assert p.pass_count() == 3
    got = p.exec(topefft.FORWARD)
    assert rel_l2(got, want) < tol
    back = p.exec(topefft.INVERSE)
    assert rel_l2(back, x) < tol
    p.destroy()
    fw.destroy()


def test_chunked_real():
    # spectrum of 512 x 512 x 256: four chunks of 64 planes (132 MiB)
    dims = (512, 512, 256)
    rng = np.random.default_rng(11)
    f = [rng.uniform(-1, 1, n) for n in dims]
    x = np.einsum("k,j,i->kji", f[2], f[1], f[0]).reshape(-1)
    X = [np.fft.rfft(f[0]), np.fft.fft(f[1]), np.fft.fft(f[2])]
    want = np.einsum("k,j,i->kji", X[2], X[1], X[0]).reshape(-1)
    fw = topefft.Framework()
    p = topefft.RealPlan(fw, dims, x)
    got = p.forward()
    assert rel_l2(got, want) < 1e-12
    assert rel_l2(p.inverse(), x) < 1e-12
    p.destroy()
    fw.destroy()


def test_chunked_caller_array():
    import torch
    dims = (512, 512, 256)
    rng = np.random.default_rng(13)
    x, f = separable(dims, rng)
    d = torch.from_numpy(x.astype(np.complex64)).cuda()
    fw = topefft.Framework()
    p = topefft.Plan(fw, dims, np.zeros(d.numel(), np.complex64), precision=topefft.PREC_F32)
    torch.cuda.synchronize()
    p.exec_ptr(d.data_ptr(), topefft.FORWARD)
    fw.synchronize()
    got = d.cpu().numpy()
    want = np.einsum("k,j,i->kji", f[2], f[1], f[0]).reshape(-1)
    assert rel_l2(got, want) < 1e-6
    p.destroy()
    fw.destroy()
