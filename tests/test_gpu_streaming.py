"""Plans of 512 MiB and more, whose passes stream through L2: rows of every
streamed length in one pass, both precisions, with a row count that leaves part
of a tile, through a caller's array (sampled rows against numpy, all rows by the
round trip); a packed uneven batch of that size; and the transforms whose
first or last pass moves the data (2^24, 2^25, a batch of four-step rows)
against numpy.  complex128 rel-L2 <= 1e-12, complex64 <= 1e-6."""
import ctypes

import numpy as np
import pytest

import topefft
from conftest import rel_l2

pytestmark = pytest.mark.gpu


def run_ptr(fw, plan, ptr, direction):
    fw.lib.topePlanExecPtr(ctypes.byref(fw.f), plan.impl, ctypes.c_void_p(ptr), direction)
    fw.check("topePlanExecPtr")


@pytest.mark.parametrize("n", [64, 128, 256, 512, 1024, 2048, 4096, 8192])
@pytest.mark.parametrize("prec", ["f64", "f32"])
def test_streamed_rows(n, prec):
    import torch
    f32 = prec == "f32"
    tol = 1e-6 if f32 else 1e-12
    count = (1 << (26 if f32 else 25)) // n + 3
    dt = torch.complex64 if f32 else torch.complex128
    g = torch.Generator(device="cuda")
    g.manual_seed(n)
    x = torch.randn(count * n, dtype=dt, device="cuda", generator=g)
    t = x.clone()
    fw = topefft.Framework()
    p = topefft.BatchPlan(fw, n, count, np.zeros(count * n, np.complex64 if f32 else np.complex128),
                          topefft.PREC_F32 if f32 else topefft.PREC_F64)
    torch.cuda.synchronize()
    run_ptr(fw, p, t.data_ptr(), topefft.FORWARD)
    fw.synchronize()
    rows = np.unique(np.concatenate([[0, 1, count - 2, count - 1], np.random.default_rng(n).integers(0, count, 60)]))
    idx = torch.from_numpy(rows).cuda()
    got = t.view(count, n)[idx].cpu().numpy()
    want = np.fft.fft(x.view(count, n)[idx].cpu().numpy().astype(np.complex128), axis=1)
    run_ptr(fw, p, t.data_ptr(), topefft.INVERSE)
    fw.synchronize()
    off = float((t - x).abs().square().sum().sqrt() / x.abs().square().sum().sqrt())
    p.destroy()
    fw.destroy()
    assert rel_l2(got, want) < tol
    assert off < tol


def test_streamed_uneven():
    rng = np.random.default_rng(5)
    sizes = (1 << rng.integers(4, 15, 12000)).astype(np.int32)
    assert sizes.sum() * 16 >= 512 << 20
    x = rng.uniform(-1, 1, int(sizes.sum())) + 1j * rng.uniform(-1, 1, int(sizes.sum()))
    fw = topefft.Framework()
    p = topefft.ManyPlan(fw, sizes, x)
    offs = p.offsets()
    got = p.exec(topefft.FORWARD)
    back = p.exec(topefft.INVERSE)
    p.destroy()
    fw.destroy()
    for i in list(range(0, sizes.size, 37)) + [sizes.size - 1]:
        s = slice(int(offs[i]), int(offs[i]) + int(sizes[i]))
        assert rel_l2(got[s], np.fft.fft(x[s])) < 1e-12, (i, sizes[i])
    assert rel_l2(back, x) < 1e-12


@pytest.mark.parametrize("n,count", [(1 << 24, 1), (1 << 25, 1), (1 << 14, 2049)])
def test_streamed_moving_passes(n, count):
    import torch
    rng = np.random.default_rng(count)
    x = (rng.uniform(-1, 1, n * count) + 1j * rng.uniform(-1, 1, n * count))
    want = np.fft.fft(x.reshape(count, n), axis=1).reshape(-1)
    fw = topefft.Framework()
    p = topefft.BatchPlan(fw, n, count, x) if count > 1 else topefft.Plan(fw, (n,), x)
    t = torch.from_numpy(x.copy()).cuda()
    torch.cuda.synchronize()
    run_ptr(fw, p, t.data_ptr(), topefft.FORWARD)
    fw.synchronize()
    assert rel_l2(t.cpu().numpy(), want) < 1e-12
    run_ptr(fw, p, t.data_ptr(), topefft.INVERSE)
    fw.synchronize()
    assert rel_l2(t.cpu().numpy(), x) < 1e-12
    assert rel_l2(p.exec(topefft.FORWARD), want) < 1e-12
    assert rel_l2(p.exec(topefft.INVERSE), x) < 1e-12
    p.destroy()
    fw.destroy()
