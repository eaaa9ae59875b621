"""Caller-owned arrays with plans whose own data ends in their second buffer:
the result lands in the caller's array without a copy, by a pass list of its
own or by one pass writing the other buffer.  Lengths of two passes, of three
(2^25), the largest of two (2^24: another schedule for callers), batches, one
long axis beside short ones, both precisions; against the plan's own exec on
the same input (rel-L2 <= 1e-12, 1e-6 for complex64), with the plan's own
array untouched and its own exec right afterwards."""
import ctypes

import numpy as np
import pytest

import topefft
from conftest import rel_l2

pytestmark = pytest.mark.gpu


def run_ptr(fw, plan, ptr, direction):
    fw.lib.topePlanExecPtr(ctypes.byref(fw.f), plan.impl, ctypes.c_void_p(ptr), direction)
    fw.check("topePlanExecPtr")


@pytest.mark.parametrize("make", [
    ("1d", (1 << 13,)), ("1d", (1 << 16,)), ("1d", (1 << 23,)), ("1d", (1 << 24,)), ("1d", (1 << 25,)),
    ("1d", (8192, 6)), ("1d", (6, 8192)), ("1d", (8, 8192, 4)), ("1d", (8192, 4, 8192)), ("1d", (17,)),
    ("b64", (1 << 13, 5)), ("b64", (1 << 24, 2)), ("b32", (1 << 14, 9)), ("b32", (1 << 24, 1))],
    ids=lambda m: m[0] + "_" + "x".join(map(str, m[1])))
def test_caller_array_matches_own(make):
    import torch
    kind, dims = make
    n = int(np.prod(dims))
    f32 = kind == "b32"
    rng = np.random.default_rng(n % 1000)
    x = (rng.uniform(-1, 1, n) + 1j * rng.uniform(-1, 1, n)).astype(np.complex64 if f32 else np.complex128)
    tol = 1e-6 if f32 else 1e-12
    fw = topefft.Framework()
    if kind == "1d":
        p = topefft.Plan(fw, dims, x)
    else:
        p = topefft.BatchPlan(fw, dims[0], dims[1], x, topefft.PREC_F32 if f32 else topefft.PREC_F64)
    t = torch.from_numpy(x.copy()).cuda()
    torch.cuda.synchronize()
    run_ptr(fw, p, t.data_ptr(), topefft.FORWARD)
    fw.synchronize()
    got = t.cpu().numpy()
    own = p.exec(topefft.FORWARD)  # the plan's array still holds x
    run_ptr(fw, p, t.data_ptr(), topefft.INVERSE)
    fw.synchronize()
    back = t.cpu().numpy()
    own_back = p.exec(topefft.INVERSE)
    p.destroy()
    fw.destroy()
    assert rel_l2(got, own) < tol
    assert rel_l2(back, x) < tol
    assert rel_l2(own_back, x) < tol
