"""Synchronous execs whose result fits the pinned staging buffer (256 KiB): the
sizes around that limit, frameworks that come and go (the buffer is given back
with the last and taken again), and several threads with a framework each, of
which one at a time holds the buffer and the others download by themselves."""
import threading

import numpy as np
import pytest

import topefft
from conftest import rel_l2

pytestmark = pytest.mark.gpu


def seeded(n, salt):
    rng = np.random.default_rng(salt)
    return rng.uniform(-1, 1, n) + 1j * rng.uniform(-1, 1, n)


@pytest.mark.parametrize("n", [2, 3, 100, 1024, 16384, 32768])
def test_staged_exec(n):
    for rep in range(2):  # a fresh framework each time
        x = seeded(n, n + rep)
        fw = topefft.Framework()
        p = topefft.Plan(fw, (n,), x)
        k0, m0 = p.t.totalKernel, p.t.totalMemory
        got = p.exec(topefft.FORWARD)
        back = p.exec(topefft.INVERSE)
        assert p.t.totalKernel > k0 and p.t.totalMemory > m0
        assert fw.lib.profileThis(fw.f.event) > 0
        p.destroy()
        fw.destroy()
        assert rel_l2(got, np.fft.fft(x)) < 1e-12
        assert rel_l2(back, x) < 1e-12


def test_staged_exec_complex64_batch():
    # 3 x 5 complex64 values: an odd number of 8-byte elements
    x = seeded(15, 4).astype(np.complex64)
    fw = topefft.Framework()
    p = topefft.BatchPlan(fw, 5, 3, x, topefft.PREC_F32)
    got = p.exec(topefft.FORWARD)
    p.destroy()
    fw.destroy()
    assert rel_l2(got, np.fft.fft(x.reshape(3, 5).astype(np.complex128), axis=1).reshape(-1)) < 1e-6


def test_staged_exec_threads():
    bad = []

    def work(k):
        x = seeded(512 << k, 60 + k)
        want = np.fft.fft(x)
        fw = topefft.Framework()
        p = topefft.Plan(fw, (x.size,), x)
        for _ in range(40):
            if rel_l2(p.exec(topefft.FORWARD), want) > 1e-12 or rel_l2(p.exec(topefft.INVERSE), x) > 1e-11:
                bad.append(k)
        p.destroy()
        fw.destroy()

    ts = [threading.Thread(target=work, args=(k,)) for k in range(4)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not bad, bad
