"""Lengths with a prime factor above 7 and at most 2048, whose whole chirp-z
convolution runs inside a workgroup: the smallest and largest length of each
convolution size M = 32 .. 4096, as contiguous rows, as strided columns and as
the middle axis of a volume, with line counts that leave partial tiles, in
both directions, against the FP64 oracle (rel-L2 <= 1e-12)."""
import numpy as np
import pytest

import topefft
from conftest import rel_l2

pytestmark = pytest.mark.gpu

# M = 32: 11, 13; 64: 17, 31; ... 4096: 1031, 2047
LENGTHS = [11, 13, 17, 31, 33, 62, 67, 127, 130, 254, 257, 509, 513, 1023, 1031, 2047]


def seeded(dims, salt):
    rng = np.random.default_rng(salt + int(np.prod(dims)))
    n = int(np.prod(dims))
    return rng.uniform(-1, 1, n) + 1j * rng.uniform(-1, 1, n)


@pytest.mark.parametrize("n", LENGTHS)
def test_chirp_lines(oracle, n):
    # rows, columns (7 and 35 lines: part of a tile, a full one and a
    # remainder), the middle axis of a volume
    for dims in [(n, 3), (7, n), (35, n), (3, n, 2)] if n < 1000 else [(n, 3), (7, n), (3, n, 2)]:
        x = seeded(dims, 5)
        fw = topefft.Framework()
        p = topefft.Plan(fw, dims, x)
        names = p.pass_names()
        fwd = p.exec(topefft.FORWARD)
        back = p.exec(topefft.INVERSE)
        again = p.exec(topefft.INVERSE)
        p.destroy()
        fw.destroy()
        assert names.count("chirp_pre") == 1 and "chirp_mul" not in names, names
        assert rel_l2(fwd, oracle.dft(x, dims, topefft.FORWARD)) < 1e-12, dims
        assert rel_l2(back, x) < 1e-12, dims
        assert rel_l2(again, oracle.dft(x, dims, topefft.INVERSE)) < 1e-12, dims


def test_chirp_lines_wide_tiles(oracle):
    # enough columns for the wide tiles (512 blocks or more) with a remainder
    for dims in [(2049, 600), (4100, 11, 2), (8194, 127)]:
        x = seeded(dims, 9)
        fw = topefft.Framework()
        p = topefft.Plan(fw, dims, x)
        got = p.exec(topefft.FORWARD)
        back = p.exec(topefft.INVERSE)
        p.destroy()
        fw.destroy()
        assert rel_l2(got, np.fft.fftn(x.reshape(dims[::-1])).reshape(-1)) < 1e-12, dims
        assert rel_l2(back, x) < 1e-12, dims


def test_chirp_batch_and_caller_array(oracle):
    # FP64 batches of such lengths; their plans still take no caller array
    n, count = 97, 21
    x = seeded((n, count), 3)
    fw = topefft.Framework()
    p = topefft.BatchPlan(fw, n, count, x)
    fwd = p.exec(topefft.FORWARD)
    back = p.exec(topefft.INVERSE)
    want = np.concatenate([oracle.dft(x[i * n:(i + 1) * n], (n,), topefft.FORWARD) for i in range(count)])
    assert rel_l2(fwd, want) < 1e-12 and rel_l2(back, x) < 1e-12
    fw.lib.topePlanExecPtr(fw.f, p.impl, p.t.data, topefft.FORWARD)
    assert fw.f.error == topefft.TOPE_ERROR_UNSUPPORTED
    p.destroy()
    fw.destroy()
