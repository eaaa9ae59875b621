"""Workloads of the transform library for performance measurement.

A case is a dict of plain values.  Its "kind" says through which entry point
a program runs it:

  host    tope1DPlanInit / tope1DExec: the array lives in the plan, every
          Exec downloads its result into the caller's host array
  array   plan for a 1D, 2D or 3D array, run on the caller's device arrays
          (topePlanExecPtr)
  own     the same plans run on their own device array (tope*DExecDevice):
          lengths with a prime factor above 7, whose padded plans take no
          caller array
  batch   `count` transforms of one length (topeBatchPlanInit), on the
          caller's device arrays
  uneven  packed batch of power-of-two lengths (topeManyPlanInit), on the
          caller's device arrays
  real    real-to-complex and complex-to-real (topeRealPlanInitEx), on the
          caller's device arrays

One pass is one FORWARD and one INVERSE transform, each of an array of its
own (the host kind transforms the plan's array there and back).  The arrays
change roles from pass to pass -- what was transformed forward is transformed
back by the next pass -- so the values stay bounded however often a case runs.
"""
import ctypes
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "tope-fft_amd", "python"))

import topefft  # noqa: E402

MODES = {"valu": topefft.MODE_VALU, "mfma_fp16x3": topefft.MODE_MFMA_FP16X3, "mfma_bf16x6": topefft.MODE_MFMA_BF16X6}


def listed():
    return [
        # the library's own call sequence at a short length: the latency of
        # one synchronous call with its download
        {"name": "host_1d_1024", "kind": "host", "nx": 1024},
        # one mid-sized signal on the device: launches and their gaps
        {"name": "c2c_1d_65536", "kind": "array", "prec": "f64", "mode": "valu", "nx": 65536, "ny": 1, "nz": 1},
        # a long signal (radio and seismic traces): two strided passes over 256 MiB
        {"name": "c2c_1d_16777216", "kind": "array", "prec": "f64", "mode": "valu", "nx": 1 << 24, "ny": 1, "nz": 1},
        # images and 2D spectral solvers, the library's headline shape
        {"name": "c2c_2d_4096", "kind": "array", "prec": "f64", "mode": "valu", "nx": 4096, "ny": 4096, "nz": 1},
        # 3D spectral solvers in double precision
        {"name": "c2c_3d_256", "kind": "array", "prec": "f64", "mode": "valu", "nx": 256, "ny": 256, "nz": 256},
        # a large 3D field in single precision
        {"name": "c2c_3d_512_c64", "kind": "array", "prec": "f32", "mode": "valu", "nx": 512, "ny": 512, "nz": 512},
        # many equal signals in single precision on the matrix cores
        {"name": "batch_4096x4096_mfma", "kind": "batch", "prec": "f32", "mode": "mfma_fp16x3", "n": 4096, "count": 4096},
        # many signals of uneven length, packed back to back
        {"name": "uneven_20000", "kind": "uneven", "prec": "f64", "count": 20000, "lmin": 6, "lmax": 14},
        # real images: half spectrum and back
        {"name": "real_2d_4096", "kind": "real", "prec": "f64", "nx": 4096, "ny": 4096, "nz": 1},
        # array sizes chosen by the problem, not by the transform: products of 2, 3, 5 and 7
        {"name": "smooth_2d_3000", "kind": "array", "prec": "f64", "mode": "valu", "nx": 3000, "ny": 3000, "nz": 1},
        {"name": "smooth_3d_100", "kind": "array", "prec": "f64", "mode": "valu", "nx": 100, "ny": 100, "nz": 100},
        # and sizes with large prime factors
        {"name": "prime_2d_1009", "kind": "own", "nx": 1009, "ny": 1009, "nz": 1},
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _smooth(n):
    for p in (2, 3, 5, 7):
        while n % p == 0:
            n //= p
    return n == 1


def _near_smooth(n):
    """The nearest length at or below n without prime factors above 7."""
    while not _smooth(n):
        n -= 1
    return n


def draw(rng):
    kind = rng.choice(["host", "pow2", "pow2", "smooth", "smooth", "own", "batch", "uneven", "real"])
    prec = rng.choice(["f64", "f32"])
    if kind == "host":
        return {"kind": "host", "nx": _log_int(rng, 8, 16384)}
    if kind == "pow2":
        nd = rng.choice([1, 2, 3])
        if nd == 1:  # one signal: complex128 (a complex64 signal is a batch of one)
            return {"kind": "array", "prec": "f64", "mode": "valu", "nx": 1 << rng.randint(10, 24), "ny": 1, "nz": 1}
        total = rng.randint(14, 24)
        if nd == 2:
            a = rng.randint(max(4, total - 12), min(12, total - 4))
            lx, ly, lz = a, total - a, 0
        else:
            a = rng.randint(3, total // 2)
            b = rng.randint(max(3, total - a - 11), max(3, min(11, total - a - 3)))
            lx, ly, lz = a, b, total - a - b
        mode = rng.choice(["valu", "mfma_fp16x3"]) if prec == "f32" else "valu"
        return {"kind": "array", "prec": prec, "mode": mode, "nx": 1 << lx, "ny": 1 << ly, "nz": 1 << lz}
    if kind == "smooth":
        nd = rng.choice([2, 2, 3])
        # a plan with one axis that is no power of two
        d = [_near_smooth(_log_int(rng, 24, 4096 if nd == 2 else 256)) for _ in range(nd)] + [1] * (3 - nd)
        if all(v & (v - 1) == 0 for v in d):
            d[0] = 240
        return {"kind": "array", "prec": prec, "mode": "valu", "nx": d[0], "ny": d[1], "nz": d[2]}
    if kind == "own":
        nd = rng.choice([1, 2, 3])
        hi = (1 << 20, 2000, 160)[nd - 1]
        d = []
        for _ in range(nd):
            n = _log_int(rng, (100, 50, 20)[nd - 1], hi)
            while _smooth(n):
                n += 1
            d.append(n)
        d += [1] * (3 - nd)
        return {"kind": "own", "nx": d[0], "ny": d[1], "nz": d[2]}
    if kind == "batch":
        mode = rng.choice(["valu", "mfma_fp16x3", "mfma_bf16x6"]) if prec == "f32" else "valu"
        n = 1 << (rng.randint(8, 12) if mode != "valu" else rng.randint(6, 14))
        if mode == "valu" and rng.random() < 0.3:
            n = _near_smooth(_log_int(rng, 60, 4000))
        return {"kind": "batch", "prec": prec, "mode": mode, "n": n, "count": _log_int(rng, 16, max(17, (1 << 24) // n))}
    if kind == "uneven":
        lmin = rng.randint(4, 10)
        return {"kind": "uneven", "prec": prec, "count": _log_int(rng, 100, 20000), "lmin": lmin,
                "lmax": rng.randint(lmin, 13 if lmin > 8 else 14)}
    nd = rng.choice([1, 2, 3])
    if nd == 1:
        d = [1 << rng.randint(8, 22), 1, 1]
    elif rng.random() < 0.5:
        e = [rng.randint(5, (12, 8)[nd - 2]) for _ in range(nd)]
        d = [1 << v for v in e] + [1] * (3 - nd)
    else:
        d = [2 * _near_smooth(_log_int(rng, 20, (1500, 100)[nd - 2]))]
        d += [_near_smooth(_log_int(rng, 24, (3000, 200)[nd - 2])) for _ in range(nd - 1)] + [1] * (3 - nd)
    return {"kind": "real", "prec": prec, "nx": d[0], "ny": d[1], "nz": d[2]}


def _dims(case):
    """The array's lengths without trailing ones, x first."""
    d = [case["nx"], case.get("ny", 1), case.get("nz", 1)]
    while len(d) > 1 and d[-1] == 1:
        d.pop()
    return tuple(d)


def _shape(case):
    return tuple(reversed(_dims(case)))


def _sizes(case, seed):
    """Lengths of an uneven batch: powers of two, log-uniform."""
    r = np.random.RandomState(seed % (1 << 31))
    return (1 << r.randint(case["lmin"], case["lmax"] + 1, case["count"])).astype(np.int32)


def _size_seed(case):
    """The lengths belong to the case, the values to the seed."""
    return 1000003 * case["lmin"] + 1009 * case["lmax"] + case["count"]


def work(case):
    kind = case["kind"]
    cb = 8 if case.get("prec") == "f32" else 16
    if kind == "uneven":
        s = _sizes(case, _size_seed(case)).astype(np.float64)
        elems, flops = float(s.sum()), float((5 * s * np.log2(s)).sum())
        return {"bytes": 2 * 2 * cb * elems, "flops": 2 * flops}
    if kind == "batch":
        elems, lg = float(case["n"]) * case["count"], math.log2(case["n"])
        return {"bytes": 2 * 2 * cb * elems, "flops": 2 * 5 * elems * lg}
    elems = float(np.prod([float(v) for v in _dims(case)]))
    flops = 2 * 5 * elems * math.log2(elems)
    if kind == "real":
        half = elems / case["nx"] * (case["nx"] // 2 + 1)
        return {"bytes": 2 * (cb / 2 * elems + cb * half), "flops": flops / 2}
    return {"bytes": 2 * 2 * cb * elems, "flops": flops}


def _uniform(n, prec, gen, amplitude=1.0):
    """n complex values, both parts uniform in [-1, 1) times `amplitude`."""
    v = torch.rand(2 * n, dtype=torch.float32 if prec == "f32" else torch.float64, device=gen.device, generator=gen)
    v.mul_(2.0).sub_(1.0)
    if amplitude != 1.0:
        v.mul_(amplitude)
    return torch.view_as_complex(v.view(n, 2))


def _gen(case, seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _inputs(case, seed):
    """The array to transform forward and the one to transform back."""
    g = _gen(case, seed)
    kind, prec = case["kind"], case.get("prec", "f64")
    if kind == "uneven":
        n = int(_sizes(case, _size_seed(case)).sum())
        return _uniform(n, prec, g), _uniform(n, prec, g, 64.0)
    if kind == "batch":
        n = case["n"] * case["count"]
        return _uniform(n, prec, g), _uniform(n, prec, g, math.sqrt(case["n"]))
    n = int(np.prod(_dims(case)))
    if kind != "real":
        return _uniform(n, prec, g), _uniform(n, prec, g, math.sqrt(n))
    rdt = torch.float32 if prec == "f32" else torch.float64
    x = torch.rand(n, dtype=rdt, device="cuda", generator=g).mul_(2.0).sub_(1.0)
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    h = nx // 2 + 1
    X = _uniform(h * ny * nz, prec, g, math.sqrt(n)).view(nz, ny, h)
    for k in (0, h - 1):  # the columns kx = 0 and nx/2 of a real array's spectrum are Hermitian
        c = X[:, :, k].clone()
        m = torch.roll(torch.flip(c, (0, 1)), (1, 1), (0, 1)).conj()
        X[:, :, k] = 0.5 * (c + m)
    return x, X


_work_stream = None


class _Plans:
    """A framework with its plans; both go when the state goes.  Every
    framework enqueues on the program's one work stream, so transforms of
    different states run one after the other."""

    def __init__(self):
        global _work_stream
        if _work_stream is None:
            _work_stream = torch.cuda.Stream()
        self.fw = topefft.Framework()
        self.fw.set_stream(_work_stream.cuda_stream)
        self.plans = []

    def add(self, plan):
        self.plans.append(plan)
        return plan

    def __del__(self):
        for p in self.plans:
            p.destroy()
        self.fw.destroy()


class _Device:
    """A plan's device array for torch, without a copy; a tensor made of it keeps the plan."""

    def __init__(self, ptr, plan, owner):
        n = plan.n
        self.owner = owner
        self.__cuda_array_interface__ = {"data": (ptr, False), "shape": (n,), "typestr": "<c16", "version": 2}


def _own_arrays(plan, owner):
    """The plan's two device arrays by address (an Exec may leave its result in either)."""
    return {p: torch.as_tensor(_Device(p, plan, owner), device="cuda") for p in (plan.t.data, plan.t.scratch) if p}


def prepare(case, seed):
    kind, prec = case["kind"], case.get("prec", "f64")
    P = topefft.PREC_F32 if prec == "f32" else topefft.PREC_F64
    ctx = _Plans()
    fw = ctx.fw
    host_t = np.complex64 if prec == "f32" else np.complex128
    a, b = _inputs(case, seed)
    if kind == "host":
        plan = ctx.add(topefft.Plan(fw, _dims(case), a.cpu().numpy()))
        return {"kind": kind, "ctx": ctx, "plan": plan, "out": [np.empty(plan.n, np.complex128) for _ in range(2)]}
    if kind == "own":
        pa = ctx.add(topefft.Plan(fw, _dims(case), a.cpu().numpy()))
        pb = ctx.add(topefft.Plan(fw, _dims(case), b.cpu().numpy()))
        return {"kind": kind, "ctx": ctx, "plans": [(pa, _own_arrays(pa, ctx)), (pb, _own_arrays(pb, ctx))]}
    if kind == "uneven":
        sizes = _sizes(case, _size_seed(case))
        plan = ctx.add(topefft.ManyPlan(fw, sizes, np.zeros(int(sizes.sum()), host_t), P))
        return {"kind": kind, "ctx": ctx, "plan": plan, "arrays": [a, b]}
    if kind == "batch":
        plan = ctx.add(topefft.BatchPlan(fw, case["n"], case["count"], np.zeros(case["n"] * case["count"], host_t), P,
                                         MODES[case["mode"]]))
        return {"kind": kind, "ctx": ctx, "plan": plan, "arrays": [a, b]}
    if kind == "real":
        nx, ny, nz = case["nx"], case["ny"], case["nz"]
        plan = ctx.add(topefft.RealPlan(fw, (nx, ny, nz), np.zeros(nx * ny * nz, np.float32 if prec == "f32" else np.float64), P))
        h, pitch = nx // 2 + 1, plan.t.pitch
        pairs = []
        for k in range(2):  # (real array, spectrum at the plan's pitch, its columns 0 .. nx/2)
            real = a if k == 0 else torch.empty_like(a)
            spec = torch.zeros(nz * ny, pitch, dtype=b.dtype, device="cuda")
            if k == 1:
                spec[:, :h] = b.view(nz * ny, h)
            pairs.append((real, spec, spec[:, :h]))
        return {"kind": kind, "ctx": ctx, "plan": plan, "pairs": pairs}
    d = _dims(case)
    zeros = np.zeros(int(np.prod(d)), host_t)
    if len(d) == 1:
        plan = ctx.add(topefft.Plan(fw, d, zeros))
    elif prec == "f32":
        plan = ctx.add(topefft.Plan(fw, d, zeros, precision=P, mode=MODES[case["mode"]]))
    else:
        plan = ctx.add(topefft.Plan(fw, d, zeros))
    return {"kind": kind, "ctx": ctx, "plan": plan, "arrays": [a, b]}


def run(state):
    kind = state["kind"]
    F, B = topefft.FORWARD, topefft.INVERSE
    if kind == "host":
        plan, out = state["plan"], state["out"]
        return [plan.exec(F, out[0]), plan.exec(B, out[1])]
    if kind == "own":
        (pa, va), (pb, vb) = state["plans"]
        state["plans"].reverse()
        pa.exec_device(F)
        pb.exec_device(B)
        return [va[pa.t.data], vb[pb.t.data]]
    plan = state["plan"]
    if kind == "real":
        (ra, sa, ha), (rb, sb, hb) = state["pairs"]
        state["pairs"].reverse()
        plan.exec_ptr(ra.data_ptr(), sa.data_ptr(), F)
        plan.exec_ptr(rb.data_ptr(), sb.data_ptr(), B)
        return [ha, rb]
    a, b = state["arrays"]
    state["arrays"].reverse()
    if kind == "batch":
        fw = plan.fw
        fw.lib.topePlanExecPtr(ctypes.byref(fw.f), plan.impl, ctypes.c_void_p(a.data_ptr()), F)
        fw.check("topePlanExecPtr")
        fw.lib.topePlanExecPtr(ctypes.byref(fw.f), plan.impl, ctypes.c_void_p(b.data_ptr()), B)
        fw.check("topePlanExecPtr")
    else:
        plan.exec_ptr(a.data_ptr(), F)
        plan.exec_ptr(b.data_ptr(), B)
    return [a, b]


def _in_64_bits(t):
    return t.cpu().to(torch.complex128 if t.is_complex() else torch.float64)


def exact(case, seed):
    kind = case["kind"]
    a, b = (_in_64_bits(t) for t in _inputs(case, seed))
    if kind == "uneven":
        sizes = _sizes(case, _size_seed(case)).astype(np.int64)
        offs = np.cumsum(sizes) - sizes
        fa, fb = torch.empty_like(a), torch.empty_like(b)
        for n in np.unique(sizes):
            at = torch.from_numpy((offs[sizes == n][:, None] + np.arange(n)[None, :]).reshape(-1))
            fa[at] = torch.fft.fft(a[at].view(-1, int(n))).reshape(-1)
            fb[at] = torch.fft.ifft(b[at].view(-1, int(n))).reshape(-1)
        return [fa, fb]
    if kind == "batch":
        n = case["n"]
        return [torch.fft.fft(a.view(-1, n)).reshape(-1), torch.fft.ifft(b.view(-1, n)).reshape(-1)]
    s = _shape(case)
    if kind == "host":  # there and back: the second answer is the input
        return [torch.fft.fft(a), a]
    if kind == "real":
        nx, ny, nz = case["nx"], case["ny"], case["nz"]
        h = nx // 2 + 1
        return [torch.fft.rfftn(a.view(nz, ny, nx)).reshape(nz * ny, h),
                torch.fft.irfftn(b.view(nz, ny, h), (nz, ny, nx)).reshape(-1)]
    return [torch.fft.fftn(a.view(s)).reshape(-1), torch.fft.ifftn(b.view(s)).reshape(-1)]
