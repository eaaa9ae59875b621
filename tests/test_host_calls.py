"""What the library asks of the HIP runtime, on the CPU: libtopefft.so in a
process of its own with the runtime calls counted (hip_call_log.c), so kernel
launches, copies and events of an entry point can be compared with what the
library says of itself."""
import os
import subprocess
import sys

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
PYDIR = os.path.join(os.path.dirname(HERE), "tope-fft_amd", "python")

PRELUDE = """
import ctypes as C, sys
log = C.CDLL(sys.argv[1], mode=C.RTLD_GLOBAL)
sys.path.insert(0, sys.argv[2])
import numpy as np
import topefft
F, B = topefft.FORWARD, topefft.INVERSE
log.log_launches.restype = C.c_long
log.log_sequence.restype = C.c_ulong

def launches(call):
    before = log.log_launches()
    call()
    return log.log_launches() - before

def sequence(call):
    log.log_sequence()
    call()
    return log.log_sequence()
"""


@pytest.fixture(scope="module")
def run(tmp_path_factory):
    import topefft
    if not os.path.exists(topefft.LIB_PATH):
        pytest.skip("libtopefft.so not built")
    so = str(tmp_path_factory.mktemp("log") / "hip_call_log.so")
    inc = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "include")
    subprocess.run(["gcc", "-shared", "-fPIC", "-O1", "-w", "-I", inc, "-o", so,
                    os.path.join(HERE, "hip_call_log.c")], check=True)

    def go(body):
        r = subprocess.run([sys.executable, "-c", PRELUDE + body, so, PYDIR], capture_output=True, text=True,
                           timeout=300)
        assert r.returncode == 0, r.stderr[-2000:]
        return r.stdout

    return go


# FP64 2^24 is the length whose callers' arrays run another schedule than the
# plan's own array; 2^16 runs one with exchanged buffers, 4096 x 64 the same
# passes in both
@pytest.mark.parametrize("dims", [(1 << 24,), (1 << 16,), (4096, 64)], ids=lambda d: "x".join(map(str, d)))
def test_pass_times_of_caller_array(run, dims):
    """Names, count and times follow the schedule that the timed call ran."""
    run(f"""
dims = {dims!r}
fw = topefft.Framework()
p = topefft.Plan(fw, dims, np.zeros(int(np.prod(dims)), complex))
own, data = p.pass_names(), p.t.data
a = np.zeros(8, complex)
ptr = a.ctypes.data // 16 * 16
n_own, n_ptr = launches(lambda: p.exec_device(F)), launches(lambda: p.exec_ptr(ptr, F))
p.pass_timing(True)
for _ in range(3):
    assert launches(lambda: p.exec_ptr(ptr, F)) == n_ptr
ms, names = p.pass_times(), p.pass_names()
assert len(ms) == len(names) == p.pass_count() == n_ptr, (ms, names)
assert list(ms) == [1.0] * n_ptr, ms
# both schedules in one recording: the last one's times alone
p.exec_ptr(ptr, B)
assert launches(lambda: p.exec_device(F)) == n_own
assert p.pass_names() == own
assert list(p.pass_times()) == [1.0] * n_own
p.exec_device(F)
p.exec_ptr(ptr, F)
assert list(p.pass_times()) == [1.0] * n_ptr
for i in range(n_ptr):
    assert p.time_pass(i, F, 4) == 1.0
# switched on again: the plan's own schedule until a transform is timed
p.pass_timing(False)
p.pass_timing(True)
assert p.pass_names() == own and list(p.pass_times()) == [0.0] * n_own
p.pass_timing(False)
p.exec_ptr(ptr, F)
assert p.pass_names() == own
p.destroy()
""")


# 3D arrays of 512 MiB and more run their X and Y passes over chunks of
# planes: complex64 512 x 512 x 256 in two, FP64 512^3 in eight, a real array
# whose inverse runs the chunks last; 64 x 32 x 16 is not chunked
@pytest.mark.parametrize("kind,dims,chunks", [("f32", (512, 512, 256), 2), ("f64", (512, 512, 512), 8),
                                              ("real", (1024, 512, 256), 8), ("f64", (64, 32, 16), 1)],
                         ids=lambda v: "x".join(map(str, v)) if isinstance(v, tuple) else str(v))
def test_timed_transforms_make_the_same_launches(run, kind, dims, chunks):
    """Timing changes nothing of the schedule, and a pass's time is the sum of its launches."""
    run(f"""
kind, dims, chunks = {kind!r}, {dims!r}, {chunks!r}
fw = topefft.Framework()
n = int(np.prod(dims))
if kind == "real":
    p = topefft.RealPlan(fw, dims, np.zeros(n))
    impl = p.t.impl
elif kind == "f32":
    p = topefft.Plan(fw, dims, np.zeros(n, np.complex64), precision=topefft.PREC_F32)
    impl = p.impl
else:
    p = topefft.Plan(fw, dims, np.zeros(n, complex))
    impl = p.impl
ms = (C.c_double * 8)()
for d in (F, B):
    assert launches(lambda: p.exec_device(d)) == 2 * chunks + 1
    want = sequence(lambda: p.exec_device(d))
    fw.lib.topePlanPassTiming(impl, 1)
    for _ in range(3):
        assert sequence(lambda: p.exec_device(d)) == want
    got = fw.lib.topePlanPassTimes(C.byref(fw.f), impl, ms, 8)
    fw.lib.topePlanPassTiming(impl, 0)
    assert got == p.pass_count() == 3
    assert sorted(ms[:3]) == [1, chunks, chunks], ms[:3]
p.destroy()
""")


@pytest.mark.parametrize("order", ["small first", "large first"])
def test_exec_event_fences(run, order):
    """An Exec of up to 256 KiB records its transform with events that have no
    system-scope fence and a fenced one behind its copy, a larger Exec fenced ones
    throughout, whichever the framework ran first; profileThis reads the last one's."""
    run(f"""
fw = topefft.Framework()
small = topefft.Plan(fw, (1024,), np.zeros(1024, complex))
large = topefft.Plan(fw, (1 << 16,), np.zeros(1 << 16, complex))
PLAIN, FENCED = 0x20000000, 0  # hipEventDisableSystemFence, hipEventDefault
flags = (C.c_uint * 64)()

def events(p):
    log.log_records(flags, 64)
    p.exec(F)
    return list(flags[:log.log_records(flags, 64)])

want = {{"small": [PLAIN, PLAIN, FENCED], "large": [FENCED] * 4}}
for who in {["small", "large", "small", "large"] if order == "small first" else ["large", "small", "large", "small"]!r}:
    p = small if who == "small" else large
    assert events(p) == want[who], (who, flags[:4])
    assert fw.lib.profileThis(fw.f.event) == 1e6 * p.pass_count()  # a launch counts a millisecond
small.destroy()
large.destroy()
""")
