"""Solves while single allocations find no memory: argv = the library of
refuse.c.  A program of its own, since the library has to be loaded before
what calls hipMalloc."""

import ctypes
import os
import sys

import numpy as np

R = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
ROOT = os.path.dirname(os.path.dirname(os.path.dirname(os.path.abspath(__file__))))
sys.path[:0] = [ROOT, os.path.join(ROOT, "tests")]
import arcanefem_amd as A  # noqa: E402
from test_gpu_resident import band, checkerboard_blocks, device_system  # noqa: E402
from test_gpu_resident_limit import RESIDENT, resident_launches, shuffled  # noqa: E402

LIB = A.lib()
HIP = ctypes.CDLL(next(line.split()[-1] for line in open("/proc/self/maps") if "libamdhip64.so" in line))
R.refuse_real(ctypes.cast(HIP.hipMalloc, ctypes.c_void_p))
R.refuse_arm.argtypes = [ctypes.c_long] * 2
R.refuse_refused.restype = R.refuse_calls.restype = ctypes.c_long
R.refuse_arm(0, 0)
A.init(0)
assert len(RESIDENT) == 3


def sweep(name, make, solve):
    """The k-th allocation of a solve finds no memory, nor does its second
    try, for every k: the solve goes on without the one-launch kernel, and the
    next one does not try it."""
    k = 0
    while True:
        s, check, keep = make()
        R.refuse_arm(k, 2)
        n, r = resident_launches(A, lambda: solve(s))
        refused, calls = R.refuse_refused(), R.refuse_calls()
        R.refuse_arm(0, 0)
        check(r)
        assert (n == 0) == (refused > 0), (name, k, n, refused)
        n, r = resident_launches(A, lambda: solve(s))
        check(r)
        assert (n == 0) == (refused > 0), (name, k, n, refused)
        if not refused:
            break
        assert refused == 2
        k += 1
    assert calls == k
    print(f"{name}: {k} allocations", flush=True)
    assert k >= 8


def single(method):
    def make():
        M = band(5000, [1, 2, 70], shift=0.05)
        s, d = device_system(A, M)
        b = np.random.default_rng(1).normal(size=5000)
        s.rhs().upload(b)
        if method == 3:
            rid = np.repeat(np.arange(5000), np.diff(M.indptr))
            s.set_spai(A.DeviceArray.from_numpy(np.where(M.indices == rid, 1.0, 0.0).astype(np.float32)))
        y = A.DeviceArray(5000, np.float64)
        s.spmv(s.rhs(), y)  # what the streaming kernels need is there

        def check(r):
            assert r.converged and np.linalg.norm(b - M @ s.solution().numpy()) <= 1.01e-8 * np.linalg.norm(b)

        return s, check, (d, y)

    sweep(f"method {method}", make, lambda s: s.solve(raise_on_failure=False, method=method, rtol=1e-8))


def morton():
    def make():
        s, M, keep = shuffled(A)
        b = s.rhs().numpy()
        y = A.DeviceArray(M.shape[0], np.float64)
        s.spmv(s.rhs(), y)

        def check(r):
            assert r.converged and np.linalg.norm(b - M @ s.solution().numpy()) <= 1.01e-8 * np.linalg.norm(b)

        return s, check, (keep, y)

    sweep("rows in Morton order", make, lambda s: s.solve(raise_on_failure=False, rtol=1e-8))


def batch():
    def make():
        s, offs, keep = checkerboard_blocks(A, [20, 33, 8])
        bs = A.BatchSolver(s, offs)
        bs.solve(rtol=1e-8, persistent=2)

        def check(r):
            assert all(q.converged and q.relres <= 1e-8 for q in r[0])

        return bs, check, (s, keep)

    sweep("batch", make, lambda bs: bs.solve(raise_on_failure=False, rtol=1e-8))


for m in (0, 1, 3):
    single(m)
morton()
batch()
print("done", flush=True)
