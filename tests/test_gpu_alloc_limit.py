"""Device memory that is not there: one-launch solves need a copy of the matrix
and vectors of their own; without them the solve takes the kernels that had
run it before."""

import os
import subprocess
import sys

import pytest

from conftest import ROOT

pytestmark = pytest.mark.gpu

HERE = os.path.join(ROOT, "tests", "alloc_limit")


def test_solves_without_memory_for_the_one_launch_kernel(afem_gpu, tmp_path):
    print("[case] refused allocations", flush=True)
    assert afem_gpu is not None
    so = str(tmp_path / "refuse.so")
    subprocess.run(["gcc", "-O1", "-shared", "-fPIC", os.path.join(HERE, "refuse.c"), "-o", so], check=True)
    p = subprocess.run([sys.executable, "-u", os.path.join(HERE, "solves.py"), so], capture_output=True, text=True,
                       timeout=100)
    print(p.stdout[-2000:], p.stderr[-3000:], flush=True)
    assert p.returncode == 0 and "done" in p.stdout
