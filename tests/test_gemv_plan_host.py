"""The host side of the standalone GEMV plan over a HIP runtime of stubs
(hip_stub.cpp), without a GPU: where its pinned memory is refused, the plan
copies instead; its timing runs read defined memory; what a run allocates."""
import os
import shutil
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(ROOT, "cis2-lab-archive_amd")
ROCM = "/opt/rocm"

SETUP = """
import ctypes, sys
import numpy as np
sys.path.insert(0, %r)
stub = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
from cis2amd import GemvPlan
def check(M, x, y):
    assert np.array_equal(y, x[..., :1] + np.arange(M, dtype=np.float32)), y
M, K = 40, 8
x = np.arange(1, 9, dtype=np.float32)
X = np.arange(8, 8 + 5 * K, dtype=np.float32).reshape(5, K)
""" % PKG


@pytest.fixture(scope="module")
def stub(tmp_path_factory):
    gxx = shutil.which("g++")
    if not gxx or not os.path.isdir(os.path.join(ROCM, "include", "hip")):
        pytest.skip("no g++ or no HIP headers")
    so = tmp_path_factory.mktemp("stub") / "libhipstub.so"
    b = subprocess.run([gxx, "-std=c++17", "-O1", "-shared", "-fPIC", "-D__HIP_PLATFORM_AMD__",
                        "-I" + os.path.join(ROCM, "include"), "-o", str(so),
                        os.path.join(ROOT, "tests", "hip_stub.cpp")],
                       capture_output=True, text=True, timeout=300)
    assert b.returncode == 0, b.stderr[-2000:]
    return str(so)


def run_stubbed(stub, setup, body):
    r = subprocess.run([sys.executable, "-c", setup + body, stub], capture_output=True, text=True,
                       timeout=120)
    assert r.returncode == 0, r.stderr[-2000:]


def run(stub, body):
    run_stubbed(stub, SETUP, body)


@pytest.mark.parametrize("pinned", [0, 1, 2, 100])
def test_plan_without_pinned_memory(stub, pinned):
    """`pinned` allocations of pinned memory succeed: the plan is made, lone
    and batched products go through it, and everything is given back."""
    run(stub, """
stub.stub_allow_pinned(%d)
p = GemvPlan(np.ones((M, K), np.float32))
check(M, x, p(x))
check(M, X, p.run_batch(X))
check(M, x, p(x))
assert stub.stub_launches() == 3 and stub.stub_undefined_inputs() == 0
p.close()
assert stub.stub_live() == 0
""" % pinned)


@pytest.mark.parametrize("rows", [40, 16 * 513], ids=["lone-kernel", "streaming-kernel"])
def test_timing_runs_have_defined_inputs(stub, rows):
    """plan_time and plan_time_batch multiply memory that was written, before
    and after a run."""
    run(stub, """
M = %d
p = GemvPlan(np.ones((M, K), np.float32), copies=2)
p.time(3)
check(M, x, p(x))
p.time(3)
p.time_batch(2, 3)
check(M, X[:3], p.run_batch(X[:3]))
p.time_batch(3, 3)
p.time_batch(4, 3)
assert stub.stub_launches() == 2 * (2 + 3) + 1 + 4 + 1 + 4 + 4
assert stub.stub_undefined_inputs() == 0
p.close()
assert stub.stub_live() == 0
""" % rows)


def test_allocations_of_a_plan(stub):
    """A batched run allocates where it is larger than those before it: its
    device inputs and, where the plan's first pinned block is too small, one
    pinned block; every other run allocates nothing."""
    run(stub, """
p = GemvPlan(np.ones((M, K), np.float32))
n0 = stub.stub_allocations()
check(M, x, p(x))
assert stub.stub_allocations() == n0
check(M, X, p.run_batch(X))
assert stub.stub_allocations() <= n0 + 2
n1 = stub.stub_allocations()
check(M, X[:2], p.run_batch(X[:2]))
check(M, x, p(x))
check(M, X, p.run_batch(X))
assert stub.stub_allocations() == n1
p.close()
assert stub.stub_live() == 0
""")
