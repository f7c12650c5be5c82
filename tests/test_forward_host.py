"""The host side of the forward passes over a HIP runtime of stubs
(hip_stub.cpp), without a GPU: which kernels a call launches, and what it does
where an allocation is refused."""
import pytest

from test_gemv_plan_host import PKG, run_stubbed, stub  # noqa: F401

SETUP = """
import ctypes, os, sys
import numpy as np
sys.path.insert(0, %r)
os.environ["CIS2_DECODE_LOCK"] = "0"
stub = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
stub.stub_device_most.argtypes = [ctypes.c_size_t]
from cis2amd import Cis2Error, Cis2Model, artifacts
def count(part):
    return stub.stub_launched(part.encode())
spec = artifacts.ModelSpec("host", 64, 96, 1, 4, 4, 128, 1e-5, 10000.0, True, head_dim=64)
w = artifacts.Weights(spec, 1)
""" % PKG


@pytest.mark.parametrize("tree", [0, 1], ids=["seq", "tree"])
def test_prefill_without_memory_for_the_attention_tiles(stub, tree):  # noqa: F811
    """The tiles' scratch (1.5 MB here, the largest allocation) is refused:
    the rows attend in the per-row kernels, now and once there is memory again
    in tiles."""
    run_stubbed(stub, SETUP, """
n = 300
m = Cis2Model(spec, w, max_pos=n, reduction_mode=%d)
call = lambda: m.forward_rows(np.zeros(n), np.arange(n), np.arange(n) %% 128)
stub.stub_device_most(1 << 20)
call()
assert count("k_attention_tiles") == 0
assert count("k_attention_rows") + count("k_attention_wave") == 1
stub.stub_device_most(1 << 40)
call()
assert count("k_attention_tiles") == 1
m.close()
assert stub.stub_live() == 0
""" % tree)


def test_prefill_too_long_for_the_per_row_attention(stub):  # noqa: F811
    """A prompt whose rows only the tiles can take: refused as out of memory."""
    run_stubbed(stub, SETUP, """
n = 16384
m = Cis2Model(spec, w, max_pos=n)
stub.stub_device_most(100 << 20)
try:
    m.forward_rows(np.zeros(n), np.arange(n), np.arange(n) % 128, want_logits=False)
    assert False
except Cis2Error as e:
    assert "tile" in str(e), e
m.close()
assert stub.stub_live() == 0
""")


@pytest.mark.parametrize("pinned,kernel", [(2, "k_embed"), (3, "k_decode")],
                         ids=["refused", "granted"])
def test_context_without_pinned_memory_for_single_rows(stub, pinned, kernel):  # noqa: F811
    """`pinned` allocations of pinned memory succeed, two of them the decode
    ring's: a context is made either way, and a single row goes through the
    persistent kernel where its logits have mapped memory."""
    run_stubbed(stub, SETUP, """
stub.stub_allow_pinned(%d)
m = Cis2Model(spec, w, max_pos=64)
m.forward_token(0, 5)
assert count("k_embed") + count("k_decode") == count(%r) == 1
m.close()
assert stub.stub_live() == 0
""" % (pinned, kernel))
