"""Host code of the library on a recorded HIP runtime (host_runs.py)."""
from __future__ import annotations

import os
import shutil

import pytest

import host_runs
from macroflow3d_amd import _lib

pytestmark = pytest.mark.skipif(shutil.which("g++") is None or not os.path.exists(_lib.LIB_PATH),
                                reason="needs g++ and the built library")

NET = """
net = C.c_void_p()
assert lib.mf3d_wsnet_create(ref(net)) == 0
g, bc = core.Grid3D(32, 32, 32).c(), core.BCSpec.darcy_x().c()
K = h = C.c_void_p(1 << 43)
loss = C.c_double()
def gradients():
    stub.clear()
    st = lib.mf3d_wsnet_gradients(net, None, ref(g), ref(bc), K, 0, h, 32 ** 3, ref(loss))
    return st, stub.log()
"""


@pytest.mark.parametrize("step", ["hipMemset", "zero_kernel", "hipDeviceSynchronize"])
def test_failed_gradient_scratch_is_not_used(step):
    """A failure while the weight gradients' scratch is made ready leaves no scratch:
    the next call makes it anew before any kernel takes its operands from it."""
    (first, second, log), = host_runs.run(NET + f"""
stub.fail({step!r})
st, _ = gradients()
st2, log = gradients()
show([st, st2, log])
""")
    if first == 0:  # this step is not part of making the scratch
        return
    assert second == 0
    zero = [i for i, n in enumerate(log) if "zero_kernel" in n or n == "hipMemset"]
    use = [i for i, n in enumerate(log) if "planar_kernel" in n]
    assert zero and use and zero[0] < use[0]


def test_first_gradients_wait_for_their_own_stream_only():
    """The first training sample of a size stalls no other stream."""
    log, = host_runs.run(NET + "show(gradients()[1])")
    assert "hipDeviceSynchronize" not in log and "hipMemset" not in log
    assert any("wgrad_kernel" in n for n in log)
