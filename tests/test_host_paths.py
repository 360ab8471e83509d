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


VCYCLE = """
def vcycle(shape, levels, mixed, counts=(2, 2), fuse=-1):
    g, bc = core.Grid3D(*shape).c(), core.BCSpec.darcy_x().c()
    cfg = _lib.mf3d_head_solve_config()
    lib.mf3d_default_config(ref(cfg))
    cfg.mg_levels, cfg.precond_precision = levels, int(mixed)
    cfg.coef_format = 1  # BF16
    cfg.mg_pre_smooth, cfg.mg_post_smooth = counts
    ws, v, n = C.c_void_p(), C.c_void_p(1 << 43), g.nx * g.ny * g.nz
    assert lib.mf3d_workspace_create(ref(ws)) == 0
    assert lib.mf3d_workspace_set_tuning(ws, 17, fuse) == 0
    assert lib.mf3d_mg_setup(ws, None, ref(g), ref(bc), ref(cfg), v, n) == 0
    stub.clear()
    assert lib.mf3d_mg_precondition(ws, None, v, v, n) == 0
    lib.mf3d_workspace_destroy(ws)
    return stub.log()
"""


def _count(log, name):
    return sum(name in n for n in log)


@pytest.mark.parametrize("shape,levels,fused", [
    ((256, 256, 256), 5, 1), ((1024, 128, 128), 5, 1), ((64, 64, 2048), 4, 1),
    ((8192, 32, 32), 4, 1), ((2048, 512, 8), 3, 1), ((512, 512, 512), 5, 2),
    # tiles of 28 places x 24 rows mostly outside the domain
    ((1024, 8, 1024), 3, 0), ((16, 1024, 512), 3, 0), ((8, 1024, 1024), 3, 0),
    ((16, 4096, 4096), 3, 0),
    ((128, 128, 128), 5, 0)])
def test_fp32_levels_in_fused_passes(shape, levels, fused):
    """Two fused passes for each level whose tiles are full, counted from the finest."""
    log, = host_runs.run(VCYCLE + f"show(vcycle({shape}, {levels}, True))")
    assert _count(log, "fused_kernel") == 2 * fused


# V-cycle levels: 64^3 two waves of FP64 windows, 32^3 one, 16^3 and below one workgroup
@pytest.mark.parametrize("mixed,counts,passes", [
    (False, (2, 2), 2 + 2 + 2), (False, (1, 1), 0 + 2 + 2), (False, (2, 1), 0 + 2 + 2),
    (False, (3, 3), 0 + 4 + 0), (False, (4, 4), 0 + 4 + 0), (False, (1, 3), 0 + 3 + 0),
    # FP32: not the finest level
    (True, (2, 2), 0 + 2 + 2), (True, (1, 1), 0 + 2 + 2), (True, (4, 4), 0 + 4 + 0)])
def test_small_levels_in_window_passes(mixed, counts, passes):
    """Window passes where they are fewer waves than half the launches they replace."""
    log, = host_runs.run(VCYCLE + f"show(vcycle((64, 64, 64), 4, {mixed}, {counts}))")
    assert _count(log, "block_kernel") == passes
    log, = host_runs.run(VCYCLE + f"show(vcycle((64, 64, 64), 4, {mixed}, {counts}, fuse=0))")
    assert _count(log, "block_kernel") == 0


SOLVE = """
def solve(shape, levels, mixed, fuse, h=1 << 43):
    g, bc = core.Grid3D(*shape).c(), core.BCSpec.darcy_x().c()
    cfg, res = _lib.mf3d_head_solve_config(), _lib.mf3d_head_solve_result()
    lib.mf3d_default_config(ref(cfg))
    cfg.mg_levels, cfg.precond_precision, cfg.coef_format = levels, int(mixed), 1
    ws, n = C.c_void_p(), g.nx * g.ny * g.nz
    assert lib.mf3d_workspace_create(ref(ws)) == 0
    assert lib.mf3d_workspace_set_tuning(ws, 17, fuse) == 0
    stub.clear()
    st = lib.mf3d_solve_head(ws, None, ref(g), ref(bc), ref(cfg), C.c_void_p(1 << 43),
                             C.c_void_p(h), n, ref(res))
    log, used, said = stub.log(), stub.in_use(), lib.mf3d_workspace_bytes(ws)
    lib.mf3d_workspace_destroy(ws)
    assert stub.in_use() == 0 and used == said
    return st, used, log
"""


@pytest.mark.parametrize("head", [1 << 43, (1 << 43) + 8])  # the second is solved in a copy
@pytest.mark.parametrize("shape,levels,mixed", [((256, 256, 256), 5, True),
                                                ((256, 256, 256), 5, False),
                                                ((64, 64, 64), 4, False),
                                                ((128, 128, 128), 5, True)])
def test_memory_for_half_sweeps_is_enough(shape, levels, mixed, head):
    """The fused and window passes' buffers give way: a solve that fits without them
    fits, on half-sweeps, and with room for some of them takes those."""
    off, on, tight, less, some = host_runs.run(SOLVE + f"""
args = {shape}, {levels}, {mixed}
off, on = solve(*args, 0, {head}), solve(*args, -1, {head})
show(off); show(on)
stub.limit(off[1])
show(solve(*args, -1, {head}))
stub.limit(off[1] - 1)
show(solve(*args, -1, {head}))
stub.limit((off[1] + on[1]) // 2)
show(solve(*args, -1, {head}))
""")
    passes = lambda log: _count(log, "block_kernel") + _count(log, "fused")  # noqa: E731
    assert off[0] == on[0] == tight[0] == some[0] == 0 and less[0] == 5  # MF3D_ERR_ALLOC
    assert passes(on[2]) > passes(off[2]) == 0
    assert off[1] < on[1] <= 1.15 * off[1]
    assert tight[1] == off[1] and passes(tight[2]) == 0
    assert off[1] <= some[1] <= (off[1] + on[1]) // 2


@pytest.mark.parametrize("mixed,level,kernels", [
    (True, 0, ["fused_kernel", "fused_kernel"]), (True, 1, None),
    (False, 0, ["fused64_kernel", "fused64_kernel"]), (False, 4, None)])
def test_fused_passes_of_one_level(mixed, level, kernels):
    """mf3d_mg_passes launches what a V-cycle launches on that level, or refuses."""
    code = VCYCLE.replace("    lib.mf3d_workspace_destroy(ws)", f"""    vc = stub.log()
    stub.clear()
    show([lib.mf3d_mg_passes(ws, None, {level}, 1), stub.log(), vc])
    lib.mf3d_workspace_destroy(ws)""")
    (st, log, vc), = host_runs.run(code + f"vcycle((256, 256, 256), 5, {mixed})")
    if kernels is None:
        assert st == 7 and log == []  # MF3D_ERR_UNSUPPORTED
        return
    assert st == 0 and len(log) == 2 and all(k in n for k, n in zip(kernels, log))
    # (without PCG's partial sums the FP64 result stays in natural order too)
    assert log[0] in vc and log[1] in vc
