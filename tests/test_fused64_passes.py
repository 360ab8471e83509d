"""Fused smoothing passes of the FP64 V-cycle (fused64.hip) against the half-sweep
kernels they replace, at sizes whose tiles, rims and z-chunks end unevenly, for
every boundary mix."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from helpers import BC_MIXES, bc_pair, random_K, rel_l2
from macroflow3d_amd import numerics as nm
from macroflow3d_amd import physics as ph
from macroflow3d_amd.core import Grid3D
from macroflow3d_amd.kfield import lognormal_lnK

pytestmark = pytest.mark.gpu

# levels above the windows' range (512 of 8^3), the coarse one colour-split: tiles of
# 24 x 24 cells with remainders in x and y, a thin z, several z-chunks
SHAPES = [((80, 72, 56), 4), ((136, 104, 24), 4), ((160, 104, 16), 4), ((48, 40, 200), 4)]


@pytest.mark.parametrize("mix", list(BC_MIXES))
@pytest.mark.parametrize("shape,levels", SHAPES)
def test_fused64_vcycle_matches_half_sweeps(ctx, shape, levels, mix):
    """The same sums up to the order of the x terms: some 1e-16 a cell and half-sweep,
    times the coarsest system's condition (< 1e4)."""
    g = Grid3D(*shape)
    bc, _ = bc_pair(mix)
    n = g.num_cells()
    K = torch.as_tensor(random_K(n, 71)).to(ctx.device)
    r = torch.as_tensor(np.random.default_rng(72).standard_normal(n)).to(ctx.device)
    # the direct coarsest solve: GSRB has no fixed order on odd periodic axes
    cfg = ph.HeadSolveConfig.fp64_direct(1e-10, levels)
    z = []
    for fuse in (0, 1):
        ws = ph.FlowWorkspace()
        ws.set_tuning(ph.FlowWorkspace.TUNE_FUSE, fuse)
        M = nm.MultigridPreconditioner.build(ctx, ws, g, bc, cfg, K)
        out = ctx.empty(n)
        M.apply(ctx, r, out)
        ctx.synchronize()
        z.append(out.cpu().numpy())
        ws.close()
    assert np.isfinite(z[1]).all()
    assert rel_l2(z[1], z[0]) < 1e-11


@pytest.mark.parametrize("mix", list(BC_MIXES))
@pytest.mark.parametrize("shape,levels", [((16, 64, 512), 4), ((40, 16, 640), 4), ((96, 16, 352), 4)])
def test_fused64_vcycle_narrower_than_a_tile(ctx, shape, levels, mix):
    """Domains of fewer places or rows than a tile: on periodic sides it wraps onto
    itself."""
    test_fused64_vcycle_matches_half_sweeps(ctx, shape, levels, mix)


@pytest.mark.parametrize("graph", [0, 1])
@pytest.mark.parametrize("fold_r", [0, 1])
@pytest.mark.parametrize("shape,levels", [((80, 72, 64), 4), ((192, 96, 48), 5)])
def test_fused64_solve_matches_half_sweeps(ctx, shape, levels, fold_r, graph):
    """The solve around them: r update, (r, r) and (r, z) grouped differently, so
    heads equal to the stopping tolerance's rounding and equal iterations."""
    g = Grid3D(*shape)
    bc, _ = bc_pair("darcy_x")
    K = torch.exp(lognormal_lnK(*shape, 2.0, 5.0, 41, device=ctx.device)[0])
    heads, its = [], []
    for fuse in (0, 1):
        ws = ph.FlowWorkspace()
        ws.set_tuning(ph.FlowWorkspace.TUNE_FUSE, fuse)
        ws.set_tuning(ph.FlowWorkspace.TUNE_FOLD_R, fold_r)
        ws.set_tuning(ph.FlowWorkspace.TUNE_GRAPH, graph)
        h = ctx.zeros(g.num_cells())
        res = ph.solve_head(h, K, g, bc, ph.HeadSolveConfig.fp64_direct(1e-10, levels), ctx, ws)
        assert res.converged and res.true_residual <= 1e-10 * res.bnorm
        heads.append(h.cpu().numpy())
        its.append(res.num_iterations)
        ws.close()
    assert its[0] == its[1]
    assert rel_l2(heads[1], heads[0]) < 1e-11
