"""Fused smoothing passes of the FP32 V-cycle (fused32.hip) against the
half-sweep kernels they replace: the same V-cycle bit for bit, at sizes whose
tiles, rims and z-chunks end unevenly, for every boundary mix."""
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

# one tile and less; several with remainders in x and y; the thinnest z; six
# z-chunks of 34 planes with a shorter last one
SHAPES = [((64, 48, 8), 3), ((120, 72, 40), 4), ((264, 104, 16), 4), ((64, 64, 200), 4)]


@pytest.mark.parametrize("coef", [ph.CoefFormat.BF16, ph.CoefFormat.FP16])
@pytest.mark.parametrize("mix", list(BC_MIXES))
@pytest.mark.parametrize("shape,levels", SHAPES)
def test_fused_vcycle_equals_half_sweeps(ctx, shape, levels, mix, coef):
    g = Grid3D(*shape)
    bc, _ = bc_pair(mix)
    n = g.num_cells()
    K = torch.as_tensor(random_K(n, 31)).to(ctx.device)
    r = torch.as_tensor(np.random.default_rng(32).standard_normal(n)).to(ctx.device)
    # the direct coarsest solve: several of these coarsest grids have an odd
    # periodic axis, where neighbours share a colour and GSRB has no fixed order
    cfg = ph.HeadSolveConfig.mixed(1e-10, levels, coef)
    z = []
    for fuse in (0, 1):
        ws = ph.FlowWorkspace()
        ws.set_tuning(ph.FlowWorkspace.TUNE_FUSE, fuse)
        M = nm.MultigridPreconditioner.build(ctx, ws, g, bc, cfg, K)
        out = ctx.empty(n)
        M.apply(ctx, r, out)
        ctx.synchronize()
        z.append(out)
        ws.close()
    assert torch.isfinite(z[1]).all()
    assert torch.equal(z[0], z[1])


@pytest.mark.parametrize("mix", list(BC_MIXES))
@pytest.mark.parametrize("shape,levels", [((96, 16, 128), 3), ((16, 64, 128), 3), ((8, 96, 256), 3),
                                          ((24, 8, 320), 3)])
def test_fused_vcycle_narrower_than_a_tile(ctx, shape, levels, mix):
    """Domains of fewer rows or places than a tile: on periodic sides it wraps onto
    itself."""
    test_fused_vcycle_equals_half_sweeps(ctx, shape, levels, mix, ph.CoefFormat.BF16)


@pytest.mark.parametrize("graph", [0, 1])
@pytest.mark.parametrize("fold_r", [0, 1])
@pytest.mark.parametrize("shape", [(64, 64, 64), (128, 96, 48)])
def test_fused_solve_matches_half_sweeps(ctx, shape, fold_r, graph):
    """The solve around them, with the r update folded into the half-sweeps' first one
    or before the passes: (r, r) grouped differently, which decides only when to
    stop (test_batched.py holds the heads to equality)."""
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
        res = ph.solve_head(h, K, g, bc, ph.HeadSolveConfig.mixed(1e-10, 4), ctx, ws)
        assert res.converged and res.true_residual <= 1e-10 * res.bnorm
        heads.append(h.cpu().numpy())
        its.append(res.num_iterations)
        ws.close()
    assert its[0] == its[1]
    assert rel_l2(heads[1], heads[0]) < 1e-12
