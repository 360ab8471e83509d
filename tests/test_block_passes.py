"""Window passes of the V-cycle's small levels (block.hip) against the half-sweep
kernels they replace, at sizes whose windows end unevenly, wrap onto themselves or
leave the window mostly empty, for every boundary mix and smoothing count."""
from __future__ import annotations

import numpy as np
import pytest
import torch

import oracle as O
from helpers import BC_MIXES, bc_pair, grid_pair, random_K, rel_l2
from macroflow3d_amd import numerics as nm
from macroflow3d_amd import physics as ph
from macroflow3d_amd.core import Grid3D
from macroflow3d_amd.kfield import lognormal_lnK

pytestmark = pytest.mark.gpu

F32 = ph.PrecondPrecision.FP32
# finest shape, levels: natural and colour-split levels below and at the top, one
# window and many, axes of 2 and 4 cells under a periodic window of 16
SHAPES = [((16, 16, 16), 2), ((48, 32, 16), 3), ((80, 48, 32), 4), ((136, 16, 8), 3),
          ((24, 8, 112), 3), ((104, 56, 40), 4)]
COUNTS = [(2, 2), (1, 1), (3, 2), (4, 5)]


def _apply(ctx, shape, levels, mix, counts, precision, fuse, coef=ph.CoefFormat.BF16):
    g = Grid3D(*shape)
    bc, _ = bc_pair(mix)
    n = g.num_cells()
    K = torch.as_tensor(random_K(n, 51)).to(ctx.device)
    r = torch.as_tensor(np.random.default_rng(52).standard_normal(n)).to(ctx.device)
    # the direct coarsest solve: GSRB has no fixed order on odd periodic axes
    cfg = ph.HeadSolveConfig.fp64_direct(1e-10, levels)
    cfg.precond_precision, cfg.coef_format = precision, coef
    cfg.mg_pre_smooth, cfg.mg_post_smooth = counts
    ws = ph.FlowWorkspace()
    ws.set_tuning(ph.FlowWorkspace.TUNE_FUSE, fuse)
    M = nm.MultigridPreconditioner.build(ctx, ws, g, bc, cfg, K)
    out = ctx.empty(n)
    M.apply(ctx, r, out)
    ctx.synchronize()
    ws.close()
    return out


@pytest.mark.parametrize("counts", COUNTS)
@pytest.mark.parametrize("mix", list(BC_MIXES))
@pytest.mark.parametrize("shape,levels", SHAPES)
def test_fp32_window_passes_equal_half_sweeps(ctx, shape, levels, mix, counts):
    """The FP32 sums are the same, in the same order: bit for bit."""
    coef = ph.CoefFormat.FP16 if counts == (1, 1) else ph.CoefFormat.BF16
    z = [_apply(ctx, shape, levels, mix, counts, F32, fuse, coef) for fuse in (0, -1)]
    assert torch.isfinite(z[1]).all()
    assert torch.equal(z[0], z[1])


@pytest.mark.parametrize("counts", COUNTS)
@pytest.mark.parametrize("mix", list(BC_MIXES))
@pytest.mark.parametrize("shape,levels", SHAPES)
def test_fp64_window_passes_match_half_sweeps(ctx, shape, levels, mix, counts):
    """FP64 differs by the order of the x terms: some 1e-16 a cell and half-sweep,
    times the coarsest system's condition (< 1e4)."""
    z = [_apply(ctx, shape, levels, mix, counts, ph.PrecondPrecision.FP64, fuse).cpu().numpy()
         for fuse in (0, -1)]
    assert np.isfinite(z[1]).all()
    assert rel_l2(z[1], z[0]) < 1e-11


@pytest.mark.parametrize("coef", list(ph.CoefFormat))
@pytest.mark.parametrize("counts", [(2, 2), (1, 1), (3, 2), (4, 3)])
@pytest.mark.parametrize("mix", ["darcy_x", "periodic_x_dirichlet_z", "all_periodic"])
@pytest.mark.parametrize("shape,levels", [((80, 48, 32), 4), ((136, 16, 8), 3), ((104, 56, 40), 4)])
def test_fp32_window_passes_every_face_format(ctx, shape, levels, mix, counts, coef):
    """Every face format, smoothing counts for which the windows are slower included
    (forced; with (2, 2) a forced level may take the fused passes: the default then)."""
    fuse = -1 if counts == (2, 2) else 1
    z = [_apply(ctx, shape, levels, mix, counts, F32, f, coef) for f in (0, fuse)]
    assert torch.isfinite(z[1]).all()
    assert torch.equal(z[0], z[1])


@pytest.mark.parametrize("counts", [(1, 1), (3, 3), (4, 5)])
@pytest.mark.parametrize("shape,levels", [((64, 64, 64), 4), ((48, 32, 16), 3)])
def test_fp64_window_passes_forced(ctx, shape, levels, counts):
    z = [_apply(ctx, shape, levels, "darcy_x", counts, ph.PrecondPrecision.FP64, f).cpu().numpy()
         for f in (0, 1)]
    assert np.isfinite(z[1]).all()
    assert rel_l2(z[1], z[0]) < 1e-11  # (test_fp64_window_passes_match_half_sweeps)


@pytest.mark.parametrize("graph", [0, 1])
@pytest.mark.parametrize("fold_r", [0, 1])
@pytest.mark.parametrize("shape", [(32, 32, 32), (40, 56, 24)])
def test_fp64_solve_on_window_passes(ctx, shape, fold_r, graph):
    """The solve around them: r update, (r, r) and (r, z) grouped differently, so
    heads equal to the stopping tolerance's rounding and equal iterations."""
    g = Grid3D(*shape)
    bc, _ = bc_pair("darcy_x")
    K = torch.exp(lognormal_lnK(*shape, 2.0, 5.0, 41, device=ctx.device)[0])
    heads, its = [], []
    for fuse in (0, -1):
        ws = ph.FlowWorkspace()
        ws.set_tuning(ph.FlowWorkspace.TUNE_FUSE, fuse)
        ws.set_tuning(ph.FlowWorkspace.TUNE_FOLD_R, fold_r)
        ws.set_tuning(ph.FlowWorkspace.TUNE_GRAPH, graph)
        h = ctx.zeros(g.num_cells())
        res = ph.solve_head(h, K, g, bc, ph.HeadSolveConfig.fp64_direct(1e-10, 3), ctx, ws)
        assert res.converged and res.true_residual <= 1e-10 * res.bnorm
        heads.append(h.cpu().numpy())
        its.append(res.num_iterations)
        ws.close()
    assert its[0] == its[1]
    assert rel_l2(heads[1], heads[0]) < 1e-11


@pytest.mark.parametrize("shape,mix", [
    ((16, 16, 16), "all_periodic"), ((18, 14, 10), "all_neumann"), ((2, 4, 512), "periodic_yz"),
    ((15, 13, 11), "darcy_x"), ((7, 16, 31), "all_dirichlet"), ((14, 9, 3), "all_neumann"),
    ((3, 5, 273), "darcy_x"), ((5, 2, 2), "periodic_yz")])
def test_small_level_iterations_match_oracle(ctx, shape, mix):
    """One-workgroup GSRB of a whole small level (pairs of the linear order, odd
    and even axes), 7 iterations from zero: the same sums to rounding."""
    g, og = grid_pair(*shape)
    bc, obc = bc_pair(mix)
    n = g.num_cells()
    K, r = random_K(n, 61), np.random.default_rng(62).standard_normal(n)
    cfg = ph.HeadSolveConfig(mg_levels=1, mg_coarse_iters=7)
    ws = ph.FlowWorkspace()
    M = nm.MultigridPreconditioner.build(ctx, ws, g, bc, cfg, torch.as_tensor(K).to(ctx.device))
    out = ctx.empty(n)
    M.apply(ctx, torch.as_tensor(r).to(ctx.device), out)
    ctx.synchronize()
    ref = O.gsrb_smooth_3d(og, obc, mix == "all_neumann" or mix == "all_periodic",
                           np.zeros(n), r, K, 7)
    assert rel_l2(out.cpu().numpy(), ref) < 1e-12
    ws.close()
