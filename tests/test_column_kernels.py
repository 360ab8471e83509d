"""Smoother, residual and operator straight from K (column_kernel) against the
oracle at the sizes where the pair march can go wrong: odd rows (a last pair of
one cell), one-cell axes, arrays at an odd offset (no 16-byte loads), several
planes per workgroup with a short last chunk, and cells of zero conductivity.
The oracle walks faces, edges and vertices as the reference does, which leaves
out cells of a one-cell axis; those shapes are compared with numpy."""
from __future__ import annotations

import numpy as np
import pytest
import torch

import oracle as O
from helpers import bc_pair, grid_pair, random_K, rel_err
from macroflow3d_amd import multigrid as mg
from macroflow3d_amd import numerics as nm
from macroflow3d_amd.core import PinSpec

pytestmark = pytest.mark.gpu

# each cell's terms are the oracle's, rounded at most a few ulp apart
TOL = 1e-12
SHAPES = [(1, 4, 3), (5, 1, 2), (7, 6, 5), (33, 8, 4), (200, 130, 91), (129, 150, 90)]


def numpy_faces(g, bc, K):
    """(conductance, neighbour index or -1) of every cell's x-, x+, .. z+ face."""
    dims = (g.nx, g.ny, g.nz)
    o = np.arange(g.num_cells())
    pos = (o % g.nx, o // g.nx % g.ny, o // (g.nx * g.ny))
    out = []
    for f, face in enumerate(bc.faces()):
        ax, step = f // 2, 1 if f % 2 else -1
        p = list(pos)
        p[ax] = (pos[ax] + step) % dims[ax]
        nb = p[0] + g.nx * (p[1] + g.ny * p[2])
        edge = pos[ax] == (dims[ax] - 1 if f % 2 else 0)
        c = 2.0 / (1.0 / K + 1.0 / K[nb])
        if face.type != 2:  # not periodic
            c = np.where(edge, 2.0 * K if face.type == 0 else 0.0, c)
            nb = np.where(edge, -1, nb)
        out.append((c, nb, edge))
    return out


def numpy_residual(g, bc, pin, x, b, K):
    F = numpy_faces(g, bc, K)
    s = sum(c * (x - np.where(nb < 0, 0.0, x[nb])) for c, nb, _ in F)
    s[0] += sum(c[0] for c, _, _ in F) * x[0] if pin else 0.0
    return b + s / g.dx ** 2


def numpy_apply(g, bc, pin, K, x):
    F = numpy_faces(g, bc, K)
    s = sum(c * (x - np.where(nb < 0, 0.0, x[nb])) for c, nb, _ in F)
    s[0] += sum(c[0] for c, _, edge in F if not edge[0]) * x[0] if pin else 0.0
    return -s / g.dx ** 2


def numpy_gsrb(g, bc, pin, x, b, K):
    F = numpy_faces(g, bc, K)
    o = np.arange(g.num_cells())
    colour = (o % g.nx + o // g.nx % g.ny + o // (g.nx * g.ny)) % 2
    d = sum(c for c, _, _ in F)
    d[0] *= 2.0 if pin else 1.0
    x = x.copy()
    for q in (0, 1):
        v = sum(c * np.where(nb < 0, 0.0, x[nb]) for c, nb, _ in F)
        x = np.where(colour == q, (v - b * g.dx ** 2) / d, x)
    return x


def dev(a, ctx, off=0):
    t = torch.empty(a.size + off, dtype=torch.float64, device=ctx.device)[off:]
    t.copy_(torch.as_tensor(a))
    return t


def host(t):
    torch.cuda.synchronize()
    return t.cpu().numpy()


@pytest.mark.parametrize("off", [0, 1])
@pytest.mark.parametrize("mix", ["darcy_x", "all_dirichlet", "periodic_yz", "all_neumann"])
@pytest.mark.parametrize("shape", SHAPES)
def test_column_kernels_match_oracle(ctx, shape, mix, off):
    g, og = grid_pair(*shape, dx=0.5)
    bc, obc = bc_pair(mix)
    n, pin = g.num_cells(), mix == "all_neumann"
    rng = np.random.default_rng(11)
    K, x, b = random_K(n, 12), rng.standard_normal(n), rng.standard_normal(n)
    Kd, xd, bd = dev(K, ctx, off), dev(x, ctx, off), dev(b, ctx, off)
    r = dev(np.zeros(n), ctx, off)
    thin = min(shape) == 1
    mg.compute_residual_3d(ctx, g, xd, bd, Kd, r, bc, PinSpec(pin))
    ref = (numpy_residual(g, bc, pin, x, b, K) if thin
           else O.compute_residual_3d(og, obc, pin, x, b, K))
    assert rel_err(host(r), ref) < TOL
    nm.VarCoeffLaplacian(g, Kd, bc, PinSpec(pin)).apply(ctx, xd, r)
    ref = numpy_apply(g, bc, pin, K, x) if thin else O.varcoeff_apply(og, obc, pin, K, x)
    assert rel_err(host(r), ref) < TOL
    # a periodic axis of odd length joins two cells of one colour: no red-black order
    if not (mix == "periodic_yz" and (shape[1] % 2 or shape[2] % 2)):
        mg.gsrb_smooth_3d(ctx, g, xd, bd, Kd, 1, bc, PinSpec(pin))
        ref = (numpy_gsrb(g, bc, pin, x, b, K) if thin
               else O.gsrb_smooth_3d(og, obc, pin, x, b, K, 1))
        assert rel_err(host(xd), ref) < TOL


def test_cells_of_zero_conductivity_close_their_faces(ctx):
    g, og = grid_pair(10, 6, 4)
    bc, obc = bc_pair("darcy_x")
    n = g.num_cells()
    rng = np.random.default_rng(13)
    K, x, b = random_K(n, 14), rng.standard_normal(n), rng.standard_normal(n)
    K[[0, 33, 34, 44, n - 1]] = 0.0
    with np.errstate(divide="ignore"):
        ro, yo = O.compute_residual_3d(og, obc, False, x, b, K), O.varcoeff_apply(og, obc, False, K, x)
    r = ctx.empty(n)
    mg.compute_residual_3d(ctx, g, dev(x, ctx), dev(b, ctx), dev(K, ctx), r, bc)
    assert rel_err(host(r), ro) < TOL
    nm.VarCoeffLaplacian(g, dev(K, ctx), bc).apply(ctx, dev(x, ctx), r)
    assert rel_err(host(r), yo) < TOL


# planes of few columns (several chunks a workgroup), either side of the 1024 columns from
# which a workgroup stays in one chunk; 4x4x140000: two planes a thread
@pytest.mark.parametrize("off", [0, 1])
@pytest.mark.parametrize("mix", ["darcy_x", "periodic_yz", "all_neumann"])
@pytest.mark.parametrize("shape", [(1, 1, 5000), (2, 2, 3000), (3, 4, 700), (1, 64, 64),
                                   (511, 4, 6), (510, 4, 6), (511, 3, 10), (4, 4, 140000)])
def test_narrow_columns_match_oracle(ctx, shape, mix, off):
    test_column_kernels_match_oracle(ctx, shape, mix, off)


def test_smoother_meets_cells_of_zero_conductivity(ctx):
    """Such a cell has no diagonal: its value and, through 0 times that, its neighbours'
    are what IEEE division and multiplication make them; all others are untouched."""
    g, og = grid_pair(10, 6, 4)
    bc, obc = bc_pair("darcy_x")
    n = g.num_cells()
    rng = np.random.default_rng(13)
    K, x, b = random_K(n, 14), rng.standard_normal(n), rng.standard_normal(n)
    K[[0, 33, 34, 44, n - 1]] = 0.0
    b[33] = 0.0
    with np.errstate(all="ignore"):
        ref = O.gsrb_smooth_3d(og, obc, False, x, b, K, 1)
    xd = dev(x, ctx)
    mg.gsrb_smooth_3d(ctx, g, xd, dev(b, ctx), dev(K, ctx), 1, bc)
    got, ok = host(xd), np.isfinite(ref)
    assert 0 < (~ok).sum() < n // 4
    assert np.array_equal(got[~ok], ref[~ok], equal_nan=True)
    assert rel_err(got[ok], ref[ok]) < TOL


def _exact(shape, bc, K, x, b):
    """(residual, x after one GSRB iteration) in the kernel's own steps, each rounded
    once: fractions, rounded by float()."""
    from fractions import Fraction as Q
    nx, ny, nz = shape
    at = {c: c[0] + nx * (c[1] + ny * c[2]) for c in np.ndindex(*shape)}
    ik = [float(1 / Q(k)) for k in K]
    types = [f.type for f in bc.faces()]

    def sides(c):  # (neighbour or None, Dirichlet) for x+, x-, y+, y-, z+, z-
        for ax in range(3):
            for up in (1, 0):
                q = list(c)
                q[ax] += 1 if up else -1
                if 0 <= q[ax] < shape[ax]:
                    yield at[tuple(q)], False
                elif types[2 * ax + up] == 2:
                    q[ax] %= shape[ax]
                    yield at[tuple(q)], False
                else:
                    yield None, types[2 * ax + up] == 0

    def fma(a, u, v):
        return float(Q(a) * Q(u) + Q(v))

    res = np.empty(len(K))
    for c, o in at.items():
        r = 0.0
        sd = list(sides(c))
        for nb, dirichlet in (sd[0], sd[2], sd[1], sd[3], sd[4], sd[5]):
            if nb is None:
                r = fma(2.0 * K[o] if dirichlet else 0.0, x[o], r)
            else:
                r = float(Q(r) + Q(float(Q(2.0 * (x[o] - x[nb])) / Q(ik[o] + ik[nb]))))
        res[o] = b[o] + r
    y = np.array(x)
    for colour in (0, 1):
        for c, o in at.items():
            if sum(c) % 2 != colour:
                continue
            f = [(2.0 * K[o] if d else 0.0) if nb is None else 2.0 * float(1 / Q(ik[o] + ik[nb]))
                 for nb, d in sides(c)]
            v = [0.0 if nb is None else y[nb] for nb, _ in sides(c)]
            n, d = v[0] * f[0], f[0]
            for q in range(1, 6):
                n, d = fma(v[q], f[q], n), d + f[q]
            y[o] = float(Q(fma(-b[o], 1.0, n)) / Q(d))
    return res, y


@pytest.mark.parametrize("mix", ["darcy_x", "all_dirichlet", "periodic_yz"])
@pytest.mark.parametrize("shape", [(6, 4, 4), (7, 4, 6), (12, 6, 2)])
def test_one_rounding_a_term(ctx, shape, mix):
    """Reciprocals and quotients are the rounded ones, and a term of the smoother's sum
    and of a Dirichlet face joins by one multiply-add: bit for bit."""
    g, _ = grid_pair(*shape)
    bc, _ = bc_pair(mix)
    n = g.num_cells()
    rng = np.random.default_rng(17)
    K, x, b = random_K(n, 18, 2.0), rng.standard_normal(n), rng.standard_normal(n)
    ref, y = _exact(shape, bc, K.tolist(), x.tolist(), b.tolist())
    r, xd = ctx.empty(n), dev(x, ctx)
    mg.compute_residual_3d(ctx, g, xd, dev(b, ctx), dev(K, ctx), r, bc)
    assert np.array_equal(host(r), ref)
    mg.gsrb_smooth_3d(ctx, g, xd, dev(b, ctx), dev(K, ctx), 1, bc)
    assert np.array_equal(host(xd), y)
