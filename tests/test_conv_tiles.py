"""Convolution and weight gradient at the sizes where their launch geometry
changes: waves sharing a tile's k steps (16, 4 and 1 of them), rows that are no
multiple of 8 voxels (zero-padded groups), a last partial tile, one-row grids, and more
voxels than 64 slices of the weight gradient hold at 16 steps each. The oracle
sums in FP64 from the same BF16 operands; outputs are BF16 (2^-9 relative per
value) and the FP32 sums of up to 4e4 products agree to 1e-4."""
from __future__ import annotations

import ctypes as C

import numpy as np
import pytest
import torch

from macroflow3d_amd import _lib
from macroflow3d_amd.core import Grid3D
from oracle import cnn_oracle as CO

pytestmark = pytest.mark.gpu


def _rel(a, b):
    return float(np.linalg.norm(a - b) / np.linalg.norm(b))


@pytest.mark.parametrize("shape,cin,cout", [
    ((1, 1, 1), 64, 64), ((5, 3, 7), 16, 16), ((17, 11, 11), 32, 64),   # 16 waves a tile
    ((13, 16, 10), 64, 32), ((20, 20, 20), 16, 32),                     # 4 waves a tile
    ((23, 21, 20), 32, 16),                                             # one wave a tile
    ((40, 36, 28), 16, 16)])                                            # over 64 slices
def test_convolution_gradients_over_launch_shapes(ctx, shape, cin, cout):
    nx, ny, nz = shape
    rng = np.random.default_rng(nx + cin + cout)
    x = CO.bf16(rng.standard_normal((nz, ny, nx, cin)))
    dy = CO.bf16(rng.standard_normal((nz, ny, nx, cout)))
    w = rng.standard_normal((cout, 27, cin)) * 0.2
    g = Grid3D(nx, ny, nz).c()
    dev = lambda a, t: torch.as_tensor(np.ascontiguousarray(a), dtype=torch.float32).to(t).to(ctx.device)  # noqa: E731
    X, dY, wd = dev(x, torch.bfloat16), dev(dy, torch.bfloat16), dev(w, torch.float32)
    host = lambda t: t.float().cpu().numpy().astype(np.float64)  # noqa: E731
    print(f"convolution {shape} {cin}->{cout}", flush=True)
    Y = torch.empty((nz, ny, nx, cout), dtype=torch.bfloat16, device=ctx.device)
    _lib.call("mf3d_conv3d_forward", ctx.handle, C.byref(g), cin, cout, X.data_ptr(),
              wd.data_ptr(), None, None, 0, Y.data_ptr())
    assert _rel(host(Y), CO.conv(x, CO.bf16(w))) < 8e-3
    dX = torch.empty((nz, ny, nx, cin), dtype=torch.bfloat16, device=ctx.device)
    _lib.call("mf3d_conv3d_backward_data", ctx.handle, C.byref(g), cin, cout, dY.data_ptr(),
              wd.data_ptr(), None, dX.data_ptr())
    assert _rel(host(dX), CO.conv_bwd_data(dy, CO.bf16(w))) < 8e-3
    gw = torch.empty((cout, 27, cin), dtype=torch.float32, device=ctx.device)
    gb = torch.empty(cout, dtype=torch.float32, device=ctx.device)
    rw, rb = CO.conv_bwd_weights(x, dy)
    _lib.call("mf3d_conv3d_backward_weights", ctx.handle, C.byref(g), cin, cout, X.data_ptr(),
              dY.data_ptr(), gw.data_ptr(), gb.data_ptr())
    assert _rel(host(gw), rw) < 1e-4
    assert _rel(host(gb), rb) < 1e-4


@pytest.mark.parametrize("shape", [(9, 3, 2), (14, 4, 3), (8, 2, 2), (5, 1, 1), (24, 20, 3)])
def test_weight_gradient_of_infinite_inputs(ctx, shape):
    """An infinite input reaches the taps whose sums hold it, as an infinity, and no
    other: products outside the sums (rows' ends, past the last voxel) are 0 x 0."""
    nx, ny, nz = shape
    rng = np.random.default_rng(nx)
    x = CO.bf16(rng.standard_normal((nz, ny, nx, 16)))
    dy = CO.bf16(0.5 + rng.random((nz, ny, nx, 16)))  # positive: inf, never inf - inf
    x[0, 0, 0, 1] = x[-1, -1, -1, 2] = x[0, 0, -1, 3] = np.inf
    ref = np.zeros((16, 27, 16))
    for tap in range(27):
        d = (tap // 9 - 1, tap // 3 % 3 - 1, tap % 3 - 1)  # z, y, x
        src = tuple(slice(max(0, s), n + min(0, s)) for s, n in zip(d, (nz, ny, nx)))
        dst = tuple(slice(max(0, -s), n + min(0, -s)) for s, n in zip(d, (nz, ny, nx)))
        a, b = dy[dst].reshape(-1, 16), x[src].reshape(-1, 16)
        for c in range(16):
            ref[:, tap, c] = (a * b[:, c:c + 1]).sum(0)
    dev = lambda t: torch.as_tensor(np.ascontiguousarray(t), dtype=torch.float32).to(torch.bfloat16).to(ctx.device)  # noqa: E731
    X, dY = dev(x), dev(dy)
    g = Grid3D(nx, ny, nz).c()
    gw = torch.empty((16, 27, 16), dtype=torch.float32, device=ctx.device)
    gb = torch.empty(16, dtype=torch.float32, device=ctx.device)
    _lib.call("mf3d_conv3d_backward_weights", ctx.handle, C.byref(g), 16, 16, X.data_ptr(),
              dY.data_ptr(), gw.data_ptr(), gb.data_ptr())
    got, fin = gw.cpu().numpy().astype(np.float64), np.isfinite(ref)
    assert (~fin).any() and np.array_equal(np.isposinf(got), np.isposinf(ref))
    assert not np.isnan(got).any()
    assert np.abs(got[fin] - ref[fin]).max() < 1e-4 * np.abs(ref[fin]).max()
