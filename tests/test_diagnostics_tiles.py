"""Velocity diagnostics at the edges of the kernel's tiles (64 x 14 columns, chunks
of planes): exact multiples, one cell more and less, one plane a chunk and many."""
from __future__ import annotations

import pytest

import test_diagnostics as td

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(64, 14, 9), (65, 15, 3), (63, 13, 130), (128, 28, 40),
                                   (129, 1, 5), (3, 200, 4), (200, 3, 1)])
def test_diagnostics_tile_edges(ctx, shape):
    td.test_diagnostics_match_oracle(ctx, shape)
