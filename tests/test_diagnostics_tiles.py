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


# tiles of 4 rows (all of them held), 8 (all, 6 stored) and 16 (all, 14 stored)
@pytest.mark.parametrize("shape", [(65, 4, 37), (70, 3, 9), (66, 5, 7), (64, 8, 40), (40, 9, 6),
                                   (61, 7, 300), (1000, 14, 70), (130, 16, 80), (180, 150, 4),
                                   (3, 1145, 3), (1, 1, 1), (2, 1, 4000), (5, 6, 3000)])
def test_diagnostics_tile_heights(ctx, shape):
    td.test_diagnostics_match_oracle(ctx, shape)
