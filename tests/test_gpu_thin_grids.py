"""Grids of few rows and several regions: one row of 8-row bricks, which regions of
6 rows a wave do not end on.  Against the same references and bounds as the
other sizes of the blocked sweeps."""
import pytest

import tests.test_gpu_sweep_tiles as tiles

pytestmark = pytest.mark.gpu

SIZES = [(200, 8), (180, 2), (300, 6), (1000, 7), (131, 9), (400, 13)]


@pytest.mark.parametrize("w,h", SIZES)
@pytest.mark.parametrize("k", [5, 16, 30])
def test_thin_grids(ctx, oracle, rng, w, h, k):
    tiles.test_blocked_sweeps_residual_rule(ctx, rng, w, h, k)
    tiles.test_blocked_sweeps_max_update_rule(ctx, oracle, rng, w, h, k)
