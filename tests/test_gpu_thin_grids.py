"""Grids of few rows and several regions: one row of 8-row bricks, which regions of
6 rows a wave do not end on.  Against the same references and bounds as the
other sizes of the blocked sweeps.  And grids so long that the words of the
max-update rule outgrow what few reduction blocks leave beside their sums."""
import numpy as np
import pytest

import tests.test_gpu_sweep_tiles as tiles
import tests.test_zz_no_alloc as noalloc
from poisson_caustic_design_amd import capi

pytestmark = pytest.mark.gpu

SIZES = [(200, 8), (180, 2), (300, 6), (1000, 7), (131, 9), (400, 13)]


@pytest.mark.parametrize("w,h", SIZES)
@pytest.mark.parametrize("k", [5, 16, 30])
def test_thin_grids(ctx, oracle, rng, w, h, k):
    tiles.test_blocked_sweeps_residual_rule(ctx, rng, w, h, k)
    tiles.test_blocked_sweeps_max_update_rule(ctx, oracle, rng, w, h, k)


LONG = [(60000, 3), (45001, 4)]


@pytest.mark.parametrize("w,h", LONG)
def test_long_grids_max_update_rule(ctx, oracle, rng, w, h):
    tiles.test_blocked_sweeps_max_update_rule(ctx, oracle, rng, w, h, 33)
    tiles.test_fp64_sweeps(ctx, oracle, rng, w, h, 33)
    tiles.test_max_update_stop_inside_a_launch_keeps_that_iterate(ctx, rng, w, h)


@pytest.mark.parametrize("w,h", LONG)
@pytest.mark.parametrize("precision", [capi.PREC_MIXED, capi.PREC_FP64])
def test_long_grids_without_allocation(ctx, rng, w, h, precision):
    """The same kernels on the static scratch, whose solve state lies behind the
    partials: bit-equal to the allocating solve."""
    b, _, p0 = tiles.make(rng, w, h, False)
    o = capi.default_opts(stop=capi.STOP_MAX_UPDATE, tol=0.0, max_sweeps=40, omega=1.5,
                          precision=precision)
    L = capi.load()
    (ra, pa, sa), (rn, pn, sn) = [noalloc.solve(ctx, f, b, p0, o) for f in
                                  (L.cd_poisson_solve_device, L.cd_poisson_solve_device_noalloc)]
    assert ra == rn == capi.NOT_CONVERGED and sa.sweeps == sn.sweeps == 40
    assert np.array_equal(pa, pn) and sa.last_max_update == sn.last_max_update > 0
