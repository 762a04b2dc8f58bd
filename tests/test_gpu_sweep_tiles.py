"""The temporally blocked sweeps at the sizes where their tiling can go wrong:
grids of one region, one cell more or less, odd sides, many tiles, several
launches.  FP64 sweeps equal the oracle's red-black iterates to FP64 rounding;
with holes (FP32 sweeps on an FP32 right-hand side) to FP32 rounding of the
update; and a max-update stop inside a launch ends at the sweep at which the
oracle stops."""
import numpy as np
import pytest

from oracle.bind import RED_BLACK
from poisson_caustic_design_amd import capi

pytestmark = pytest.mark.gpu

# one region is 128 x 64; regions at the border have no halo there
SIZES = [(2, 2), (3, 2), (2, 5), (127, 63), (128, 64), (129, 64), (128, 65), (130, 66), (131, 67),
         (257, 40), (61, 300), (333, 129), (512, 384)]


def make(rng, w, h, holes):
    b = rng.standard_normal((h, w))
    if holes:
        for _ in range(4):
            x, y = int(rng.integers(0, w)), int(rng.integers(0, h))
            b[y:y + h // 7 + 1, x:x + w // 9 + 1] = np.nan
        b[0, 0] = np.nan
    m = ~np.isnan(b)
    b[m] -= b[m].mean()
    return b, m, 0.1 * rng.standard_normal((h, w))


@pytest.mark.parametrize("w,h", SIZES)
@pytest.mark.parametrize("k", [1, 7, 33])
def test_fp64_sweeps(ctx, oracle, rng, w, h, k):
    b, _, p0 = make(rng, w, h, False)
    for stop in (capi.STOP_MAX_UPDATE, capi.STOP_RESIDUAL):
        o = capi.default_opts(max_sweeps=k, stop=stop, tol=0.0, precision=capi.PREC_FP64,
                              omega=-1.0)
        g, st = ctx.poisson_solve(b, p0, o)
        ref, _ = oracle.poisson_sor(b, p0, k, max_update_tol=1e-300, ordering=RED_BLACK)
        assert st.sweeps == k
        assert np.abs(g - ref).max() <= 1e-12 * np.abs(ref).max(), (w, h)


@pytest.mark.parametrize("w,h", [s for s in SIZES if s[0] * s[1] > 100])
@pytest.mark.parametrize("precision", [capi.PREC_FP64, capi.PREC_MIXED])
def test_sweeps_with_holes(ctx, oracle, rng, w, h, precision):
    k = 21
    b, m, p0 = make(rng, w, h, True)
    o = capi.default_opts(max_sweeps=k, stop=capi.STOP_RESIDUAL, tol=0.0, precision=precision,
                          omega=1.7, check_every=k)
    g, st = ctx.poisson_solve(b, p0, o)
    ref, _ = oracle.poisson_sor(b, p0, k, max_update_tol=1e-300, ordering=RED_BLACK, omega=1.7)
    assert st.sweeps == k and np.isnan(g[~m]).all()
    ok = m & np.isfinite(ref)  # a cell with no neighbour left divides by zero
    scale = np.abs((ref - p0)[ok]).max()
    # FP32: 2^-24 per operation, a few operations a sweep, each sweep's error
    # carried on by the next ones (no growth): 21 * 8 * 2^-24 = 1e-5
    tol = 1e-12 if precision == capi.PREC_FP64 else 1e-5
    assert np.abs((g - ref)[ok]).max() <= tol * scale, (w, h)


@pytest.mark.parametrize("w,h", [(61, 40), (128, 64), (200, 136), (333, 129)])
def test_fp64_max_update_stops_at_the_oracle_sweep(ctx, oracle, rng, w, h):
    """FP64 sweeps stop at the first sweep whose largest update is below the
    threshold, wherever in a launch it falls, and keep that sweep's iterate."""
    b, _, p0 = make(rng, w, h, False)
    for tol in (3e-2, 1e-3, 1e-4):
        o = capi.default_opts(stop=capi.STOP_MAX_UPDATE, tol=tol, precision=capi.PREC_FP64,
                              omega=-1.0)
        g, st = ctx.poisson_solve(b, p0, o)
        ref, rst = oracle.poisson_sor(b, p0, 100000, max_update_tol=tol, ordering=RED_BLACK)
        assert st.status == capi.OK and st.sweeps == rst.sweeps
        assert st.last_max_update < tol
        assert np.abs(g - ref).max() <= 1e-11 * np.abs(ref).max()
