"""Batches of more sweeps than one launch takes on a grid of one region (16384):
two launches, against the references of tests/test_gpu_sweep_tiles.py.  omega is
small, so that the last launch's few sweeps still move the iterate."""
import numpy as np
import pytest

import tests.test_gpu_sweep_tiles as tiles
from oracle.bind import RED_BLACK
from poisson_caustic_design_amd import capi

pytestmark = pytest.mark.gpu

K, OMEGA = 16391, 1e-3


def opts(**kw):
    return capi.default_opts(max_sweeps=K, check_every=K, stop=capi.STOP_RESIDUAL, tol=0.0,
                             omega=OMEGA, **kw)


def test_fp64(ctx, oracle, rng):
    b, _, p0 = tiles.make(rng, 23, 14, False)
    g, st = ctx.poisson_solve(b, p0, opts(precision=capi.PREC_FP64))
    ref, _ = oracle.poisson_sor(b, p0, K, max_update_tol=1e-300, ordering=RED_BLACK, omega=OMEGA)
    short, _ = oracle.poisson_sor(b, p0, K - 7, max_update_tol=1e-300, ordering=RED_BLACK,
                                  omega=OMEGA)
    # a sweep's 8 roundings of 2^-53, carried on without growth
    tol = K * 2.0 ** -50 * np.abs(ref).max()
    assert st.sweeps == K and st.checks == 2
    assert np.abs(g - ref).max() <= tol < np.abs(short - ref).max()


@pytest.mark.parametrize("w,h", [(12, 7), (9, 16)])
def test_residual_rule(ctx, rng, w, h):
    """Integers of sum zero: the residual is exact in BF16 and its mean zero, so
    the restatement works on the same numbers."""
    b = rng.integers(-8, 9, (h, w)).astype(np.float64)
    b[0, 0] -= b.sum()
    g, st = ctx.poisson_solve(b, np.zeros((h, w)), opts())
    ref = tiles.residual_rule_sweeps(b, np.zeros((h, w)), K, OMEGA)
    short = tiles.residual_rule_sweeps(b, np.zeros((h, w)), K - 7, OMEGA)
    tol = 2.0 ** -20 * np.abs(ref).max()
    assert st.sweeps == K and st.checks == 2
    assert np.abs(g - ref).max() <= tol < np.abs(short - ref).max()
