"""Batches whose first launch goes out before the host has the previous check's
status (residual rule, several regions): the same bits, sweeps and checks as
without."""
import numpy as np
import pytest

import tests.test_gpu_sweep_tiles as tiles
from poisson_caustic_design_amd import capi

pytestmark = pytest.mark.gpu

SIZES = [(400, 257), (131, 999), (300, 300)]


@pytest.mark.parametrize("w,h", SIZES)
@pytest.mark.parametrize("every", [7, 8, 9, 13, 40, 41])
def test_batches_equal_solves_of_one_batch_each(ctx, rng, w, h, every):
    """7: no early launch, 8: it takes the whole batch.  A solve that ends with its
    first batch has none, and starts from the same residual as the next batch."""
    b, _, p = tiles.make(rng, w, h, False)
    for n in (5 * every, 4 * every + 3, 4 * every + min(9, every)):  # last batch whole, cut short
        kw = dict(stop=capi.STOP_RESIDUAL, tol=0.0, omega=1.6, check_every=every)
        g, st = ctx.poisson_solve(b, p, capi.default_opts(max_sweeps=n, **kw))
        f = p
        for first in range(0, n, every):
            f, _ = ctx.poisson_solve(b, f, capi.default_opts(max_sweeps=min(every, n - first), **kw))
        assert st.sweeps == n and st.checks == 1 + (n + every - 1) // every
        assert np.array_equal(f, g), n


@pytest.mark.parametrize("w,h", SIZES)
def test_solves_equal_profiled_ones(ctx, rng, w, h):
    """To a tolerance, with batches of the solver's choice: a profiled context
    waits for every check."""
    b, _, p = tiles.make(rng, w, h, False)
    for tol in (1e-3, 1e-6, 1e-9):
        g, st = ctx.poisson_solve(b, p, capi.default_opts(tol=tol))
        ctx.set_profiling(True)
        try:
            f, sf = ctx.poisson_solve(b, p, capi.default_opts(tol=tol))
        finally:
            ctx.set_profiling(False)
        assert st.status == sf.status == capi.OK
        assert (st.sweeps, st.checks, st.rel_residual) == (sf.sweeps, sf.checks, sf.rel_residual)
        assert np.array_equal(f, g), tol
