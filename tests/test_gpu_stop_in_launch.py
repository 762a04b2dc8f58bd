"""Max-update stops inside a batch's last launch on grids of more regions than fit
the GPU at once: the launch that decides repeats part of it while workgroups that
start later still read the words they decide by."""
import numpy as np
import pytest

import tests.test_gpu_sweep_tiles as tiles
from poisson_caustic_design_amd import capi

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("w,h", [(2048, 2048), (3001, 1999)])
def test_stop_in_a_batchs_last_launch(ctx, rng, w, h):
    """Bit-equal to the group of 5 sweeps that holds the stop, and the 5 that
    confirm it, taken with no stop."""
    b, _, p0 = tiles.make(rng, w, h, False)
    kw = dict(stop=capi.STOP_MAX_UPDATE, omega=1.5)
    mu = [np.inf]
    for n in range(1, 27):
        _, st = ctx.poisson_solve(b, p0, capi.default_opts(tol=0.0, check_every=n, max_sweeps=n,
                                                           **kw))
        mu.append(st.last_max_update)
    stops = 0
    for j in (7, 11, 13, 18, 24):
        tol = mu[j] * (1 + 1e-6)
        if min(mu[:j]) < tol:  # (an earlier sweep meets it)
            continue
        s = (j + 4) // 5 * 5
        g, st = ctx.poisson_solve(b, p0, capi.default_opts(tol=tol, check_every=s + 5, **kw))
        f, sf = ctx.poisson_solve(b, p0, capi.default_opts(tol=0.0, check_every=s, max_sweeps=s + 5,
                                                           **kw))
        if st.checks != 3:
            continue  # the confirming sweeps did not meet the rule: more batches follow
        assert st.status == capi.OK and st.last_max_update < tol
        assert np.array_equal(f, g), j
        stops += 1
    assert stops >= 3
