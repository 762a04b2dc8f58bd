"""Solves that start their corrections from zero without a cleared buffer: what
an earlier solve left in the buffers (here infinities and NaN, from a
right-hand side beyond FP32's range) must not reach the next one's results, on
sides that leave padding in the bricked layout and on full bricks."""
import numpy as np
import pytest

from oracle.netref import NetRef
from poisson_caustic_design_amd import capi

pytestmark = pytest.mark.gpu


def rhs(w, h):
    b = np.random.default_rng(4).standard_normal((h, w)) * 0.1
    b += np.outer(np.cos(np.pi * (np.arange(h) + 0.5) / h), np.cos(np.pi * (np.arange(w) + 0.5) / w))
    return b - b.mean()


@pytest.mark.parametrize("w,h", [(136, 136), (200, 264), (256, 256), (1000, 488)])
@pytest.mark.parametrize("form", ["residual", "max_update", "learned", "learned_mid"])
def test_what_an_earlier_solve_left_is_not_used(ctx, w, h, form):
    net = None
    kw = dict(tol=1e-5, max_sweeps=400)
    if form == "max_update":
        kw = dict(tol=1e-3, stop=capi.STOP_MAX_UPDATE, max_sweeps=400)
    elif form.startswith("learned"):
        mid = form == "learned_mid"
        net = capi.Net(ctx, capi.default_arch(levels=2, channels=[8, 8, 0, 0, 0, 0], linear=1,
                                              coarsen=8 if mid else 4, smooth_sweeps=4,
                                              out_smooth=0, mid_sweeps=4 if mid else 0))
        net.set_params(NetRef(2, (8, 8), linear=True).random_params(5, head_scale=0.05))
        ctx.set_net(net)
        kw = dict(tol=1e-12, learned_init=1, max_sweeps=24)
    try:
        b, zero = rhs(w, h), np.zeros((h, w))
        o = capi.default_opts(**kw)
        ref, st = ctx.poisson_solve(b, zero, o)
        assert np.isfinite(ref).all() and st.sweeps > 0
        for scale in (1e200, 1e305):
            ctx.poisson_solve(b * scale, zero, o, allow=(capi.OK, capi.NAN_, capi.NOT_CONVERGED))
            got, st2 = ctx.poisson_solve(b, zero, o)
            assert np.array_equal(got, ref)
            assert (st2.sweeps, st2.checks) == (st.sweeps, st.checks)
    finally:
        if net is not None:
            ctx.set_net(None)
            net.close()
