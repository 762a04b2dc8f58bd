"""The check that takes a learned iteration's step, at the sizes where its rows
and columns can go wrong: widths that end inside a workgroup's 64 columns and on
their border, heights that end inside its rows, one to eight rows per thread.
Three iterations, stopped by the sweep limit: the reported residual is that of
the returned iterate, recomputed in numpy (FP64 rounding of sums of cells about
1e4 times the residual: below 1e-8 of it), and every step lowers the energy of
the problem (the residual itself may rise)."""
import numpy as np
import pytest

from oracle.netref import NetRef
from poisson_caustic_design_amd import capi

pytestmark = pytest.mark.gpu


def residual_and_energy(b, phi):
    p = np.pad(phi, 1, mode="edge")  # a missing neighbour counts as the cell itself
    lap = p[1:-1, :-2] + p[:-2, 1:-1] + p[1:-1, 2:] + p[2:, 1:-1] - 4 * phi
    b = b - b.mean()
    r = b - lap
    return np.linalg.norm(r - r.mean()) / np.linalg.norm(b), (phi * (b - 0.5 * lap)).sum()


# rows per thread: 1, 2 (from 2^20 cells), 4, 8 (from 2^22)
@pytest.mark.parametrize("w,h", [(136, 200), (192, 136), (264, 152), (1032, 1024), (1024, 1048),
                                 (2056, 1032), (2048, 2056)])
def test_residual_after_learned_steps(ctx, w, h):
    arch = capi.default_arch(levels=2, channels=[8, 8, 0, 0, 0, 0], linear=1, coarsen=4,
                             smooth_sweeps=4, out_smooth=0, mid_sweeps=0)
    net = capi.Net(ctx, arch)
    net.set_params(NetRef(2, (8, 8), linear=True).random_params(5, head_scale=0.05))
    rng = np.random.default_rng(2)
    b = rng.standard_normal((h, w)) + 3 * np.outer(np.cos(np.pi * (np.arange(h) + 0.5) / h),
                                                  np.cos(3 * np.pi * (np.arange(w) + 0.5) / w))
    b -= b.mean()
    ctx.set_net(net)
    last = 0.0  # the start's energy
    try:
        for its in (1, 2, 3):
            o = capi.default_opts(tol=1e-12, learned_init=1, max_sweeps=4 * its)
            phi, st = ctx.poisson_solve(b, np.zeros_like(b), o)
            assert st.learned_applied == its and st.sweeps == 4 * its
            rel, energy = residual_and_energy(b, phi)
            assert abs(st.rel_residual - rel) <= 1e-8 * rel, its
            assert energy < last, its
            last = energy
    finally:
        ctx.set_net(None)
        net.close()
