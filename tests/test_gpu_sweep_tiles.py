"""The temporally blocked sweeps at the sizes where their tiling can go wrong:
grids of one region, one cell more or less, odd sides, many tiles, several
launches.  FP64 sweeps equal the oracle's red-black iterates to FP64 rounding;
with holes (FP32 sweeps on an FP32 right-hand side) to FP32 rounding of the
update, on the bricked layout to the rounding of its right-hand side; and a
max-update stop inside a launch ends at the sweep at which the oracle stops, or
at the iterate of the same number of sweeps taken without a stop."""
import numpy as np
import pytest
import torch

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


def bf16(a):
    u = np.asarray(a, dtype=np.float32).view(np.uint32).astype(np.uint64)
    return ((((u + 0x7FFF + ((u >> 16) & 1)) >> 16) << 16).astype(np.uint32)).view(np.float32)


def residual_rule_sweeps(b, p0, k, omega):
    """One batch of k sweeps under the residual rule, restated in numpy: FP32 on a
    correction e of p0, right-hand side the FP64 residual rounded to BF16, the
    update v' = oc S + ((1 - omega) v + nq), nq = (mean - r) oc, with fused
    multiply-adds (long double, rounded once to FP32)."""
    h, w = b.shape
    f32, ld = np.float32, np.longdouble
    pad = lambda a: np.pad(a, 1)
    one = pad(np.ones((h, w)))
    nb = [(slice(1, -1), slice(0, -2)), (slice(0, -2), slice(1, -1)),   # left, up
          (slice(1, -1), slice(2, None)), (slice(2, None), slice(1, -1))]  # right, down
    cnt = sum(one[n] for n in nb)
    q = pad(p0)
    r = (b - b.mean()) - (((q[nb[0]] + q[nb[1]]) + q[nb[2]]) + q[nb[3]] - cnt * p0)
    om = f32(omega)
    oc = np.choose(4 - cnt.astype(int), [om / f32(4), om / f32(3), om / f32(2)])
    nq = (f32(r.mean()) - bf16(r)) * oc
    c1 = f32(1) - f32(4) * (om / f32(4))
    fma = lambda a, x, c: (a.astype(ld) * x.astype(ld) + c.astype(ld)).astype(f32)
    e = np.zeros((h, w), dtype=f32)
    colour = np.add.outer(np.arange(h), np.arange(w)) & 1
    for _ in range(k):
        for c in (0, 1):
            q = pad(e)
            s = ((q[nb[0]] + q[nb[1]]) + q[nb[2]]) + q[nb[3]]
            v = fma(oc, s, fma(np.full_like(e, c1), e, nq))
            e = np.where(colour == c, v, e)
    return p0 + e.astype(np.float64)


# regions of 64, 96 and 128 rows; launches of up to 19 sweeps
BLOCKED = SIZES + [(128, 96), (129, 97), (128, 128), (127, 129), (640, 1030), (1024, 700)]


@pytest.mark.parametrize("w,h", BLOCKED)
@pytest.mark.parametrize("k", [3, 16, 41])
def test_blocked_sweeps_residual_rule(ctx, rng, w, h, k):
    """The sweeps equal their restatement to a few FP32 roundings of the update
    (the mean of r, about 1e-17, and ties of its BF16 rounding are all that can
    differ; an indexing or ordering error is O(1))."""
    b, _, p0 = make(rng, w, h, False)
    o = capi.default_opts(max_sweeps=k, stop=capi.STOP_RESIDUAL, tol=0.0, omega=1.6,
                          check_every=k)
    g, st = ctx.poisson_solve(b, p0, o)
    ref = residual_rule_sweeps(b, p0, k, 1.6)
    assert st.sweeps == k
    assert np.abs(g - ref).max() <= 2.0 ** -20 * np.abs(ref - p0).max(), (w, h)


@pytest.mark.parametrize("w,h", BLOCKED)
@pytest.mark.parametrize("k", [3, 16, 41])
def test_blocked_sweeps_max_update_rule(ctx, oracle, rng, w, h, k):
    """FP32 sweeps on an FP32 right-hand side: 2^-24 per operation, about 8
    operations a sweep."""
    b, _, p0 = make(rng, w, h, False)
    o = capi.default_opts(max_sweeps=k, stop=capi.STOP_MAX_UPDATE, tol=0.0, omega=1.6,
                          check_every=k)
    g, st = ctx.poisson_solve(b, p0, o)
    ref, _ = oracle.poisson_sor(b, p0, k, max_update_tol=1e-300, ordering=RED_BLACK, omega=1.6)
    assert st.sweeps == k
    scale = np.abs(ref - p0).max()
    assert np.abs(g - ref).max() <= 8 * k * 2.0 ** -24 * scale, (w, h)


# odd and even sides over several regions: border cells in a region's last lane
# or before it, a wave's last row on, above or below the grid's last row, waves
# that sit out a launch's later sweeps on one side and on both
@pytest.mark.parametrize("w,h", [(255, 301), (254, 302), (400, 257), (129, 999), (300, 130)])
def test_blocked_sweeps_borders(ctx, oracle, rng, w, h):
    test_blocked_sweeps_residual_rule(ctx, rng, w, h, 45)
    test_blocked_sweeps_max_update_rule(ctx, oracle, rng, w, h, 45)


@pytest.mark.parametrize("w,h", [(61, 40), (128, 64), (200, 136), (333, 129), (640, 520)])
def test_max_update_stop_inside_a_launch_keeps_that_iterate(ctx, rng, w, h):
    """The first sweep below the threshold, found from runs of 1, 2, ... sweeps,
    ends the batch with its group of 5, wherever in a launch that falls: the
    result is bit-equal to that many sweeps taken with no stop (tolerance 0) and
    the 5 that confirm it (whatever the stop, the reported count is the
    enqueued batch's)."""
    b, _, p0 = make(rng, w, h, False)
    kw = dict(stop=capi.STOP_MAX_UPDATE, omega=1.5)
    mu = [np.inf]
    while mu[-1] >= 1e-2 and len(mu) < 200:
        n = len(mu)
        _, st = ctx.poisson_solve(b, p0, capi.default_opts(tol=0.0, check_every=n, max_sweeps=n,
                                                           **kw))
        mu.append(st.last_max_update)
    stops = set()
    for tol in np.geomspace(mu[3], min(mu) * 1.01, 12):
        j = next(i for i, m in enumerate(mu) if m < tol)
        s = (j + 4) // 5 * 5
        g, st = ctx.poisson_solve(b, p0, capi.default_opts(tol=tol, check_every=1000, **kw))
        if st.checks != 3:
            continue  # the confirming sweeps did not meet the rule: more batches follow
        f, _ = ctx.poisson_solve(b, p0, capi.default_opts(tol=0.0, check_every=s, max_sweeps=s + 5,
                                                          **kw))
        assert st.status == capi.OK and st.last_max_update < tol
        assert np.array_equal(f, g), (tol, j)
        stops.add(s)
    assert len(stops) >= 3


# grids of one region run whole solves in one launch; one cell more does not
REGION = [(2, 2), (5, 3), (31, 32), (64, 33), (100, 64), (127, 65), (128, 128)]


@pytest.mark.parametrize("w,h", REGION)
def test_one_region_solves_match_larger_route(ctx, rng, w, h):
    """The one-launch solve against the solve of the same problem through the
    hole-mask route's FP64 sweeps: both end at the tolerance, so the mean-free
    solutions agree to it (the residual's factor on the error is below
    (n / pi)^2 / 4 < 420 at 128)."""
    b, _, p0 = make(rng, w, h, False)
    tol = 1e-10
    g, st = ctx.poisson_solve(b, p0, capi.default_opts(tol=tol))
    ref, sr = ctx.poisson_solve(b, p0, capi.default_opts(tol=tol, precision=capi.PREC_FP64))
    assert st.status == sr.status == capi.OK and st.rel_residual <= tol
    assert st.checks >= 2 and st.initial_rel_residual > tol
    d = (g - g.mean()) - (ref - ref.mean())
    assert np.abs(d).max() <= 2 * 420 * tol * np.linalg.norm(b)


@pytest.mark.parametrize("w,h", REGION + [(128, 3), (3, 128), (65, 5), (64, 64), (96, 97)])
@pytest.mark.parametrize("stop,tol", [(capi.STOP_RESIDUAL, 1e-7), (capi.STOP_MAX_UPDATE, 1e-5)])
def test_one_region_solves_equal_the_launches(ctx, rng, w, h, stop, tol):
    """Sweeps, checks, statistics and result of the one-launch solve are those of
    separate launches, bit for bit (which a context with a training-pair capture
    of another geometry takes)."""
    b, _, p0 = make(rng, w, h, False)
    runs = []
    for every, cap in ((0, 100000), (13, 1000)):
        o = capi.default_opts(tol=tol, stop=stop, check_every=every, max_sweeps=cap)
        runs.append(ctx.poisson_solve(b, p0, o))
    x = torch.zeros(16, device="cuda:0")
    ctx.set_capture(x.data_ptr(), x.data_ptr(), 1, 4, 4, 64, 1)
    try:
        for (every, cap), (g, st) in zip(((0, 100000), (13, 1000)), runs):
            o = capi.default_opts(tol=tol, stop=stop, check_every=every, max_sweeps=cap)
            f, sf = ctx.poisson_solve(b, p0, o)
            assert np.array_equal(f, g)
            for k in ("status", "sweeps", "checks", "rel_residual", "initial_rel_residual",
                      "last_max_update"):
                assert getattr(sf, k) == getattr(st, k), k
    finally:
        ctx.clear_capture()


def test_one_region_solve_statuses(ctx, rng):
    b, _, p0 = make(rng, 40, 30, False)
    # cap, in the middle of a batch and of a group
    for stop in (capi.STOP_RESIDUAL, capi.STOP_MAX_UPDATE):
        _, st = ctx.poisson_solve(b, p0, capi.default_opts(tol=1e-14, stop=stop, max_sweeps=33))
        assert st.status == capi.NOT_CONVERGED and st.sweeps == 33
    # no sweeps at all leave the start as it is
    g, st = ctx.poisson_solve(b, p0, capi.default_opts(max_sweeps=0))
    assert st.status == capi.NOT_CONVERGED and st.sweeps == 0 and np.array_equal(g, p0)
    # non-finite values end the solve as such
    bad = p0.copy()
    bad[3, 4] = np.inf
    _, st = ctx.poisson_solve(b, bad, capi.default_opts(), allow=(capi.NAN_,))
    assert st.status == capi.NAN_
    # more sweeps than one launch takes: it goes on from its last check
    g, st = ctx.poisson_solve(b, p0, capi.default_opts(tol=0.0, max_sweeps=40000, check_every=1000))
    assert st.status == capi.NOT_CONVERGED and st.sweeps == 40000 and st.checks == 41
    ref, _ = ctx.poisson_solve(b, p0, capi.default_opts(tol=1e-12, precision=capi.PREC_FP64))
    d = (g - g.mean()) - (ref - ref.mean())
    assert np.abs(d).max() <= 1e-9 * np.abs(ref).max()
    # holes leave it for the route that handles them, the start still in place
    b[4, 5] = np.nan
    g, st = ctx.poisson_solve(b, p0, capi.default_opts(tol=1e-9))
    assert st.status == capi.OK and np.isnan(g).sum() == 1
