"""Convolution pairs (and head with smoothing) in one launch at the sizes where
their staging can go wrong: one 8 x 8 tile and less, images that leave partial
tiles, channel counts with and without an unrolled instantiation, patches and
weights of one round of the workgroup's loads, a part of one and several, with
and without skip inputs.  The rounding steps are those of the separate launches,
so the outputs are equal."""
import numpy as np
import pytest
import torch

from oracle.netref import NetRef
from poisson_caustic_design_amd import capi

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("out_smooth", [0, 6])
@pytest.mark.parametrize("channels,linear,batch,h,w", [
    ((8, 8), 0, 1, 2, 2), ((16, 32), 1, 2, 10, 22), ((16, 32, 32, 32), 0, 3, 8, 24),
    ((16, 16), 1, 1, 18, 34), ((32, 32, 32), 0, 1, 12, 20), ((24, 8, 24), 1, 2, 20, 12),
    ((32, 16, 32), 0, 1, 36, 28), ((64, 32), 1, 1, 14, 18), ((16, 32, 64), 1, 1, 16, 32)])
def test_paired_convolutions_equal_separate_ones(ctx, channels, linear, batch, h, w, out_smooth):
    levels = len(channels)
    arch = capi.default_arch(levels=levels, channels=list(channels) + [0] * (6 - levels),
                             linear=linear, out_smooth=out_smooth)
    net = capi.Net(ctx, arch)
    net.set_params(NetRef(levels, channels, linear=bool(linear)).random_params(11))
    x = torch.tensor(np.random.default_rng(4).standard_normal((batch, h, w)),
                     dtype=torch.float32, device="cuda:0")
    ys = []
    for fused in (True, False):
        net.set_fused_forward(fused)
        y = torch.zeros_like(x)
        torch.cuda.synchronize()
        net.forward(x.data_ptr(), y.data_ptr(), batch, h, w)
        ys.append(y.cpu().numpy())
    net.close()
    assert np.abs(ys[0]).max() > 0
    assert np.array_equal(ys[0], ys[1])


def test_resampling_of_more_rows_than_a_grid_holds(ctx):
    """2060 images of 64 rows: every resampling kernel goes round its rows.  The
    materialised forward equals the fused one, and the gradient of the mean loss
    is the mean of the quarters' gradients (whose output gradients differ by the
    exact factor 4, so every rounding to BF16 is the same) up to the order of the
    FP32 sums over 10^6 pixels: sqrt(10^6) 2^-24 = 6e-5."""
    b, h, w = 2060, 64, 8
    arch = capi.default_arch(levels=3, channels=[8, 16, 8, 0, 0, 0], linear=1, out_smooth=0)
    net = capi.Net(ctx, arch)
    net.set_params(NetRef(3, (8, 16, 8), linear=True).random_params(3))
    rng = np.random.default_rng(8)
    x, t = (torch.tensor(rng.standard_normal((b, h, w)), dtype=torch.float32, device="cuda:0")
            for _ in range(2))
    ys = []
    for fused in (True, False):
        net.set_fused_forward(fused)
        y = torch.zeros_like(x)
        torch.cuda.synchronize()
        net.forward(x.data_ptr(), y.data_ptr(), b, h, w)
        ys.append(y.cpu().numpy())
    assert np.array_equal(ys[0], ys[1])
    _, g = net.loss_grad(x.data_ptr(), t.data_ptr(), b, h, w)
    parts = []
    for q in range(4):
        i = slice(q * b // 4, (q + 1) * b // 4)
        xq, tq = x[i].contiguous(), t[i].contiguous()
        torch.cuda.synchronize()
        parts.append(net.loss_grad(xq.data_ptr(), tq.data_ptr(), b // 4, h, w)[1])
    net.close()
    mean = np.mean(parts, axis=0)
    assert np.linalg.norm(g - mean) <= 6e-5 * np.linalg.norm(mean)
