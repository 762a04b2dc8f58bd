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
