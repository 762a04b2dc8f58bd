"""The weight-gradient kernel at the sizes where its tiling can go wrong: 8 x 32
pixel tiles against images that are smaller, larger and no multiple of them,
input channels of one to eight blocks of 16 with and without a remainder, output
channels of half a block to four, linear and with ReLU masks, batches.

The reference's activations are rounded to BF16 as the kernels store them; its
gradients are not, so each of the up to 13 layers a gradient passes adds one
2^-9 rounding per element: 2^-9 sqrt(13) = 0.7 % if independent, 2 % allowed
over the whole gradient and 6 % (a block may have passed few independent
elements) on every convolution's own block, where an indexing error is O(1)."""
import numpy as np
import pytest
import torch

from oracle.netref import NetRef
from poisson_caustic_design_amd import capi

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("levels,channels,linear,batch,h,w", [
    (2, (8, 16), 1, 1, 2, 2), (2, (8, 8), 1, 3, 6, 34), (2, (16, 24), 0, 2, 18, 66),
    (3, (8, 16, 16), 0, 1, 12, 100), (2, (32, 64), 1, 1, 8, 32), (2, (64, 64), 0, 1, 10, 40),
    (4, (16, 32, 32, 32), 1, 2, 40, 72), (4, (16, 32, 64, 64), 1, 1, 64, 64)])
def test_weight_gradient(ctx, levels, channels, linear, batch, h, w):
    arch = capi.default_arch(levels=levels, channels=list(channels) + [0] * (6 - len(channels)),
                             linear=linear, out_smooth=0)
    net = capi.Net(ctx, arch)
    ref = NetRef(levels, channels, linear=bool(linear))
    net.set_params(ref.random_params(7))
    p = net.get_params().astype(np.float64)
    rng = np.random.default_rng(1)
    x, t = rng.standard_normal((batch, h, w)), 0.3 * rng.standard_normal((batch, h, w))
    dx = torch.tensor(x, dtype=torch.float32, device="cuda:0")
    dt = torch.tensor(t, dtype=torch.float32, device="cuda:0")
    torch.cuda.synchronize()
    _, g = net.loss_grad(dx.data_ptr(), dt.data_ptr(), batch, h, w)
    _, gr = ref.loss_grad(p, x, t, emulate_bf16=True)
    net.close()
    assert np.linalg.norm(g - gr) <= 2e-2 * np.linalg.norm(gr)
    for cv in ref.convs:
        a, b = (v[cv.woff:cv.woff + cv.nparam] for v in (g, gr))
        assert np.linalg.norm(a - b) <= 6e-2 * np.linalg.norm(b), (cv.level, cv.c1, cv.c2, cv.coutA)
