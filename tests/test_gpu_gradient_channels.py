"""Gradients of networks whose convolutions have 5, 7 or 9 and more blocks of 16
input channels, which only the input gradients on LDS tiles take: the reference and
bounds of the weight-gradient test, which every input gradient enters."""
import pytest

import tests.test_gpu_wgrad as wgrad

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("levels,channels,linear,batch,h,w", [
    (2, (24, 120), 1, 1, 10, 34), (2, (72, 88), 0, 2, 18, 12), (3, (40, 72, 56), 1, 1, 12, 36),
    (2, (128, 104), 1, 1, 8, 16)])
def test_gradient(ctx, levels, channels, linear, batch, h, w):
    wgrad.test_weight_gradient(ctx, levels, channels, linear, batch, h, w)
