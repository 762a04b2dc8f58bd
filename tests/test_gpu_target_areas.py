"""Target areas (quads of the regular mesh clipped to pixel squares) where the
clipping can go wrong: pixel sides that run through mesh lines, pixels larger than a
cell, cells of many pixels, meshes that are not square, the smallest mesh; against
the oracle.  An area is a sum of products of coordinates up to the mesh's size W
that cancel to cells of W^2/M^2: 8 roundings of 2^-53 W^2 each are the bound."""
import numpy as np
import pytest

from oracle.bind import OracleDesign
from poisson_caustic_design_amd import capi

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mx,my,nx,ny,W", [(2, 2, 2, 2, 1.0), (2, 2, 7, 7, 0.5), (9, 9, 8, 8, 1.0),
                                           (9, 9, 16, 16, 0.3), (9, 9, 64, 64, 2.0),
                                           (33, 33, 13, 13, 1.0), (41, 41, 163, 163, 0.7),
                                           (30, 20, 120, 80, 1.5), (65, 64, 257, 253, 1.0)])
def test_target_areas(ctx, oracle, mx, my, nx, ny, W):
    H = W * ny / nx
    img = np.random.default_rng(mx * nx).random((ny, nx))
    cd = capi.CausticDesign(ctx)
    cd.set_mesh_resolution(mx, my)
    cd.set_domain_resolution(nx, ny)
    cd.set_mesh_size(W, H)
    cd.set_lens_focal_length(1.5)
    cd.set_lens_thickness(0.1)
    cd.initialize_solvers(img)
    od = OracleDesign(oracle, mx, my, nx, ny, W, H, 1.5)
    od.init(img)
    ref = od.vec(2)
    assert np.abs(cd.target_areas - ref).max() <= 8 * 2.0**-53 * mx * my * np.abs(ref).max()
    cd.close()
