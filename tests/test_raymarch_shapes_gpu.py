"""The raymarch kernels at the edges of their tiles (8 x 8 pixels, slabs of 16 x
16 or 16 x 8 voxels) and on grids with an axis of one cell, where a sample's
corners cannot be read from one base address.

Tolerances (normalised max error against the FP64 oracle): images 1e-5,
gradients 1e-4, as for the kernels' ordinary sizes.
"""
import numpy as np
import pytest
import torch

from helpers import norm_err, scene
from oracle import oracle as orc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("grid,image", [((1, 6, 7), (8, 8)), ((7, 1, 6), (9, 7)), ((6, 7, 1), (1, 1)),
                                        ((9, 16, 16), (17, 8)), ((5, 33, 17), (7, 65))])
@pytest.mark.parametrize("channels,blend", [(1, "BEER_LAMBERT"), (2, "BEER_LAMBERT"), (4, "BEER_LAMBERT"),
                                            (4, "ALPHA"), (4, "ADDITIVE")])
@pytest.mark.parametrize("boundary,grad_mode", [("BORDER", "EXACT"), ("BORDER", "REFERENCE"), ("CLAMP", "EXACT"),
                                                ("WRAP", "REFERENCE")])
def test_tile_edges(cuda, grid, image, channels, blend, boundary, grad_mode):
    from gft.ops import raymarching_ops as ops
    if image == (1, 1) and (boundary, grad_mode) == ("BORDER", "REFERENCE"):
        pytest.skip("the only ray runs through the grid's middle, along cell centres: REFERENCE divides by weight "
                    "sums that are the rounding of 0 there")
    sc = scene(grid=grid, image=image, views=2, seed=4, channels=channels, blobs=3)
    rng = np.random.Generator(np.random.PCG64(6))
    data = (rng.uniform(0.05, 1.0, size=sc["data"].shape) * 0.05).astype(np.float32)
    cam = (sc["M"], sc["V"], sc["P"], sc["F"], sc["out_dhw"])
    ref = orc.raymarch_fwd(data, *cam, "LINEAR", boundary, blend)
    x = torch.from_numpy(data).cuda().requires_grad_(True)
    out = ops.raymarch_grid_transform(x, *cam, interpolation="LINEAR", boundary=boundary, blending_mode=blend,
                                      grad_mode=grad_mode)
    assert norm_err(out.detach().cpu().numpy(), ref) < 1e-5
    og = rng.uniform(-1, 1, size=ref.shape).astype(np.float32)
    out.backward(torch.from_numpy(og).cuda())
    gref = orc.raymarch_bwd(data, ref, og, *cam, boundary, blend, grad_mode=grad_mode)
    assert norm_err(x.grad.cpu().numpy(), gref) < 1e-4
