"""Kernel variants and dispatch branches that the ordinary sizes do not reach.

Tolerances are those of the same kernels at ordinary sizes (normalised max error
against the FP64 oracle: values 1e-5, gradients 1e-4).
"""
import numpy as np
import pytest
import torch

from helpers import norm_err, scene
from oracle import oracle as orc

pytestmark = pytest.mark.gpu


def _t(a):
    return torch.from_numpy(np.ascontiguousarray(a, dtype=np.float32)).cuda()


def _raymarch(grid, image, channels, boundary, grad_mode, views=2, filt="LINEAR"):
    from gft.ops import raymarching_ops as ops
    sc = scene(grid=grid, image=image, views=views, seed=4, channels=channels, blobs=3)
    rng = np.random.Generator(np.random.PCG64(6))
    data = (rng.uniform(0.05, 1.0, size=sc["data"].shape) * 0.05).astype(np.float32)
    cam = (sc["M"], sc["V"], sc["P"], sc["F"], sc["out_dhw"])
    ref = orc.raymarch_fwd(data, *cam, filt, boundary, "BEER_LAMBERT")
    x = _t(data).requires_grad_(grad_mode is not None)
    out = ops.raymarch_grid_transform(x, *cam, interpolation=filt, boundary=boundary, grad_mode=grad_mode or "EXACT")
    assert norm_err(out.detach().cpu().numpy(), ref) < 1e-5
    if grad_mode is None:
        return
    og = rng.uniform(-1, 1, size=ref.shape).astype(np.float32)
    out.backward(_t(og))
    gref = orc.raymarch_bwd(data, ref, og, *cam, boundary, "BEER_LAMBERT", grad_mode=grad_mode)
    assert norm_err(x.grad.cpu().numpy(), gref) < 1e-4


# the scatter's two tile sizes (EXACT 16 x 16 pixels, REFERENCE 8 x 8) on images around their edges
@pytest.mark.parametrize("image", [(1, 3), (8, 17), (15, 16), (33, 9)])
@pytest.mark.parametrize("channels", [1, 4])
@pytest.mark.parametrize("boundary,grad_mode", [("CLAMP", "REFERENCE"), ("CLAMP", "EXACT"), ("WRAP", "EXACT"),
                                                ("WRAP", "REFERENCE")])
def test_raymarch_scatter_tiles(cuda, image, channels, boundary, grad_mode):
    _raymarch((9, 17, 12), image, channels, boundary, grad_mode)


# MIN and MAX rays, whose WRAP walk of four channels asks for LDS (BORDER sums are infinite: -+FLT_MAX outside)
@pytest.mark.parametrize("boundary", ["CLAMP", "WRAP"])
@pytest.mark.parametrize("filt", ["MIN", "MAX"])
def test_raymarch_min_max_channels(cuda, boundary, filt):
    _raymarch((9, 17, 12), (17, 8), 4, boundary, None, filt=filt)


# 2^24 rows of cells: offsets no longer fit the batched reads' 24-bit products
@pytest.mark.parametrize("boundary,grad_mode", [("BORDER", "EXACT"), ("CLAMP", None)])
def test_raymarch_many_rows(cuda, boundary, grad_mode):
    _raymarch((4096, 4097, 2), (3, 2), 1, boundary, grad_mode, views=1)


# slabs of 16 x 16 x 1 voxels (4096 of them or more), ragged in x and y, the last workgroup part empty
def test_raymarch_gather_slabs(cuda):
    grid = (457, 41, 37)
    assert grid[0] * 3 * 3 >= 4096 and grid[0] * 3 * 3 % 4
    _raymarch(grid, (13, 9), 4, "BORDER", "EXACT")
