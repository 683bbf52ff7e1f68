"""The resampling kernels at the edges of their tiles: output cells go 8 x 8 x 8
(or 8 x 4 x 8) to a workgroup, and the mip pyramid is built from tiles of 32 x
16 x 16 cells, several levels at a time.

Tolerances (normalised max error): 1e-5 of the FP64 oracle for samples; 1e-6
for a pyramid, whose levels are three halved sums each (a relative error below
2^-23 per sum, 18 sums at level 6 of positive cells).
"""
import numpy as np
import pytest
import torch

from helpers import norm_err, ortho_camera, scene
from oracle import oracle as orc

pytestmark = pytest.mark.gpu

COORDS = ["TRANSFORM_LINDEPTH", "TRANSFORM", "TRANSFORM_LINDEPTH_REVERSE", "TRANSFORM_REVERSE"]


def _ops():
    from gft.ops import sampling_ops
    return sampling_ops


def _camera(depth, image, proj):
    grid = (10, 18, 14)
    sc = scene(grid=grid, image=image, views=2, seed=3)
    if proj == "ortho":
        from gft.camera import camera_params_batch
        cams = [ortho_camera(grid, image, depth, yaw=y) for y in (10.0, 50.0)]
        sc["V"], sc["P"], sc["F"] = camera_params_batch(cams)
    return sc


@pytest.mark.parametrize("shape", [(1, 1, 1), (7, 5, 9), (9, 8, 16), (16, 9, 33), (41, 17, 8)])
@pytest.mark.parametrize("coord,boundary,mips,proj", [(c, b, m, p) for c in COORDS for b, m, p in (
    ("BORDER", 0, "perspective"), ("BORDER", 3, "perspective"), ("CLAMP", 2, "perspective"), ("BORDER", 2, "ortho"))
    if (c, p) != ("TRANSFORM_LINDEPTH_REVERSE", "ortho")])
def test_transform_tile_edges(cuda, shape, coord, boundary, mips, proj):
    sc = _camera(shape[0], shape[1:], proj)
    rng = np.random.Generator(np.random.PCG64(11))
    vol = (12, 16, 14) if coord.endswith("REVERSE") else (10, 18, 14)
    data = rng.uniform(0.0, 1.0, size=(1,) + vol + (2,)).astype(np.float32)
    kw = dict(interpolation="LINEAR", boundary=boundary, mipmapping="LINEAR" if mips else "NONE", num_mipmaps=mips,
              coordinate_mode=coord)
    got = _ops().sample_grid_transform(torch.from_numpy(data).cuda(), sc["M"], sc["V"], sc["P"], sc["F"], shape,
                                       **kw).cpu().numpy()
    ref = orc.sample_transform_fwd(data, sc["M"], sc["V"], sc["P"], sc["F"], shape, prec=1, **kw)
    assert np.isfinite(got).all()
    assert norm_err(got, ref) < 1e-5


@pytest.mark.parametrize("shape", [(1, 1, 2), (2, 3, 5), (15, 16, 31), (16, 16, 32), (17, 33, 65), (64, 34, 130)])
@pytest.mark.parametrize("batch,channels,levels", [(1, 1, 1), (3, 1, 4), (2, 2, 6), (1, 4, 5)])
def test_pyramid_tile_edges(cuda, shape, batch, channels, levels):
    rng = np.random.Generator(np.random.PCG64(5))
    data = rng.uniform(0.1, 1.0, size=(batch,) + shape + (channels,)).astype(np.float32)
    got = _ops().build_mips(torch.from_numpy(data).cuda(), levels)
    usable = min(levels, min(shape).bit_length() - 1)
    assert len(got) == usable
    for b in range(batch):
        for g, r in zip(got, orc.build_mips(data[b], usable)):
            assert norm_err(g[b].cpu().numpy(), r) < 1e-6
