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


def _raymarch(grid, image, channels, boundary, grad_mode, views=2, filt="LINEAR", tol=(1e-5, 1e-4)):
    from gft.ops import raymarching_ops as ops
    sc = scene(grid=grid, image=image, views=views, seed=4, channels=channels, blobs=3)
    rng = np.random.Generator(np.random.PCG64(6))
    data = (rng.uniform(0.05, 1.0, size=sc["data"].shape) * 0.05).astype(np.float32)
    if filt == "MIN":
        data = -data  # the sampler's minimum includes 0
    cam = (sc["M"], sc["V"], sc["P"], sc["F"], sc["out_dhw"])
    ref = orc.raymarch_fwd(data, *cam, filt, boundary, "BEER_LAMBERT")
    x = _t(data).requires_grad_(grad_mode is not None)
    out = ops.raymarch_grid_transform(x, *cam, interpolation=filt, boundary=boundary, grad_mode=grad_mode or "EXACT")
    assert ref.any() and norm_err(out.detach().cpu().numpy(), ref) < tol[0]
    if grad_mode is None:
        return
    og = rng.uniform(-1, 1, size=ref.shape).astype(np.float32)
    out.backward(_t(og))
    gref = orc.raymarch_bwd(data, ref, og, *cam, boundary, "BEER_LAMBERT", grad_mode=grad_mode)
    assert gref.any() and norm_err(x.grad.cpu().numpy(), gref) < tol[1]


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


# 2^24 rows of cells: offsets no longer fit the batched reads' 24-bit products.
# (An odd image, whose middle pixels' rays run along the grid. Positions round by up
# to 2^-11 cells in each of the map's three additions, and a tap with its three axes.)
kLongRays = 9 * 2.0 ** -11


@pytest.mark.parametrize("boundary,grad_mode", [("BORDER", "EXACT"), ("CLAMP", None)])
def test_raymarch_many_rows(cuda, boundary, grad_mode):
    _raymarch((4096, 4097, 2), (3, 3), 1, boundary, grad_mode, views=1, tol=(kLongRays, kLongRays))


# slabs of 16 x 16 x 1 voxels (4096 of them or more), ragged in x and y, the last workgroup part empty
def test_raymarch_gather_slabs(cuda):
    grid = (457, 41, 37)
    assert grid[0] * 3 * 3 >= 4096 and grid[0] * 3 * 3 % 4
    _raymarch(grid, (13, 9), 4, "BORDER", "EXACT")


def _smooth(shape, channels):
    """Smooth positive cells that vanish at the faces, so that a sample a rounding
    away from a face or a cell changes by far less than the tolerance."""
    axes = [np.sin(np.pi * (np.arange(n) + 0.5) / n) ** 2 for n in shape]
    d = axes[0][:, None, None] * axes[1][:, None] * axes[2]
    return (d[None, ..., None] * (1.0 + 0.25 * np.arange(channels))).astype(np.float32)


# resample layouts: rows, and tiles of 8 x 8 x 8 cells from a 4 MB grid, 2^18
# output cells and 24 cells an axis on, where not two of CLAMP, a reverse map and
# mips meet; ragged in every axis. Values 1e-5 (the field's slope is below 0.13 a
# cell, positions of 100 cells err by 1e-5).
RESAMPLES = [(c, g, o, cm, bm, m) for c, g, o in (
    (4, (64, 65, 67), (66, 61, 67)), (4, (64, 65, 67), (63, 61, 63)), (4, (64, 65, 67), (23, 120, 99)),
    (4, (62, 63, 61), (66, 61, 67)), (1, (104, 101, 101), (25, 101, 109)), (1, (104, 101, 101), (152, 148, 151)),
    (2, (81, 80, 82), (24, 91, 131))) for cm, bm, m in (
    ("TRANSFORM_LINDEPTH", "BORDER", 0), ("TRANSFORM", "CLAMP", 0), ("TRANSFORM_LINDEPTH", "BORDER", 3),
    ("TRANSFORM_REVERSE", "CLAMP", 0), ("TRANSFORM_LINDEPTH_REVERSE", "BORDER", 0))]


@pytest.mark.parametrize("channels,grid,out,coord,boundary,mips", RESAMPLES)
def test_resample_layouts(cuda, channels, grid, out, coord, boundary, mips):
    from gft.ops import sampling_ops as ops
    sc = scene(grid=(40, 44, 42) if coord.endswith("REVERSE") else grid, image=out[1:], views=2, seed=3)
    data = _smooth(grid, channels)
    cam = (sc["M"], sc["V"], sc["P"], sc["F"])
    kw = dict(interpolation="LINEAR", boundary=boundary, mipmapping="LINEAR" if mips else "NONE", num_mipmaps=mips,
              coordinate_mode=coord)
    got = ops.sample_grid_transform(_t(data), *cam, out, **kw).cpu().numpy()
    assert norm_err(got, orc.sample_transform_fwd(data, *cam, out, prec=1, **kw)) < 1e-5


# view sums: tiles for several channels or views, rows for one scalar view or a thin grid
@pytest.mark.parametrize("channels,views,grid", [(1, 1, (26, 25, 27)), (1, 2, (26, 25, 27)), (4, 1, (26, 25, 27)),
                                                 (4, 2, (23, 25, 27)), (2, 10, (24, 33, 24))])
@pytest.mark.parametrize("boundary,mips", [("BORDER", 0), ("CLAMP", 0), ("BORDER", 2)])
def test_view_sum_layouts(cuda, channels, views, grid, boundary, mips):
    from gft.ops import sampling_ops as ops
    sc = scene(grid=grid, image=(19, 22), views=views, seed=3)
    og = np.stack([_smooth((17, 19, 22), channels)[0] * (1.0 + v) for v in range(views)])[None]
    cam = (sc["M"], sc["V"], sc["P"], sc["F"])
    kw = dict(interpolation="LINEAR", boundary=boundary, mipmapping="LINEAR" if mips else "NONE", num_mipmaps=mips,
              coordinate_mode="TRANSFORM_LINDEPTH")
    got = ops.sample_grid_transform_gather_grad(_t(og), *cam, grid, **kw).cpu().numpy()
    assert norm_err(got, orc.sample_transform_gather_grad(og, *cam, grid, **kw)) < 1e-5


# a table's levels, all in one wave: lane by lane, and level by level (one channel, LINEAR mips)
@pytest.mark.parametrize("channels", [1, 2, 4])
@pytest.mark.parametrize("boundary", ["BORDER", "CLAMP", "WRAP"])
@pytest.mark.parametrize("mip", ["NEAREST", "LINEAR"])
def test_lut_levels(cuda, channels, boundary, mip):
    from gft.ops import sampling_ops as ops
    shape = (24, 26, 28)
    data = _smooth(shape, channels)
    rng = np.random.Generator(np.random.PCG64(8))
    lut = rng.uniform(-3, 3, size=(1, 9, 11, 13, 4)).astype(np.float32)
    # levels away from the halves, where NEAREST turns
    lut[..., 3] = rng.integers(-1, 5, size=lut.shape[:-1]) + rng.uniform(-0.4, 0.4, size=lut.shape[:-1])
    kw = dict(interpolation="LINEAR", boundary=boundary, mipmapping=mip, num_mipmaps=3, cell_center_offset=0.5)
    got = ops.sample_grid_lut(_t(data), _t(lut), **kw).cpu().numpy()
    assert norm_err(got, orc.sample_lut_fwd(data, lut, prec=1, **kw)) < 1e-5


# pyramid launches of one level (a narrow grid; unaligned rows beyond 48 MB) and of
# several behind one; 1e-6 as for the other pyramids
@pytest.mark.parametrize("shape,channels,levels", [((65, 66, 7), 1, 2), ((65, 66, 7), 4, 2), ((131, 310, 313), 1, 4),
                                                   ((47, 48, 50), 2, 1), ((64, 65, 66), 1, 6)])
def test_pyramid_launches(cuda, shape, channels, levels):
    from gft.ops import sampling_ops as ops
    rng = np.random.Generator(np.random.PCG64(5))
    data = rng.uniform(0.1, 1.0, size=(1,) + shape + (channels,)).astype(np.float32)
    got = ops.build_mips(_t(data), levels)
    ref = data.astype(np.float64)
    assert len(got) == levels
    for m in range(levels):
        d = [n // 2 for n in ref.shape[1:4]]
        ref = ref[:, :2 * d[0], :2 * d[1], :2 * d[2]].reshape(1, d[0], 2, d[1], 2, d[2], 2, channels).mean((2, 4, 6))
        assert norm_err(got[m].cpu().numpy(), ref) < 1e-6


# the render gathers' block shapes and waves, by blocks (nb) and pixel batches a block:
# 4x4x4 blocks, many of them and ragged in every axis (nb = 24); the same count with few
# pixels (8 waves); nb = 441 with few (2 waves); nb = 1521 with few (one wave, four
# blocks a workgroup, the last part empty); nb = 1305 (2 waves), 1521 (4); nb = 9288 (2)
@pytest.mark.parametrize("grid,image,views", [((11, 19, 23), (70, 85), 2), ((35, 58, 37), (8, 5), 3),
                                              ((97, 40, 40), (6, 5), 2), ((337, 40, 37), (12, 10), 2),
                                              ((289, 38, 34), (26, 23), 2), ((337, 40, 37), (120, 111), 2),
                                              ((258, 130, 113), (230, 196), 1)])
@pytest.mark.parametrize("lit", [False, True])
def test_render_gather_waves(cuda, grid, image, views, lit):
    from gft.pipeline import render_density, render_density_lit
    sc = scene(grid=grid, image=image, views=views, seed=sum(grid))
    cam = (sc["M"], sc["V"], sc["P"], sc["F"], sc["out_dhw"], sc["step"])
    rng = np.random.Generator(np.random.PCG64(views))
    lam = rng.uniform(0.2, 1.2, size=sc["data"].shape).astype(np.float32)
    w = rng.uniform(-1, 1, size=(1, views) + tuple(image) + (4,)).astype(np.float32)
    d, l = _t(sc["data"]).requires_grad_(True), _t(lam).requires_grad_(True)
    img = render_density_lit(d, l, *cam, ambient=0.4) if lit else render_density(d, *cam)
    img.backward(_t(w))
    img = img.detach().cpu().numpy()
    if lit:
        rd, rl = orc.render_lit_bwd(sc["data"], lam, img, w, *cam, ambient=0.4)
        assert norm_err(l.grad.cpu().numpy(), rl) < 1e-4
    else:
        rd = orc.render_density_bwd(sc["data"], img, w, *cam)
    assert norm_err(d.grad.cpu().numpy(), rd) < 1e-4


# waves per block of the batched level-0/1 gather: 2070 blocks or more with 0.5, 9.5 and 43
# estimated pixel batches (1, 2 and 4 waves), in every brick, with and without mips
@pytest.mark.parametrize("image", [(12, 10), (60, 42), (120, 95)])
@pytest.mark.parametrize("brick,mips", [(0, 3), (1, 3), (2, 1), (0, 0)])
def test_batched_gather_waves(cuda, image, brick, mips):
    from gft.batch import BatchedRenderStep
    grid, views = (460, 41, 41), 2
    sc = scene(grid=grid, image=image, views=views, seed=7)
    tgt = np.random.Generator(np.random.PCG64(3)).uniform(0, 0.5, size=(views,) + image + (3,)).astype(np.float32)
    b = BatchedRenderStep([dict(grid=grid, M=sc["M"], V=sc["V"], P=sc["P"], F=sc["F"], out_dhw=sc["out_dhw"],
                                depth_step=sc["step"], brick=brick)], num_mipmaps=mips)
    b.bind([_t(sc["data"])], [_t(tgt)])
    b.run()
    ref = orc.mip_render_fwd_bwd(sc["data"], tgt, sc["M"], sc["V"], sc["P"], sc["F"], sc["out_dhw"], sc["step"],
                                 num_mipmaps=mips)
    assert norm_err(b.grads[0].cpu().numpy(), ref["gd"]) < 1e-4


# A camera so far away (in cells) that ray positions round by more than a brick's
# slack: a CLAMP sample outside its segment's brick still goes to its own cells. All
# samples lie well inside the grid, where WRAP has the same positions and
# corners and no bricks; the two then differ by the order of their sums alone
# (float atomics of up to 100 terms a cell: 100 x 2^-24).
@pytest.mark.parametrize("distance", [1e3, 2e6, 8e6])
def test_clamp_scatter_far_camera(cuda, distance):
    from gft.pipeline import render_density
    n, half, image, S = 80, 12.0, (66, 70), 24
    near, far = distance - half, distance + half
    tan = half / far
    P = np.zeros((4, 4))
    P[0, 0] = P[1, 1] = 1.0 / tan
    P[2, 2], P[2, 3], P[3, 2] = -(far + near) / (far - near), -2 * far * near / (far - near), -1
    P[2, 0] = -1.2 * P[2, 2]  # near and far planes that lean: each pixel has a depth, and a rounding, of its own
    V, M = np.eye(4), np.eye(4)
    c, s = np.cos(0.7), np.sin(0.7)  # along a row, x hardly changes but for the rounding
    V[0, 0], V[0, 2], V[2, 0], V[2, 2], V[2, 3] = c, s, -s, c, -distance
    M[:3, 3] = -n / 2.0
    M, V, P = (np.ascontiguousarray(a.T[None], dtype=np.float32) for a in (M, V, P))
    F = np.array([[near, far, -near * tan, near * tan, near * tan, -near * tan]], dtype=np.float32)
    rng = np.random.Generator(np.random.PCG64(5))
    data = rng.uniform(0.0, 0.02, size=(1, n, n, n, 1)).astype(np.float32)
    w = rng.uniform(-1, 1, size=(1, 1) + image + (4,)).astype(np.float32)
    grads = []
    for boundary in ("CLAMP", "WRAP"):
        d = _t(data).requires_grad_(True)
        render_density(d, M, V, P, F, (S,) + image, 1.0, boundary=boundary).backward(_t(w))
        grads.append(d.grad.cpu().numpy())
    assert norm_err(grads[0], grads[1]) < 1e-5


# 2^24 rows of corner-quad bricks: their index takes 32-bit products
@pytest.mark.parametrize("boundary", ["BORDER", "CLAMP"])
def test_render_many_brick_rows(cuda, boundary):
    from gft.pipeline import render_density
    sc = scene(grid=(8192, 4100, 2), image=(3, 3), views=1, seed=4, blobs=3)
    data = np.random.Generator(np.random.PCG64(6)).uniform(0.0, 0.001, size=sc["data"].shape).astype(np.float32)
    cam = (sc["M"], sc["V"], sc["P"], sc["F"], sc["out_dhw"], sc["step"])
    d = _t(data).requires_grad_(True)
    img = render_density(d, *cam, boundary=boundary)
    ref = orc.render_density_fwd(data, *cam, boundary=boundary)
    assert ref.any() and norm_err(img.detach().cpu().numpy(), ref) < kLongRays
    w = np.random.Generator(np.random.PCG64(7)).uniform(-1, 1, size=ref.shape).astype(np.float32)
    img.backward(_t(w))
    gref = orc.render_density_bwd(data, ref, w, *cam, boundary=boundary)
    assert gref.any() and norm_err(d.grad.cpu().numpy(), gref) < kLongRays
