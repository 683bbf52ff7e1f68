"""The density render at the edges of its pixel tiles: a workgroup of the
forwards and of the scatter backward takes 16 x 4 pixels; the forwards' rows of
tiles are dealt out by eights (BORDER) or in order (CLAMP, WRAP). Images against
the FP64 oracle within 1e-5 normalised max error and gradients within 1e-4, as
at ordinary sizes.
"""
import numpy as np
import pytest
import torch

from helpers import norm_err, scene
from oracle import oracle as orc

pytestmark = pytest.mark.gpu


def _t(a):
    return torch.from_numpy(np.ascontiguousarray(a, dtype=np.float32)).cuda()


@pytest.mark.parametrize("image", [(1, 1), (3, 17), (4, 16), (33, 15), (129, 47), (70, 160)])
@pytest.mark.parametrize("kind", ["BORDER", "CLAMP", "WRAP", "lit"])
def test_forward_tiles(cuda, image, kind):
    from gft.pipeline import render_density, render_density_lit
    sc = scene(grid=(9, 15, 12), image=image, views=3, seed=sum(image))
    cam = (sc["M"], sc["V"], sc["P"], sc["F"], sc["out_dhw"], sc["step"])
    if kind == "lit":
        lam = np.random.Generator(np.random.PCG64(2)).uniform(0.2, 1.2, size=sc["data"].shape).astype(np.float32)
        got = render_density_lit(_t(sc["data"]), _t(lam), *cam, ambient=0.4)
        ref = orc.render_lit_fwd(sc["data"], lam, *cam, ambient=0.4)
    else:
        got = render_density(_t(sc["data"]), *cam, boundary=kind)
        ref = orc.render_density_fwd(sc["data"], *cam, boundary=kind)
    assert tuple(got.shape) == ref.shape
    assert norm_err(got.cpu().numpy(), ref) < 1e-5


# the last: a few pixels over many cells, whose tile's bricks exceed the LDS
@pytest.mark.parametrize("grid,image", [((9, 15, 12), (1, 1)), ((9, 15, 12), (3, 17)), ((9, 15, 12), (33, 15)),
                                        ((1, 15, 12), (20, 9)), ((9, 15, 12), (129, 47)), ((40, 52, 44), (5, 7))])
def test_clamp_scatter_tiles(cuda, grid, image):
    from gft.pipeline import render_density
    sc = scene(grid=grid, image=image, views=2, seed=sum(image))
    cam = (sc["M"], sc["V"], sc["P"], sc["F"], sc["out_dhw"], sc["step"])
    d = _t(sc["data"]).requires_grad_(True)
    img = render_density(d, *cam, boundary="CLAMP")
    w = np.random.Generator(np.random.PCG64(3)).uniform(-1, 1, size=tuple(img.shape)).astype(np.float32)
    img.backward(_t(w))
    ref = orc.render_density_bwd(sc["data"], img.detach().cpu().numpy(), w, *cam, boundary="CLAMP")
    assert norm_err(d.grad.cpu().numpy(), ref) < 1e-4
