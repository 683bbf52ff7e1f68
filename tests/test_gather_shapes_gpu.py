"""The render backward's voxel-block gathers at the edges of their rules: block
shapes and waves per block are picked by the grid's block count, so grids on
both sides of each line, ragged against the blocks, against the FP64 oracle
(gradients 1e-4 normalised max error, as the other render backward tests),
with more than 16 views (two accumulating launches) and repeated bit for bit.
"""
import numpy as np
import pytest
import torch

from helpers import norm_err, scene
from oracle import oracle as orc

pytestmark = pytest.mark.gpu


def _t(a):
    return torch.from_numpy(np.ascontiguousarray(a, dtype=np.float32)).cuda()


# blocks of 16x16x2: 1, 189, 260, 612, 660, 756
RENDER_GRIDS = [((1, 1, 1), (9, 7), 1), ((41, 97, 33), (60, 34), 3), ((52, 72, 31), (66, 40), 2),
                ((67, 81, 33), (50, 30), 18), ((66, 65, 49), (40, 90), 2), ((36, 90, 97), (70, 40), 3)]


@pytest.mark.parametrize("grid,image,views", RENDER_GRIDS)
@pytest.mark.parametrize("lit", [False, True])
def test_render_gather_block_rules(cuda, grid, image, views, lit):
    from gft.pipeline import render_density, render_density_lit
    sc = scene(grid=grid, image=image, views=views, seed=sum(grid))
    cam = (sc["M"], sc["V"], sc["P"], sc["F"], sc["out_dhw"], sc["step"])
    rng = np.random.Generator(np.random.PCG64(views))
    lam = rng.uniform(0.2, 1.2, size=sc["data"].shape).astype(np.float32)
    w = rng.uniform(-1, 1, size=(1, views) + tuple(image) + (4,)).astype(np.float32)

    def grads():
        d, l = _t(sc["data"]).requires_grad_(True), _t(lam).requires_grad_(True)
        img = render_density_lit(d, l, *cam, ambient=0.4) if lit else render_density(d, *cam)
        img.backward(_t(w))
        torch.cuda.synchronize()
        return img.detach().cpu().numpy(), d.grad, l.grad

    img, gd, gl = grads()
    if lit:
        rd, rl = orc.render_lit_bwd(sc["data"], lam, img, w, *cam, ambient=0.4)
        assert norm_err(gl.cpu().numpy(), rl) < 1e-4
    else:
        rd = orc.render_density_bwd(sc["data"], img, w, *cam)
    assert norm_err(gd.cpu().numpy(), rd) < 1e-4
    _, gd2, gl2 = grads()
    assert torch.equal(gd, gd2) and (not lit or torch.equal(gl, gl2))


@pytest.mark.parametrize("brick", [0, 1, 2])
def test_batch_gather_shared_blocks(cuda, brick):
    """The batched gather's waves share a block's pixels: reconstructions with
    fewer pixel batches than waves, with many (a small grid in large images) and
    out of the table's cost order, each against the FP64 oracle."""
    from gft.batch import BatchedRenderStep
    specs = [((20, 33, 18), (50, 40), 2), ((5, 6, 7), (90, 70), 3), ((17, 16, 31), (4, 5), 8)]
    recons, dens, tgts = [], [], []
    for k, (grid, image, views) in enumerate(specs):
        sc = scene(grid=grid, image=image, views=views, seed=90 + k)
        recons.append(dict(grid=grid, M=sc["M"], V=sc["V"], P=sc["P"], F=sc["F"], out_dhw=sc["out_dhw"],
                           depth_step=sc["step"], brick=brick))
        dens.append(sc["data"])
        tgts.append(np.random.Generator(np.random.PCG64(k)).uniform(0, 0.5, size=(views,) + image + (3,)))
    b = BatchedRenderStep(recons, num_mipmaps=3)
    b.bind([_t(d) for d in dens], [_t(t) for t in tgts])
    b.run()
    torch.cuda.synchronize()
    first = [g.clone() for g in b.grads]
    b.run()
    torch.cuda.synchronize()
    for r, d, t, g, g0 in zip(recons, dens, tgts, b.grads, first):
        ref = orc.mip_render_fwd_bwd(d, t.astype(np.float32), r["M"], r["V"], r["P"], r["F"], r["out_dhw"],
                                     r["depth_step"], num_mipmaps=3)
        assert norm_err(g.cpu().numpy(), ref["gd"]) < 1e-4
        assert torch.equal(g, g0)


@pytest.mark.parametrize("boundary", ["CLAMP", "BORDER"])
@pytest.mark.parametrize("grid,image,views", [((1, 5, 1), (20, 18), 2), ((33, 20, 47), (70, 35), 3),
                                              ((9, 70, 12), (33, 50), 5)])
def test_scatter_walk_bricks(cuda, boundary, grid, image, views):
    """The recompute walk's scatter: one-cell axes, tiles whose segments share a
    brick, rim cells outside the grid (BORDER), ragged tiles; FP64 oracle 1e-4."""
    from gft.pipeline import TransportRenderStep
    sc = scene(grid=grid, image=image, views=views, seed=sum(grid))
    tgt = np.random.Generator(np.random.PCG64(1)).uniform(0, 0.5, size=(1, views) + image + (3,)).astype(np.float32)
    step = TransportRenderStep(grid, sc["M"], sc["V"], sc["P"], sc["F"], sc["out_dhw"], sc["step"], boundary=boundary,
                               reduction="scatter", order=1)
    d, v = _t(sc["data"]), torch.zeros((1,) + grid + (3,), device="cuda")
    loss, gd, _ = step.run(d, v, _t(tgt))
    torch.cuda.synchronize()
    img = step.images.cpu().numpy()
    rl, gimg = orc.l2_loss_and_grad(img.astype(np.float64), tgt)
    ref = orc.render_density_bwd(sc["data"], img, gimg, sc["M"], sc["V"], sc["P"], sc["F"], sc["out_dhw"], sc["step"],
                                 boundary=boundary)
    assert norm_err(gd.cpu().numpy(), ref) < 1e-4
    assert abs(loss.item() - rl) <= 1e-5 * rl
