"""The render trees by name (0 the library's choice, 1 four-wide, 2 flat, 3 the
binary LBVH in every case) in the persistent path kernel: the Cornell box, which
tree 0 walks flat, and scenes and passes on both sides of the lines where tree 0
changes between the flat and the binary walk.  Every image equals the oracle's
bit for bit."""
import numpy as np
import pytest

from oracle import orc
from aurora_amd import scenes
from aurora_amd.core import Camera, RenderSettings

pytestmark = pytest.mark.gpu

TREES = (0, 1, 2, 3)


def both(ctx, arr):
    g = ctx.upload(arr)
    g.build_bvh()
    o = orc.OracleScene(arr)
    o.build_bvh()
    return g, o


def test_cornell_under_every_tree(ctx):
    g, o = both(ctx, scenes.cornell_box())
    cam = scenes.cornell_camera(40)
    rs = RenderSettings(spp=6, aov=True, spp_per_pass=4)
    want = o.render(cam, rs)
    for tree in TREES:
        ctx.set_render_tree(tree)
        try:
            for graph in (False, True):
                got = g.render(cam, RenderSettings(spp=6, aov=True, spp_per_pass=4, graph=graph))
                assert got[3]["segments"] == want[3], (tree, graph)
                for a, b in zip(got[:3], want[:3]):
                    assert np.array_equal(a.view(np.uint32), b.view(np.uint32)), (tree, graph)
        finally:
            ctx.set_render_tree(0)
    g.close()


@pytest.mark.parametrize("prims,scale", [(9, 4.0), (10, 4.0), (40, 2.5), (40, 1.0), (41, 4.0), (64, 4.0), (65, 4.0)])
def test_both_sides_of_the_flat_rule(ctx, prims, scale):
    """Few and many leaves, overlap above and below one, passes of up to 32,768
    paths and of more."""
    arr, _, _ = scenes.batch_scene(prims, prims, prims)
    if len(arr.spheres):
        arr.spheres[:, 3] *= scale
    if len(arr.quads):
        arr.quads[:, 3:] *= scale
    g, o = both(ctx, arr)
    for w, h in ((64, 48), (184, 180)):
        cam = Camera(w, h, 40.0, (0.0, 0.5, 4.0), (0.0, 0.0, 0.0))
        rs = RenderSettings(spp=1, max_depth=8, background=(0.6, 0.7, 0.9))
        want = o.render(cam, rs)
        for tree in TREES:
            ctx.set_render_tree(tree)
            try:
                got = g.render(cam, rs)
            finally:
                ctx.set_render_tree(0)
            assert got[3]["segments"] == want[3], (w, tree)
            assert np.array_equal(got[0].view(np.uint32), want[0].view(np.uint32)), (w, tree)
    g.close()


def test_unknown_trees_are_refused(ctx):
    for tree in (-1, 4):
        with pytest.raises(ValueError):
            ctx.set_render_tree(tree)
