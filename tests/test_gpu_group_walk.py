"""Ray queries without fetch counters (the group walk, four lanes per ray)
against the same queries with counters (one lane per ray): the same primitive
and the same bits of t, at the edges of a wave's 16 rays and a block's 64, past
the resident grid (where waves claim their rays), on trees of one primitive up
to one whose stack leaves shared memory, and with the hits written over rays."""
import numpy as np
import pytest

from aurora_amd import scenes

pytestmark = pytest.mark.gpu

SCENES = {
    "one": lambda: scenes.batch_scene(5, 1, 1)[0],
    "ten": lambda: scenes.batch_scene(5, 10, 10)[0],
    "textured": lambda: scenes.textured_scene(1),
    "stress": lambda: scenes.stress_scene(3000, 3001, 2),
    "deep": lambda: scenes.deep_chain_scene(),
}


def trace_both(scene, o, d, **kw):
    import torch
    n = o.shape[0]
    out = []
    for counted in (False, True):
        prim = torch.full((n,), -7, dtype=torch.int32, device="cuda")
        t = torch.full((n,), -7.0, device="cuda")
        counts = torch.zeros((n, 3), dtype=torch.int32, device="cuda") if counted else None
        scene.trace_device(o, d, prim, t, counts=counts, **kw)
        scene.ctx.synchronize()
        out.append((prim.cpu().numpy(), t.cpu().numpy().view(np.uint32)))
    return out


@pytest.mark.parametrize("name", list(SCENES))
@pytest.mark.parametrize("n", [1, 15, 16, 17, 63, 64, 65, 4097, 200_003])
def test_group_walk_equals_counted_walk(ctx, name, n):
    scene = ctx.upload(SCENES[name]())
    scene.build_bvh()
    o, d = scenes.random_rays_torch(n, [-1.5] * 3, [1.5] * 3, seed=n)
    d[::5, 0] = 0.0  # axis-parallel components: infinite reciprocals
    for kw in ({}, {"tmin": 1e-3, "tmax": 0.7}, {"tmin": -0.5}):
        (pa, ta), (pb, tb) = trace_both(scene, o, d, **kw)
        assert np.array_equal(pa, pb) and np.array_equal(ta, tb), kw
    scene.close()


def test_hits_written_over_the_rays(ctx):
    import torch
    scene = ctx.upload(SCENES["stress"]())
    scene.build_bvh()
    n = 50_001
    o, d = scenes.random_rays_torch(n, [0.0] * 3, [1.0] * 3, seed=3)
    (pa, ta), _ = trace_both(scene, o, d)
    for call in (scene.trace_device, scene.trace_device_noalloc):
        o2, d2 = o.clone(), d.clone()
        prim, t = o2.view(-1)[:n].view(torch.int32), d2.view(-1)[n:2 * n]
        call(o2, d2, prim, t)
        scene.ctx.synchronize()
        assert np.array_equal(prim.cpu().numpy(), pa)
        assert np.array_equal(t.cpu().numpy().view(np.uint32), ta)
    scene.close()
