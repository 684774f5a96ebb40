"""Batches whose wavefront bounces walk four lanes per ray with a scene per ray:
most paths in scenes of 16,384 primitives or more (spheres and quads, overlapping
ones too), among them a small scene, one of a single primitive and one whose stack
leaves shared memory.  Wavefront only, with the fused tail from 4,096 live paths
on, eager and captured: every image equals its single render in the persistent
kernel over the binary tree bit for bit.  One primitive fewer in each large scene
and the same batch walks one lane per ray."""
import numpy as np
import pytest
import torch

from aurora_amd import scenes
from aurora_amd.core import Camera, RenderSettings, render_batch

pytestmark = pytest.mark.gpu


def zeros(cam):
    return tuple(torch.zeros((cam.image_height, cam.image_width, 3), dtype=torch.float32, device="cuda")
                 for _ in range(3))


def workload(ctx, large):
    box = lambda w, h: Camera(w, h, 40.0, (0.0, 0.5, 4.0), (0.0, 0.0, 0.0))
    sky = dict(background=(0.6, 0.7, 0.9), aov=True)
    specs = [
        (scenes.batch_scene(3, large, large)[0], box(96, 80), RenderSettings(spp=3, max_depth=12, **sky)),
        (scenes.stress_scene(large // 2, large - large // 2, seed=5), scenes.stress_camera(97, 55),
         RenderSettings(spp=2, max_depth=16, tmin=1e-4, **sky)),
        (scenes.batch_scene(8, 50_000, 50_000)[0], box(64, 65), RenderSettings(spp=2, max_depth=20, seed=3, **sky)),
        (scenes.cornell_box(), scenes.cornell_camera(24), RenderSettings(spp=3, max_depth=50, aov=True)),
        (scenes.batch_scene(5, 1, 1)[0], box(17, 9), RenderSettings(spp=1, max_depth=8, **sky)),
        (scenes.deep_chain_scene(glass=True), Camera(32, 24, 40.0, (1.5, 1.2, 2.0), (0.0, 0.0, 0.0)),
         RenderSettings(spp=2, max_depth=16, tmin=1e-4, **sky)),
    ]
    items = []
    for arr, cam, rs in specs:
        sc = ctx.upload(arr)
        sc.build_bvh()
        items.append((sc, cam, rs))
    return items


@pytest.mark.parametrize("large", [16384, 16383])
def test_large_scenes_in_a_batch_equal_single_renders(ctx, large):
    items = workload(ctx, large)
    paths = [cam.image_width * cam.image_height * rs.spp for _, cam, rs in items]
    assert 2 * sum(paths[:3]) >= sum(paths) and 2 * paths[2] < sum(paths)
    singles, seg = [], 0
    try:
        ctx.set_render_tree(3)
        for sc, cam, rs in items:
            b = zeros(cam)
            seg += sc.render_device(cam, rs, *b)["segments"]
            singles.append(b)
        ctx.set_render_tree(1)
        for tail in (0, 4096, 16384):
            ctx.set_launch(tail_paths=tail)
            for graph in (False, True):
                print("large", large, "tail", tail, "graph", graph, flush=True)
                bufs = [zeros(cam) for _, cam, _ in items]
                st = render_batch(ctx, [(sc, cam, rs, *b) for (sc, cam, rs), b in zip(items, bufs)], graph=graph)
                assert st["segments"] == seg
                for k, (b, s) in enumerate(zip(bufs, singles)):
                    for x, y in zip(b, s):
                        assert np.array_equal(x.cpu().numpy().view(np.uint32), y.cpu().numpy().view(np.uint32)), (tail, graph, k)
    finally:
        ctx.set_launch()
        ctx.set_render_tree(0)
        for sc, _, _ in items:
            sc.close()
