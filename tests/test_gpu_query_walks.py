"""Ray queries without fetch counters at the lines between their walks: a ray per
place of the group walk's grid and one more, 1,024 and 32,768 primitives, rays
that go together (a camera's), rays that do not, and both in one call.  The same
primitive and the same bits of t as the counted query, which always walks one
lane per ray."""
import time

import numpy as np
import pytest
import torch

from aurora_amd import abi, scenes
from aurora_amd.core import Camera

pytestmark = pytest.mark.gpu


def rays(ctx, kind, n, seed):
    o, d = scenes.random_rays_torch(n, [-1.2] * 3, [1.2] * 3, seed=seed)
    if kind != "random":
        w = 640
        h = (n + w - 1) // w
        cam = Camera(w, h, 40.0, (0.0, 0.5, 4.0), (0.0, 0.0, 0.0))
        co, cd = torch.empty((w * h, 3), device="cuda"), torch.empty((w * h, 3), device="cuda")
        px = torch.arange(w * h, dtype=torch.int32, device="cuda")
        ctx.camera_rays_device(cam, px, torch.zeros_like(px), co, cd, seed=seed)
        ctx.synchronize()
        k = n if kind == "camera" else n // 2
        o[:k], d[:k] = co[:k], cd[:k]
    return o, d


def ask(call, n, o, d, **kw):
    prim = torch.full((n,), -7, dtype=torch.int32, device="cuda")
    t = torch.full((n,), -7.0, device="cuda")
    call(o, d, prim, t, tmin=1e-4, **kw)
    return prim, t


@pytest.mark.parametrize("prims", [0, 1, 1023, 1024, 5000, 32767, 32768])
@pytest.mark.parametrize("kind", ["camera", "random", "both"])
def test_walks_agree(ctx, prims, kind):
    print("walks", prims, kind, flush=True)
    arr = scenes.batch_scene(7, max(prims, 1), max(prims, 1))[0] if prims else scenes.stress_scene(0, 0, 1)
    scene = ctx.upload(arr)
    scene.build_bvh()
    hold = 8 * 256 * 64  # the rays that the group walk's grid holds at eight blocks per CU
    for n in (hold, hold + 1, 3 * hold + 77):
        o, d = rays(ctx, kind, n, n)
        counts = torch.zeros((n, 3), dtype=torch.int32, device="cuda")
        cp, ct = ask(scene.trace_device, n, o, d, counts=counts)
        for mode in (1, 2):  # as given, sorted
            ctx.set_ray_sort(mode)
            try:
                p, t = ask(scene.trace_device, n, o, d)
            finally:
                ctx.set_ray_sort(1)
            ctx.synchronize()
            assert torch.equal(p, cp) and torch.equal(t.view(torch.int32), ct.view(torch.int32)), (n, mode)
        for m in (65536, 65537, abi.NOALLOC_MAX_RAYS):
            if m <= n:
                p, t = ask(scene.trace_device_noalloc, m, o[:m], d[:m])
                ctx.synchronize()
                assert torch.equal(p, cp[:m]) and torch.equal(t.view(torch.int32), ct[:m].view(torch.int32)), m
    scene.close()


@pytest.mark.parametrize("prims", [500, 5000])
def test_hits_over_rays_and_a_small_grid(ctx, prims):
    """Hits written over the rays of a call that walks one lane per ray, and the
    smallest grid (one block per CU: every wave claims often)."""
    scene = ctx.upload(scenes.batch_scene(9, prims, prims)[0])
    scene.build_bvh()
    n = 200_001
    o, d = rays(ctx, "camera", n, 5)
    cp, ct = ask(scene.trace_device, n, o, d, counts=torch.zeros((n, 3), dtype=torch.int32, device="cuda"))
    ctx.synchronize()
    ctx.set_launch(extend_blocks_per_cu=1)
    try:
        p, t = ask(scene.trace_device, n, o, d)
    finally:
        ctx.set_launch()
    ctx.synchronize()
    assert torch.equal(p, cp) and torch.equal(t.view(torch.int32), ct.view(torch.int32))
    for call in (scene.trace_device, scene.trace_device_noalloc):
        o2, d2 = o.clone(), d.clone()
        p, t = o2.view(-1)[:n].view(torch.int32), d2.view(-1)[n:2 * n]
        call(o2, d2, p, t, tmin=1e-4)
        ctx.synchronize()
        assert torch.equal(p, cp) and torch.equal(t.view(torch.int32), ct.view(torch.int32))
    scene.close()


@pytest.mark.parametrize("prims", [500, 2000, 4000, 8000])
def test_a_query_without_counters_is_no_slower_than_with_them(ctx, prims):
    """A camera's rays on small scenes: the group walk took up to 1.6 times the
    counted query's time (and that one does the packing and the counting too)."""
    scene = ctx.upload(scenes.batch_scene(2, prims, prims)[0])
    scene.build_bvh()
    n = 512 * 512
    cam = Camera(512, 512, 40.0, (0.0, 0.5, 4.0), (0.0, 0.0, 0.0))
    o, d = torch.empty((n, 3), device="cuda"), torch.empty((n, 3), device="cuda")
    px = torch.arange(n, dtype=torch.int32, device="cuda")
    ctx.camera_rays_device(cam, px, torch.zeros_like(px), o, d, seed=1)
    prim, t = torch.empty(n, dtype=torch.int32, device="cuda"), torch.empty(n, device="cuda")
    counts = torch.zeros((n, 3), dtype=torch.int32, device="cuda")

    def seconds(call, **kw):
        out = []
        for _ in range(7):
            ctx.synchronize()
            t0 = time.perf_counter()
            for _ in range(10):
                call(o, d, prim, t, tmin=1e-4, **kw)
            ctx.synchronize()
            out.append((time.perf_counter() - t0) / 10)
        return float(np.median(out))

    for call in (scene.trace_device, scene.trace_device_noalloc):
        plain, counted = seconds(call), seconds(call, counts=counts)
        print(prims, call.__name__, "plain us", plain * 1e6, "counted us", counted * 1e6, flush=True)
        assert plain < 1.05 * counted
    scene.close()
