"""The LBVH at sizes where its launches change: the one-launch scan's tiles
(4096 entries: 16 sort blocks of 2048 primitives, or 4096 wide-node flags), its
last size (262,144 entries: that many flags, or 1024 sort blocks) and the first
of the three-launch scan, and levels on both sides of one block's run.  Every
word equals the oracle's build."""
import numpy as np
import pytest

from oracle import orc
from aurora_amd import scenes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [4095, 4096, 4097, 32768, 32769, 262_144, 262_145, 2_097_152, 2_097_153])
def test_build_equals_oracle_at_launch_edges(ctx, n):
    print("build", n, flush=True)
    arr = scenes.stress_scene(n // 2, n - n // 2, seed=n)
    scene = ctx.upload(arr)
    got = scene.build_bvh()
    again = scene.build_bvh()  # scratch of the first build in place
    o = orc.OracleScene(arr)
    want = o.build_bvh()
    for k in ("n_prims", "n_nodes", "n_wide", "depth", "wide_depth", "wide_form", "scene_lo", "scene_hi",
              "centroid_lo", "centroid_hi"):
        assert got[k] == want[k] and again[k] == want[k], k
    for g, w in zip(scene.order(), o.order()):
        assert np.array_equal(g, w)
    assert np.array_equal(scene.nodes(), o.nodes())
    assert np.array_equal(scene.wide(), o.wide())


def test_scenes_of_a_context_build_and_close_in_turn(ctx):
    """The builds of a context share its pinned words: scenes of different sizes
    built in turn each read their own counts, and a closed scene gives back only
    device memory, in less time than half its build took (a pinned free per scene
    took longer than the build)."""
    import time
    arrs = [scenes.batch_scene(n, n, n)[0] for n in (2, 5, 100, 3000)]
    want = []
    for arr in arrs:
        o = orc.OracleScene(arr)
        want.append(o.build_bvh())
    up = [ctx.upload(a) for a in arrs]
    for order in ((0, 1, 2, 3), (3, 1, 0, 2)):
        for k in order:
            got = up[k].build_bvh()
            for key in ("n_prims", "n_nodes", "n_wide", "depth", "wide_depth", "scene_lo", "scene_hi"):
                assert got[key] == want[k][key], (k, key)
    for s in up:
        s.close()
    build, many = [], [ctx.upload(arrs[2]) for _ in range(32)]
    for s in many:
        s.build_bvh()
        t0 = time.perf_counter()
        s.build_bvh()
        build.append(time.perf_counter() - t0)
    t0 = time.perf_counter()
    for s in many:
        s.close()
    close = (time.perf_counter() - t0) / len(many)
    print("100 primitives: build", np.median(build), "close", close, flush=True)
    assert close < 0.5 * np.median(build)
