"""The path kernel's step: a vertex's shadow rays and the next segment together.

A step takes the last window of a diffuse vertex's emitters (31 a window in
the pooled kernel, one shadow ray at a time in the single-ray kernel) together
with the segment that leaves the vertex, and every sample after the first
starts at the kept primary hit.  So the places where it can go wrong are the
window boundaries, scenes without emitters, pixels whose primary ray misses,
and one, two and several samples at depth one and more.  Every output equals
the oracle's linear scan bit for bit.
"""
import numpy as np
import pytest

import oracle_ffi
import scenes
import vkr
from gpu_util import compare, gpu_trace

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    c = vkr.Context()
    yield c
    c.close()


def _scene(n_emitters, ground):
    rng = scenes.rng_for(201, n_emitters)
    parts = [scenes.random_spheres(rng, 12, -6.0, 6.0, kinds=("diffuse", "metal", "dielectric"))]
    if n_emitters:
        parts.append(scenes.random_spheres(rng, n_emitters, -9.0, 9.0, kinds=("emissive",)))
    tris = scenes.random_soup(rng, 60, lo=-8.0, hi=8.0)
    planes = scenes.ground(-9.0) if ground else np.zeros(0, vkr.PLANE)
    return vkr.Scene(tris=tris, spheres=np.concatenate(parts), planes=planes)


@pytest.mark.parametrize("pool", [False, True], ids=["single_ray", "ray_pool"])
@pytest.mark.parametrize("spp,depth", [(1, 1), (2, 4), (5, 2)])
@pytest.mark.parametrize("n_emitters,ground", [(0, True), (1, False), (2, True), (31, True), (32, False), (62, True),
                                               (63, True)])
def test_steps_match_oracle(ctx, n_emitters, ground, spp, depth, pool):
    w, h = 41, 23
    cam = vkr.camera_from_angles((0.0, 0.0, -26.0), 0.0, 90.0)
    wl = scenes.Workload("steps", _scene(n_emitters, ground), scenes.frame(cam, np.float32(w) / np.float32(h), 0.25),
                         w, h, spp, depth)
    sid = ctx.upload(wl.scene)
    g = gpu_trace(ctx, sid, wl, flags=vkr.TRACE_RAY_POOL if pool else vkr.TRACE_NO_RAY_POOL)
    ctx.destroy_scene(sid)
    r = oracle_ffi.trace(wl.scene, wl.frame, w, h, spp, depth)
    st = compare(g, r)
    assert st["window_overflow"] == 0
    for k in ("prim_id", "hit_t_bits", "radiance_bits", "rgba8", "ray_count"):
        assert st[k] == 1.0, (k, st)
