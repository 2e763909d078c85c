"""Trees whose boxes reach the ends of the node's 16-bit half-extents, and the sphere boxes' widening.

Half-extents are rounded up to 16-bit floats: above 65504 they become infinite,
below 2^-14 they become that.  The sphere subtree's widening depends on the
least radius.  So: triangles of 1e5 and 1e6 units beside small ones, a scene of
1e-3 units, and spheres whose radii span six orders of magnitude, one of them
zero and one negative, seen from near and far.  Both kernels (single rays and
ray pool), both builders; every output equals the oracle's linear scan.
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


def _workload(name):
    rng = scenes.rng_for(501, 0)
    scale, cam_z, eps = 1.0, -40.0, 1e-3
    sph = scenes.random_spheres(rng, 120, -12.0, 12.0)
    tris = scenes.random_soup(rng, 300, lo=-15.0, hi=15.0)
    if name == "huge":
        big = scenes.random_soup(rng, 12, lo=20.0, hi=60.0, elo=1e5, ehi=1e6)
        tris = np.concatenate([tris, big])
    elif name == "tiny":
        scale, eps = 1e-4, 1e-7
    elif name == "radii":
        sph["r"] = (10.0 ** rng.uniform(-5, 1, len(sph))).astype(np.float32)
        sph["r"][3], sph["r"][5] = 0.0, -1.0
    elif name == "far":
        sph["r"] = rng.uniform(2.0, 3.0, len(sph)).astype(np.float32)
        cam_z = -1500.0
    sph = np.concatenate([sph, scenes.light_sphere((0.0, 18.0, -6.0), 2.0)])
    sph["P"] *= np.float32(scale)
    sph["r"] *= np.float32(scale)
    for k in ("v0", "v1", "v2"):
        tris[k] *= np.float32(scale)
    cam = vkr.camera_from_angles((0.0, 0.0, cam_z * scale), 0.0, 90.0)
    if name == "far":
        cam["right"] *= np.float32(0.02)
        cam["up"] *= np.float32(0.02)
    sc = vkr.Scene(spheres=sph, tris=tris)
    return scenes.Workload(name, sc, scenes.frame(cam, 1.5, 0.125), 48, 32, 2, 3), eps


@pytest.mark.parametrize("device_bvh", [False, True], ids=["host", "device"])
@pytest.mark.parametrize("pool", [False, True], ids=["single_ray", "ray_pool"])
@pytest.mark.parametrize("name", ["huge", "tiny", "radii", "far"])
def test_extents_and_radii(ctx, name, pool, device_bvh):
    wl, eps = _workload(name)

    class W:
        width, height, spp, frame = wl.width, wl.height, wl.spp, wl.frame
        params = staticmethod(lambda **kw: wl.params(epsilon=eps, **kw))

    sid = ctx.upload(wl.scene, device_bvh=device_bvh)
    g = gpu_trace(ctx, sid, W, flags=vkr.TRACE_RAY_POOL if pool else vkr.TRACE_NO_RAY_POOL)
    ctx.destroy_scene(sid)
    r = oracle_ffi.trace(wl.scene, wl.frame, wl.width, wl.height, wl.spp, wl.max_depth, epsilon=eps)
    st = compare(g, r)
    for k in ("prim_id", "hit_t_bits", "radiance_bits", "rgba8", "ray_count"):
        assert st[k] == 1.0, (k, st)
    assert (r["prim_id"] != vkr.MISS).any()
