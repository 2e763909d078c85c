"""The pooled traversal, which keeps one leaf aside while it visits more nodes.

Trees where that can go wrong: a single leaf, two, chains that end right after
a leaf, leaves of several primitives of both kinds, and primitives nested so
that a kept leaf's hit would have culled what was visited meanwhile.  Every
output equals the oracle's linear scan bit for bit.
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


def _nested(n):
    """Concentric spheres around every sphere's centre: a ray that hits one has hits behind it in other leaves."""
    rng = scenes.rng_for(601, n)
    sph = scenes.random_spheres(rng, n, -6.0, 6.0, kinds=("diffuse", "metal", "dielectric"))
    inner = np.concatenate([sph, sph, sph])
    inner["r"][n:2 * n] *= np.float32(0.75)
    inner["r"][2 * n:] *= np.float32(0.5)
    return inner


@pytest.mark.parametrize("device_bvh", [False, True], ids=["host", "device"])
@pytest.mark.parametrize("leaf", [1, 3, 8])
@pytest.mark.parametrize("n_tris,n_sph,nested", [(0, 100, 0), (2, 82, 0), (50, 3, 0), (90, 3, 0), (400, 9, 0), (60, 3, 30)])
def test_every_tree_gives_the_scan(ctx, n_tris, n_sph, nested, leaf, device_bvh):
    rng = scenes.rng_for(602, 1000 * n_tris + n_sph)
    sph = scenes.random_spheres(rng, n_sph, -9.0, 9.0, kinds=("diffuse", "metal"))
    lights = scenes.light_sphere((0.0, 9.0, -4.0), 1.5), scenes.light_sphere((-7.0, 2.0, -9.0), 1.0)
    sph = np.concatenate([sph, *lights] + ([_nested(nested)] if nested else []))
    tris = scenes.random_soup(rng, n_tris, lo=-8.0, hi=8.0, elo=1.0, ehi=6.0) if n_tris else np.zeros(0, vkr.TRIANGLE)
    w, h, spp, depth = 37, 29, 2, 4
    cam = vkr.camera_from_angles((0.0, 0.0, -28.0), 0.0, 90.0)
    wl = scenes.Workload("kept", vkr.Scene(spheres=sph, tris=tris, planes=scenes.ground(-10.0)),
                         scenes.frame(cam, np.float32(w) / np.float32(h), 0.375), w, h, spp, depth)
    sid = ctx.upload(wl.scene, max_leaf=leaf, device_bvh=device_bvh)
    got = gpu_trace(ctx, sid, wl)
    ctx.destroy_scene(sid)
    st = compare(got, oracle_ffi.trace(wl.scene, wl.frame, w, h, spp, depth))
    for k in ("prim_id", "hit_t_bits", "radiance_bits", "rgba8", "ray_count"):
        assert st[k] == 1.0, (k, st)
