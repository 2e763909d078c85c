"""Small images of scanned scenes, whose pixels are tested by four lanes each.

Sizes on both sides of the rule that chooses them (32768 and 65536 pixels on a
whole chip), waves that are partly filled, and counts of spheres, planes and
triangles around a multiple of four, so that quarters are uneven or empty.
Every output equals the plain schedule's, one lane a pixel, bit for bit.
"""
import numpy as np
import pytest

import scenes
import vkr
from gpu_util import gpu_trace

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    c = vkr.Context()
    yield c
    c.close()


def _scene(n_spheres, n_tris, n_planes):
    rng = scenes.rng_for(501, 100 * n_spheres + 10 * n_tris + n_planes)
    sph = scenes.light_sphere((0.0, 9.0, -4.0), 2.5)
    if n_spheres > 1:
        sph = np.concatenate([scenes.random_spheres(rng, n_spheres - 1, -9.0, 9.0,
                                                    kinds=("diffuse", "metal", "dielectric")), sph])
    tris = scenes.random_soup(rng, n_tris, lo=-8.0, hi=8.0, elo=2.0, ehi=9.0) if n_tris else np.zeros(0, vkr.TRIANGLE)
    M = scenes.reference_materials()
    normals = [(0, 1, 0), (1, 0, 0), (-1, 0, 0), (0, -1, 0), (0, 0, -1)][:n_planes]
    planes = (scenes.planes_from([M["matte_white"], M["matte_red"], M["matte_green"], M["matte_white"],
                                  M["matte_white"]][:n_planes], normals, [10.0, 12.0, 12.0, 12.0, 14.0][:n_planes])
              if n_planes else np.zeros(0, vkr.PLANE))
    return vkr.Scene(spheres=sph, tris=tris, planes=planes)


@pytest.mark.parametrize("size", [(1, 1), (17, 5), (64, 64), (181, 181), (182, 181), (256, 256), (257, 256)])
@pytest.mark.parametrize("counts", [(1, 0, 0), (2, 3, 1), (4, 4, 4), (6, 9, 5), (33, 0, 1), (23, 1, 2)],
                         ids=lambda c: "-".join(map(str, c)))
def test_four_lanes_give_the_image_of_one(ctx, counts, size):
    w, h = size
    cam = vkr.camera_from_angles((0.0, 0.0, -28.0), 0.0, 90.0)
    wl = scenes.Workload("quads", _scene(*counts), scenes.frame(cam, np.float32(w) / np.float32(h), 0.125), w, h, 2, 4)
    sid = ctx.upload(wl.scene)
    want = gpu_trace(ctx, sid, wl, sched=vkr.SCHED_PLAIN)
    for block in (0, 64):
        got = gpu_trace(ctx, sid, wl, sched=vkr.SCHED_PERSISTENT, block=block)
        for k in ("rgba8", "radiance", "prim_id", "hit_t", "ray_count"):
            assert np.array_equal(got[k].view(np.uint8), want[k].view(np.uint8)), (counts, size, block, k)
    ctx.destroy_scene(sid)
