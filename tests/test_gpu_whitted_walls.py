"""The Whitted kernel's walls: one division an axis inside the room, all five planes elsewhere.

Cameras and lights inside, on a wall's plane, outside every pair of walls, and
so far away or not finite that only the general test applies.  Every output
equals the oracle's bit for bit.
"""
import numpy as np
import pytest

import oracle_ffi
import scenes
import vkr
from gpu_util import compare, gpu_trace

pytestmark = pytest.mark.gpu

VIEWS = {"inside": ((10.0, 40.0, -30.0), (5.0, 64.0, 3.0)),
         "on_the_floor": ((3.0, 0.0, -20.0), (5.0, 0.0, 3.0)),
         "on_the_walls": ((64.0, 128.0, 64.0), (-64.0, 128.0, 64.0)),
         "above": ((0.0, 200.0, 10.0), (5.0, 300.0, 3.0)),
         "below": ((0.0, -50.0, 10.0), (5.0, -64.0, 3.0)),
         "left": ((-90.0, 30.0, 10.0), (-100.0, 64.0, 3.0)),
         "right": ((90.0, 30.0, 10.0), (100.0, 64.0, 3.0)),
         "behind_the_wall": ((0.0, 30.0, 100.0), (0.0, 64.0, 100.0)),
         "far": ((0.0, 1e20, 0.0), (1e30, 64.0, 0.0)),
         "infinite": ((np.inf, 30.0, 0.0), (0.0, np.inf, 0.0))}


@pytest.fixture(scope="module")
def ctx():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    c = vkr.Context()
    yield c
    c.close()


@pytest.mark.parametrize("pitch,yaw", [(0.0, 90.0), (-80.0, 10.0), (60.0, -100.0), (0.0, 180.0)])
@pytest.mark.parametrize("view", sorted(VIEWS))
def test_views(ctx, view, pitch, yaw):
    pos, light = VIEWS[view]
    w, h = 53, 47
    wl = scenes.reference_scene(w, h, 1, 1)
    wl.frame["camera"] = vkr.camera_from_angles((0.0, 0.0, 0.0), pitch, yaw)
    wl.frame["camera"]["pos"] = pos
    wl.frame["light_pos"] = light
    g = gpu_trace(ctx, 0, wl, kernel=vkr.KERNEL_WHITTED)
    r = oracle_ffi.trace(wl.scene, wl.frame, w, h, kernel=oracle_ffi.KERNEL_WHITTED)
    for k in ("rgba8", "prim_id", "ray_count"):
        assert np.array_equal(g[k].reshape(-1), r[k].reshape(-1)), (view, k)
    for k in ("radiance", "hit_t"):   # NaN for NaN: which NaN is not specified
        a, b = g[k].reshape(-1), r[k].reshape(-1)
        assert np.array_equal(np.isnan(a), np.isnan(b)), (view, k)
        n = ~np.isnan(a)
        assert np.array_equal(a[n].view(np.uint32), b[n].view(np.uint32)), (view, k)
