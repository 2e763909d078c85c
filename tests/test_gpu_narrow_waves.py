"""Waves that take fewer than 64 pixels.

Small images give each wave of the path kernel 1 to 32 pixels, by the image's
size and the scene's emitters.  The image must not depend on it: every frame
equals the plain schedule's (one pixel per lane, full waves) bit for bit, and
the pixels that leave a wave's share unfilled (sizes around the steps of the
rule, one pixel) are all there.
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


@pytest.fixture(scope="module")
def sids(ctx):
    wl = {"soup": scenes.soup100k(3, 2000, 64, 64, 2, 3, n_spheres=128),        # about 32 emitters, tree
          "few": scenes.soup100k(4, 500, 64, 64, 2, 3, n_spheres=9),            # two or three emitters
          "scan": scenes.many_emitters(40, 1),                                  # about 20 emitters, no tree
          "one": scenes.adjoint_scene(0, 64, 64, 2, 3)}                         # one emitter: single rays
    wl["scan"].scene.tris = wl["scan"].scene.tris[:4]
    return {k: (w, ctx.upload(w.scene)) for k, w in wl.items()}


@pytest.mark.parametrize("size", [(1, 1), (9, 7), (64, 64), (129, 65), (256, 255), (363, 363)])
@pytest.mark.parametrize("name", ["soup", "few", "scan", "one"])
def test_any_width_gives_the_plain_schedules_image(ctx, sids, name, size):
    base, sid = sids[name]
    w, h = size
    wl = scenes.Workload(name, base.scene, base.frame, w, h, 2, 3)
    want = gpu_trace(ctx, sid, wl, sched=vkr.SCHED_PLAIN)
    for block, chunk in ((0, 0), (64, 1), (256, 64)):
        got = gpu_trace(ctx, sid, wl, sched=vkr.SCHED_PERSISTENT, block=block, chunk=chunk)
        for k in ("rgba8", "radiance", "prim_id", "hit_t", "ray_count"):
            assert np.array_equal(got[k].view(np.uint8), want[k].view(np.uint8)), (name, size, block, chunk, k)
