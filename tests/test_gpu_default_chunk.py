"""The refill threshold that a launch takes when its caller names none.

It depends on how the scene is traced and on the sample count (64 for one ray
a lane over a scanned scene while spp times bounces is at most 32, for other
batches 32, else 8): images
on both sides of each line, of sizes whose last tiles are partly outside and
that take more pixels than the waves hold at once, equal the plain schedule's
bit for bit.
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


def _workload(kind, w, h, spp):
    if kind == "scan":
        wl = scenes.reference_scene(w, h, spp, 3)
    elif kind == "tree":
        wl = scenes.adjoint_scene(0, w, h, spp, 3)
        rng = scenes.rng_for(701, 0)
        wl.scene.tris = scenes.random_soup(rng, 300, lo=-8.0, hi=8.0)
    else:
        wl = scenes.many_emitters(40, 1)
    return scenes.Workload(kind, wl.scene, wl.frame, w, h, spp, 3)


@pytest.mark.parametrize("spp", [1, 10, 11])
@pytest.mark.parametrize("kind", ["scan", "tree", "pool"])
def test_frames(ctx, kind, spp):
    w, h = (1027, 517) if kind != "pool" else (131, 67)
    wl = _workload(kind, w, h, spp)
    sid = ctx.upload(wl.scene)
    want = gpu_trace(ctx, sid, wl, sched=vkr.SCHED_PLAIN)
    got = gpu_trace(ctx, sid, wl)
    for k in ("rgba8", "radiance", "prim_id", "hit_t", "ray_count"):
        assert np.array_equal(got[k].view(np.uint8), want[k].view(np.uint8)), (kind, spp, k)
    ctx.destroy_scene(sid)


@pytest.mark.parametrize("spp", [10, 11])
@pytest.mark.parametrize("kinds", [("scan", "scan"), ("scan", "tree", "pool"), ("scan",)])
def test_batches(ctx, kinds, spp):
    import torch
    wls = [_workload(k, 601 + 8 * i, 397, spp if i == 0 else 2) for i, k in enumerate(kinds)]
    sids = [ctx.upload(wl.scene) for wl in wls]
    outs = [torch.zeros((wl.width * wl.height, 4), dtype=torch.float32, device="cuda") for wl in wls]
    ctx.trace_batch([ctx.job(s, wl.frame, wl.params(), radiance=o) for s, wl, o in zip(sids, wls, outs)])
    torch.cuda.synchronize()
    for s, wl, o in zip(sids, wls, outs):
        want = gpu_trace(ctx, s, wl, sched=vkr.SCHED_PLAIN)["radiance"]
        got = o.cpu().numpy()
        assert np.array_equal(got.reshape(-1).view(np.uint32), np.ascontiguousarray(want).reshape(-1).view(np.uint32))
        ctx.destroy_scene(s)
