"""Scenes of a few primitives, which the path kernel scans instead of traversing.

Sizes on both sides of the line between scan and tree (56 and 80 units, a
triangle counting two), coincident spheres and planes (whose winner depends on
the scan order), a camera so far away that the distance estimates settle
nothing, and epsilons around the estimates' error.  Every output equals the
oracle's linear scan bit for bit.
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


def _check(ctx, wl, epsilon=1e-3, flags=0):
    sid = ctx.upload(wl.scene)
    g = gpu_trace(ctx, sid, wl, flags=flags) if epsilon == 1e-3 else _trace_eps(ctx, sid, wl, epsilon)
    ctx.destroy_scene(sid)
    r = oracle_ffi.trace(wl.scene, wl.frame, wl.width, wl.height, wl.spp, wl.max_depth, epsilon=epsilon)
    st = compare(g, r)
    for k in ("prim_id", "hit_t_bits", "radiance_bits", "rgba8", "ray_count"):
        assert st[k] == 1.0, (k, st)


def _trace_eps(ctx, sid, wl, epsilon):
    class W:
        width, height, spp, frame = wl.width, wl.height, wl.spp, wl.frame
        params = staticmethod(lambda **kw: wl.params(epsilon=epsilon, **kw))
    return gpu_trace(ctx, sid, W)


def _workload(spheres, tris=None, planes=None, w=45, h=31, spp=2, depth=4, cam=None):
    cam = vkr.camera_from_angles((0.0, 0.0, -28.0), 0.0, 90.0) if cam is None else cam
    sc = vkr.Scene(spheres=spheres, tris=np.zeros(0, vkr.TRIANGLE) if tris is None else tris,
                   planes=scenes.ground(-10.0) if planes is None else planes)
    return scenes.Workload("scan", sc, scenes.frame(cam, np.float32(w) / np.float32(h), 0.125), w, h, spp, depth)


@pytest.mark.parametrize("kinds", [("diffuse", "metal", "dielectric"), ("diffuse", "dielectric", "emissive")],
                         ids=["one_light", "many_lights"])
@pytest.mark.parametrize("n_spheres,n_tris", [(0, 0), (0, 1), (1, 0), (3, 4), (55, 0), (56, 0), (79, 0), (80, 0), (7, 30)])
def test_sizes(ctx, n_spheres, n_tris, kinds):
    rng = scenes.rng_for(401, 100 * n_spheres + n_tris)
    sph = scenes.random_spheres(rng, n_spheres, -10.0, 10.0, kinds=kinds) if n_spheres else np.zeros(0, vkr.SPHERE)
    if n_spheres:
        sph[-1:] = scenes.light_sphere((0.0, 9.0, -4.0), 1.5)
    tris = scenes.random_soup(rng, n_tris, lo=-8.0, hi=8.0, elo=2.0, ehi=9.0) if n_tris else None
    _check(ctx, _workload(sph, tris))


def test_reference_room(ctx):
    """Five planes meeting in edges and corners, glass, mirror, light and a triangle."""
    _check(ctx, scenes.reference_scene(96, 64, 3, 6))


def test_ties_follow_the_scan_order(ctx):
    """Copies of one sphere, spheres and planes a fraction of epsilon apart."""
    rng = scenes.rng_for(402, 0)
    sph = scenes.random_spheres(rng, 6, -6.0, 6.0, kinds=("diffuse", "metal"))
    near = sph.copy()
    near["P"][:, 2] += np.float32(4e-4)
    near["mat"]["albedo"] = near["mat"]["albedo"][::-1]
    sph = np.concatenate([sph, sph, near, scenes.light_sphere((0.0, 9.0, -4.0), 1.5)])
    M = scenes.reference_materials()
    planes = scenes.planes_from([M["matte_white"], M["matte_red"], M["matte_green"]],
                                [(0, 1, 0), (0, 1, 0), (0, 1, 0)], [9.0, 9.0005, 8.9995])
    _check(ctx, _workload(sph, planes=planes, w=64, h=48))


def test_far_camera(ctx):
    wl = scenes.far_sphere(64)
    wl.scene.tris = wl.scene.tris[:8]
    _check(ctx, wl)


@pytest.mark.parametrize("epsilon", [1e-6, 3e-5, 1e-2])
def test_epsilons(ctx, epsilon):
    rng = scenes.rng_for(403, 0)
    sph = np.concatenate([scenes.random_spheres(rng, 20, -8.0, 8.0), scenes.light_sphere((0.0, 9.0, -4.0), 1.5)])
    _check(ctx, _workload(sph, scenes.random_soup(rng, 3, lo=-6.0, hi=6.0, elo=2.0, ehi=6.0)), epsilon=epsilon)


def test_batch_of_small_scenes(ctx):
    """Waves that hold pixels of several jobs scan each job's scene in turn."""
    import torch
    jobs, want, outs, sids = [], [], [], []
    for i in range(5):
        rng = scenes.rng_for(404, i)
        sph = scenes.random_spheres(rng, 3 + 9 * i, -8.0, 8.0)
        sph = np.concatenate([sph, scenes.light_sphere((0.0, 9.0, -4.0), 1.5)])
        wl = _workload(sph, w=13 + 4 * i, h=11, spp=1 + i)
        sids.append(ctx.upload(wl.scene))
        n = wl.width * wl.height
        out = torch.zeros((n, 4), dtype=torch.float32, device="cuda")
        outs.append(out)
        jobs.append(ctx.job(sids[-1], wl.frame, wl.params(), radiance=out))
        want.append(oracle_ffi.trace(wl.scene, wl.frame, wl.width, wl.height, wl.spp, wl.max_depth)["radiance"])
    ctx.trace_batch(jobs)
    torch.cuda.synchronize()
    for out, w in zip(outs, want):
        assert np.array_equal(out.cpu().numpy().view(np.uint32), w.view(np.uint32))
    for sid in sids:
        ctx.destroy_scene(sid)
