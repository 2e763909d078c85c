"""Reciprocals and square roots made of an estimate and one Newton step.

The triangle test's 1 / det and the sphere test's sqrt(h) must be the nearest
floats, over every exponent: inside [2^-64, 2^64), where the short form is
used, at its two ends, and beyond them, where the division and the root are.
Expected values are numpy's float32 operations, which round to nearest.
"""
import numpy as np
import pytest

import vkr

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    c = vkr.Context()
    yield c
    c.close()


def _eval(ctx, op, inp):
    import torch
    i = torch.from_numpy(np.ascontiguousarray(inp, np.float32)).cuda()
    o = torch.zeros((len(inp), 8), dtype=torch.float32, device="cuda")
    ctx.debug_eval(op, i, o)
    torch.cuda.synchronize()
    return o.cpu().numpy()[:, 0]


def _same(got, want):
    return np.array_equal(got.view(np.uint32), want.view(np.uint32))


def _tri_inputs(x):
    """Triangle v0 = 0, e1 = (x, 0, 1), e2 = (0, -1, 0); ray from (x / 2, 0, 0) along z: det = x, u = 1/2 (or the
    float next to it), v = 0 and t = (x / 2) * (1 / x rounded)."""
    inp = np.zeros((len(x), 16), np.float32)
    inp[:, 0] = x * np.float32(0.5)
    inp[:, 5] = 1.0
    inp[:, 9], inp[:, 11] = x, 1.0
    inp[:, 13] = -1.0
    inp[:, 15] = 1e-38
    return inp


def _check_tri(ctx, x):
    with np.errstate(all="ignore"):
        want = (x * np.float32(0.5)) * (np.float32(1.0) / x)
    assert _same(_eval(ctx, "tri", _tri_inputs(x)), want)


def test_reciprocal_of_every_mantissa(ctx):
    """t is a multiple of the reciprocal that keeps its bits apart: from o.x = 1 it is the reciprocal itself."""
    for k in range(8):
        x = (np.arange(1 << 20, dtype=np.uint32) + np.uint32(0x3F800000 + (k << 20))).view(np.float32)
        inp = _tri_inputs(x)
        inp[:, 0] = 1.0
        assert _same(_eval(ctx, "tri", inp), np.float32(1.0) / x)


@pytest.mark.parametrize("exponent", [-125, -65, -64, -63, -1, 0, 62, 63, 64, 65, 126])
def test_reciprocal_exponents(ctx, exponent):
    rng = np.random.default_rng(exponent + 200)
    x = np.ldexp(1.0 + rng.random(4096), exponent).astype(np.float32)
    x[:2] = np.float32(2.0 ** exponent), np.nextafter(np.float32(2.0 ** exponent), np.float32(np.inf))
    _check_tri(ctx, x)


@pytest.mark.parametrize("exponent", [-66, -33, -32, -31, -30, -1, 0, 1, 29, 30, 31, 32, 60])
def test_root_exponents(ctx, exponent):
    """A ray that starts at the centre of a sphere of radius 1 with d = (dx, 0, 0) from o = c + (1, 0, 0):
    h = (2 dx)^2 rounded, t = (-2 dx - sqrt(h)) / 2."""
    rng = np.random.default_rng(exponent + 300)
    dx = np.ldexp(1.0 + rng.random(1 << 16), exponent).astype(np.float32)
    inp = np.zeros((len(dx), 16), np.float32)
    inp[:, 0] = 1.0
    inp[:, 3] = dx
    inp[:, 9] = 1.0
    b = np.float32(2.0) * dx
    want = (-b - np.sqrt(b * b)) / np.float32(2.0)
    assert _same(_eval(ctx, "sphere", inp), want)


def test_root_of_zero(ctx):
    inp = np.zeros((2, 16), np.float32)
    inp[:, 0] = 1.0, -1.0
    inp[:, 9] = 1.0
    assert np.array_equal(_eval(ctx, "sphere", inp), np.zeros(2, np.float32))
