"""Device arithmetic that reaches a float's rounding another way than a float operation.

cos and sin are evaluated twice over when the short evaluation cannot tell
which float is nearest; normalize and the quotients by one divisor go through
double reciprocals.  The arguments here are the ones where that shows: angles
whose cosine or sine lies next to the midpoint of two floats, angles past the
short evaluation's range, and vectors whose squared length is zero, denormal
or infinite.  Expected values are exact: the nearest float of a double
evaluation, and the oracle's jitter (two normalisations).
"""
import numpy as np
import pytest

import oracle_ffi
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
    return o.cpu().numpy()


def _near_midpoint(x, f, ulps):
    """The x whose f(x) in double is within `ulps` of the midpoint of two floats, but not so near that the double
    evaluation's own error (an ulp) could decide the rounding."""
    low = f(x.astype(np.float64)).view(np.uint64) & np.uint64(0x1FFFFFFF)
    d = np.abs(low.astype(np.int64) - 0x10000000)
    return x[(d <= ulps) & (d >= 8)]


@pytest.mark.parametrize("scale", [6.2831853, 1e3, 2e5, 1e9])
def test_cos_sin_next_to_midpoints(ctx, scale):
    x = (np.random.default_rng(int(scale)).random(3_000_000) * scale).astype(np.float32)
    sel = np.concatenate([_near_midpoint(x, np.cos, 1 << 14), _near_midpoint(x, np.sin, 1 << 14), x[:4096]])
    assert len(sel) > 4096 + 100
    inp = np.zeros((len(sel), 16), np.float32)
    inp[:, 0] = sel
    out = _eval(ctx, "cos", inp)
    for col, f in ((0, np.cos), (1, np.sin)):
        want = f(sel.astype(np.float64)).astype(np.float32)
        assert np.array_equal(out[:, col].view(np.uint32), want.view(np.uint32)), (scale, col)


def test_cos_sin_not_finite(ctx):
    inp = np.zeros((3, 16), np.float32)
    inp[:, 0] = (np.inf, -np.inf, np.nan)
    out = _eval(ctx, "cos", inp)
    assert np.isnan(out[:, :2]).all()


def test_jitter_lengths(ctx):
    """jitter normalises its direction and a cross product of it."""
    rng = np.random.default_rng(5)
    d = rng.normal(size=(40_000, 3)) * 10.0 ** rng.uniform(-25, 20, (40_000, 1))
    d = d.astype(np.float32)
    d[:6] = [(0, 0, 0), (1e-30, 0, 0), (3e38, 3e38, 0), (np.inf, 1, 0), (0, -0.0, 2), (1e-45, 1e-45, 1e-45)]
    inp = np.zeros((len(d), 16), np.float32)
    inp[:, 0:3] = d
    inp[:, 3] = rng.uniform(0, 6.2831853, len(d))
    inp[:, 4] = rng.uniform(0, 1, len(d))
    inp[:, 5] = np.sqrt(1 - inp[:, 4] ** 2)
    out = _eval(ctx, "jitter", inp)[:, :3]
    lib = oracle_ffi.load()
    for i in range(len(d)):
        want = oracle_ffi.F3()
        lib.vkro_jitter(oracle_ffi.f3(inp[i, 0:3]), float(inp[i, 3]), float(inp[i, 4]), float(inp[i, 5]), want)
        w = np.array(want, np.float32)
        assert np.array_equal(np.isnan(w), np.isnan(out[i])), (i, d[i], w, out[i])
        ok = ~np.isnan(w)
        assert np.array_equal(w[ok].view(np.uint32), out[i][ok].view(np.uint32)), (i, d[i], w, out[i])
