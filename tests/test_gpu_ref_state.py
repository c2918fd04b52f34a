"""The per-POI reference state (Hessian factor, steepest-descent sums), whose
moments are summed in 32-bit integers down row ranges of a subset column, on
images that drive those sums to their limits: 0 / 255 stripes with central
differences of +-255 everywhere, and random 0 / 255 pixels, with subsets up to
the largest, one POI per wavefront (few POIs) and per half-wavefront.

One IC-GN iteration from integer guesses uses only that state and exact integer
sums, so against the FP64 oracle it differs by the FP32 rounding of dp and of
the update: six roundings of 2^-24 on terms below |u| + |dp| + 1 for the shift,
and of terms below 2 for the gradients (the update's products are of order one
while |dp| stays below 1/2, which the test checks)."""
import numpy as np
import pytest

import oracle
from tw_amd import api

pytestmark = pytest.mark.gpu

SIZE, ROI = 300, (1, 1, 298, 298)


def _image(kind):
    rng = np.random.default_rng(kind)
    y, x = np.mgrid[0:SIZE, 0:SIZE]
    if kind == 0:                                       # |gx| = 255 in most pixels
        img = ((x // 2) & 1) * 255
        flip = rng.random((SIZE, SIZE)) < 0.02
    elif kind == 1:                                     # |gx| = |gy| = 255: the mixed moments too
        img = (((x + y) // 2) & 1) * 255
        flip = rng.random((SIZE, SIZE)) < 0.02
    else:
        img, flip = rng.integers(0, 2, (SIZE, SIZE)) * 255, np.zeros((SIZE, SIZE), bool)
    return np.where(flip, 255 - img, img).astype(np.uint8)


@pytest.mark.parametrize("kind", [0, 1, 2])
@pytest.mark.parametrize("sx,sy,n", [(20, 20, 90), (20, 20, 5000), (27, 28, 5000), (30, 30, 90), (30, 30, 5000),
                                     (60, 60, 90), (60, 60, 5000), (5, 60, 5000)])
def test_integer_moments_at_their_limits(kind, sx, sy, n):
    print(f"[gpu-test] reference state kind {kind} subset {sx} {sy} POIs {n}", flush=True)
    ref = _image(kind)
    rng = np.random.default_rng(100 + kind)
    noise = rng.integers(-6, 7, ref.shape)
    tar = np.clip(ref.astype(np.int32) * 0.9 + 12 + noise, 0, 255).astype(np.uint8)
    poi = rng.integers(62, SIZE - 62, (n, 2)).astype(np.int32)
    zero = np.zeros(n, np.float32)
    cfg = api.make_config(SIZE, SIZE, *ROI, sx, sy, 5, 5, 0, 0, 32, max_iter=1, delta_p=0.0)
    with api.Context(cfg) as ctx:
        ctx.set_reference(ref)
        ctx.set_target(tar)
        dp = ctx.array(poi.shape, np.int32).upload(poi)
        u, v = ctx.array(n, np.float32).upload(zero), ctx.array(n, np.float32).upload(zero)
        p6, fl = ctx.array((n, 6), np.float32).fill(0), ctx.array(n, np.uint8).fill(255)
        ctx.icgn(dp, n, u, v, p6, None, fl)
        ctx.sync()
        got, flags = p6.download()[:90].astype(np.float64), fl.download()[:90]
    sample = np.ascontiguousarray(poi[:90])
    z = np.zeros(90)
    o = oracle.icgn(ref, tar, ROI, sx, sy, sample, z, z, max_iter=1, delta_p=0.0, precision="f64")
    assert np.array_equal(flags, o["flags"]) and (flags == oracle.SUCCESS).all()
    err, want = np.abs(got - o["p6"]), np.abs(o["p6"])
    assert want.max() < 0.5
    assert np.all(err[:, [0, 3]] <= 6 * 2.0 ** -24 * (2 * want[:, [0, 3]] + 1)), err[:, [0, 3]].max()
    assert np.all(err[:, [1, 2, 4, 5]] <= 6 * 2.0 ** -24 * 2), err[:, [1, 2, 4, 5]].max()
