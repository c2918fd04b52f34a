"""IC-GN's walk over the subset (strips of columns, each column cut into row
ranges, one lane per column and range; twdic_internal.h strip_plan) at subset
sizes where it can go wrong: one strip and several, strips one column wide,
ranges of unequal length, the largest subset, subsets far from square, with
half- and whole-wavefronts.

After one iteration the sums are sums of integers, exact in FP64 on both
sides, so the result differs from the FP64 oracle's by the FP32 rounding of
the update alone: the six components of dp (2^-24 relative), then for u at
most four more roundings of terms below |u| + 1, and for the gradients four of
terms near 1, i.e. 5 x 2^-24 (|u| + 1) and 5 x 2^-24.  (The bicubic passes
walk the same table; the sweep and parity tests hold them to the oracle.)"""
import numpy as np
import pytest

import oracle
from tw_amd import api

pytestmark = pytest.mark.gpu

SIZE, ROI = 420, (1, 1, 418, 418)


@pytest.fixture(scope="module")
def pair():
    d = api.affine(1.3, -0.8, 0.004, -0.003, 0.002, SIZE / 2, SIZE / 2)
    return api.synth_pair(SIZE, SIZE, int(0.015 * SIZE * SIZE), 8101, d, noise_sigma=2.0)


@pytest.mark.parametrize("half", [False, True])
@pytest.mark.parametrize("sx,sy", [(3, 3), (7, 9), (15, 15), (16, 16), (22, 23), (31, 32), (4, 60), (60, 5), (60, 60)])
def test_strip_walk_against_oracle(pair, sx, sy, half):
    ref, tar = pair
    print(f"[gpu-test] strips sx {sx} sy {sy} half {half}", flush=True)
    at = np.arange(117, 117 + 182)                      # 33,124 POIs: half-wavefronts
    yy, xx = np.meshgrid(at, at, indexing="ij")
    poi = np.stack([yy.ravel(), xx.ravel()], 1).astype(np.int32)
    pick = np.sort(np.random.default_rng(10 * sx + sy).choice(len(poi), 96, replace=False))
    if not half:
        poi, pick = np.ascontiguousarray(poi[pick]), np.arange(96)
    sample = np.ascontiguousarray(poi[pick])
    u0, v0 = np.full(len(poi), 1, np.float32), np.full(len(poi), -1, np.float32)
    cfg = api.make_config(SIZE, SIZE, *ROI, sx, sy, 5, 5, 0, 0, 32, max_iter=1, delta_p=0.0)
    with api.Context(cfg) as ctx:
        ctx.set_reference(ref)
        ctx.set_target(tar)
        dp = ctx.array(poi.shape, np.int32).upload(poi)
        u, v = ctx.array(len(poi), np.float32).upload(u0), ctx.array(len(poi), np.float32).upload(v0)
        p6 = ctx.array((len(poi), 6), np.float32).fill(0)
        fl = ctx.array(len(poi), np.uint8).fill(255)
        ctx.icgn(dp, len(poi), u, v, p6, None, fl)
        ctx.sync()
        got, flags = p6.download()[pick].astype(np.float64), fl.download()[pick]
    o = oracle.icgn(ref, tar, ROI, sx, sy, sample, u0[pick].astype(np.float64), v0[pick].astype(np.float64),
                    max_iter=1, delta_p=0.0, precision="f64")
    assert np.array_equal(flags, o["flags"])
    ok = flags == oracle.SUCCESS
    assert ok.sum() >= 90
    err, want = np.abs(got - o["p6"])[ok], np.abs(o["p6"])[ok]
    shift, grad = err[:, [0, 3]], err[:, [1, 2, 4, 5]]
    assert np.all(shift <= 5 * 2.0 ** -24 * (want[:, [0, 3]] + 1)), shift.max()
    assert np.all(grad <= 5 * 2.0 ** -24), grad.max()
