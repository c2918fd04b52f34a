"""IC-GN from the handed-out table (LUT, B-spline) in both lane layouts: 33,000
POIs run on half-wavefronts, 20,000 of them on whole ones.  The layouts differ in
the order of their FP64 partial sums, so the flags must be equal, the iteration
counts equal on at least 99.9 % of the POIs, and u, v and the gradients equal to
1e-5 px and 1e-7 where the counts agree; a sample of the large set is held to the
oracle's bars."""
import numpy as np
import pytest

import oracle
from tests import cases
from tests.gpu_helpers import check_icgn, ctx_for, run_icgn
from tw_amd import api

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("interp", [api.INTERP_LUT, api.INTERP_BSPLINE])
@pytest.mark.parametrize("S", [10, 16])
def test_table_layouts_agree(S, interp):
    print(f"[gpu-test] table, mode {interp} S {S}", flush=True)
    c = cases.speckle_512()
    c.S, c.margin = S, 0
    if interp == api.INTERP_BSPLINE:
        c.roi = (1, 1, 508, 508)
    rng = np.random.default_rng(S)
    poi = rng.integers(40, 470, (33000, 2)).astype(np.int32)
    u0, v0 = np.full(len(poi), 2, np.float32), np.full(len(poi), -2, np.float32)
    sub = np.sort(rng.choice(len(poi), 20000, replace=False))
    with ctx_for(c, interp=interp) as ctx:
        ctx.buffer(api.BUF_LUT)                                     # handed out: read from here on
        big = run_icgn(ctx, poi, u0, v0)
        small = run_icgn(ctx, np.ascontiguousarray(poi[sub]), u0[sub], v0[sub])
    b = {k: a[sub] for k, a in big.items()}
    assert np.array_equal(b["flags"], small["flags"]) and (b["flags"] == 0).mean() > 0.99
    same = b["iters"] == small["iters"]
    assert same.mean() >= 0.999, same.mean()
    du = np.maximum(np.abs(b["u"] - small["u"]), np.abs(b["v"] - small["v"]))[same]
    dg = np.abs(b["p6"][:, [1, 2, 4, 5]] - small["p6"][:, [1, 2, 4, 5]])[same]
    assert du.max() <= 1e-5 and dg.max() <= 1e-7, (du.max(), dg.max())
    idx = np.sort(rng.choice(len(poi), 128, replace=False))
    mode = "bspline" if interp == api.INTERP_BSPLINE else "bicubic"
    sp = np.ascontiguousarray(poi[idx])
    o = oracle.icgn(c.ref, c.tar, c.roi, S, S, sp, u0[idx], v0[idx], interp=mode)
    o64 = oracle.icgn(c.ref, c.tar, c.roi, S, S, sp, u0[idx].astype(np.float64), v0[idx].astype(np.float64),
                      precision="f64", interp=mode)
    # the FP32 path's own distance from FP64, as in the lane-layout test of the other layouts
    ok = (o["iters"] == o64["iters"]) & (o["flags"] == 0)
    own_u = float(np.max(np.maximum(np.abs(o["u"] - o64["u"]), np.abs(o["v"] - o64["v"]))[ok]))
    own_g = float(np.max(np.abs(o["p6"][:, [1, 2, 4, 5]] - o64["p6"][:, [1, 2, 4, 5]])[ok]))
    own = int(np.count_nonzero(o["iters"] != o64["iters"]))
    check_icgn({k: a[idx] for k, a in big.items()}, o, utol=max(1e-4, 2 * own_u), gtol=max(1e-6, 2 * own_g),
               max_flips=max(2, 3 * own + 2))
