"""The LUT and B-spline interpolation modes read layouts of their own (the
target's row polynomials, and planes of coefficients) as long as the LUT buffer
has not been handed out (twdic_get_buffer), and the LUT itself from then on.
Both evaluate the same cell polynomials in the same order from the same or
exact coefficients, so every output must be equal bit for bit; the LUT handed out
must be the current target's, from the calls that ran before and after, eager
and through a captured frame."""
import numpy as np
import pytest

import oracle
from tests import cases
from tests.gpu_helpers import ctx_for
from tw_amd import api

pytestmark = pytest.mark.gpu

OUT = dict(u=np.float32, v=np.float32, zncc=np.float32, p6=np.float32, iters=np.int32, flags=np.uint8)


def _frame(ctx, dpoi, n, replay=False):
    o = getattr(ctx, "_out", None)
    if o is None:
        o = ctx._out = {k: ctx.array((n, 6) if k == "p6" else n, d) for k, d in OUT.items()}
    args = (dpoi, n, *(o[k] for k in OUT))
    if replay:
        ctx.frame_replay()
    else:
        ctx.frame(*args)
    ctx.sync()
    return {k: a.download() for k, a in o.items()}, args


def _lut(ctx, c):
    _, _, w, h = c.roi
    return ctx.download_buffer(api.BUF_LUT, (h, w, 16), np.float32)


@pytest.mark.parametrize("S", [10, 15, 24])
@pytest.mark.parametrize("interp", [api.INTERP_LUT, api.INTERP_BSPLINE])
def test_own_layout_and_table_agree_bitwise(interp, S):
    c = cases.speckle_512()
    c.S, c.margin = S, 0
    table_of = oracle.bicubic_lut
    if interp == api.INTERP_BSPLINE:
        c.roi, table_of = (1, 1, 508, 508), oracle.bspline_lut
    tar2 = np.ascontiguousarray(np.roll(c.tar, 1, axis=1))
    poi = np.random.default_rng(S).integers(60, 452, (700, 2)).astype(np.int32)
    print(f"[gpu-test] interpolation mode {interp} S {S}", flush=True)
    with ctx_for(c, interp=interp) as plane, ctx_for(c, interp=interp) as table:
        table.buffer(api.BUF_LUT)                                   # handed out before the first call
        pd, td = (x.array(poi.shape, np.int32).upload(poi) for x in (plane, table))
        for k, tar in enumerate((c.tar, tar2)):
            for x in (plane, table):
                x.set_target(tar)
            a, args = _frame(plane, pd, len(poi))
            b, _ = _frame(table, td, len(poi))
            assert (b["flags"] == 0).mean() > 0.9
            for f in OUT:
                assert np.array_equal(a[f], b[f]), (k, f)
            assert np.array_equal(_lut(table, c), table_of(tar, *c.roi))
        plane.frame_capture(*args)
        plane.set_target(c.tar)
        table.set_target(c.tar)
        b, _ = _frame(table, td, len(poi))
        for handed in (False, True):
            if handed:                                              # the replay's target, then kept up
                assert np.array_equal(_lut(plane, c), table_of(c.tar, *c.roi))
                plane.set_target(tar2)
                _frame(plane, pd, len(poi), replay=True)
                assert np.array_equal(_lut(plane, c), table_of(tar2, *c.roi))
                plane.set_target(c.tar)
            a, _ = _frame(plane, pd, len(poi), replay=True)
            for f in OUT:
                assert np.array_equal(a[f], b[f]), (handed, f)
        a, _ = _frame(plane, pd, len(poi))                          # eager, from the table now
        for f in OUT:
            assert np.array_equal(a[f], b[f]), f
