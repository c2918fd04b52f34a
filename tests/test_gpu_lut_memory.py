"""Device memory of the LUT and B-spline modes.  The layouts that IC-GN reads
while the LUT is not handed out (16 and 64 bytes per ROI pixel) are an addition
to the LUT: a context is created without them where only the LUT fits, with the
same results, and they are given back when the LUT is handed out before they
were used."""
import ctypes as C

import numpy as np
import pytest

from tw_amd import api

pytestmark = pytest.mark.gpu

SIZE = 4096
EXTRA = {api.INTERP_LUT: 16, api.INTERP_BSPLINE: 64}


def _free(hip):
    free, total = C.c_size_t(), C.c_size_t()
    assert hip.hipMemGetInfo(C.byref(free), C.byref(total)) == 0
    return free.value


def _config(interp):
    return api.make_config(SIZE, SIZE, 1, 1, SIZE - 3, SIZE - 3, 10, 10, 8, 8, 30, 30, 32, interp=interp)


def _results(interp, ref, tar, poi):
    with api.Context(_config(interp)) as c:
        c.set_reference(ref)
        c.set_target(tar)
        n = len(poi)
        dp = c.array(poi.shape, np.int32).upload(poi)
        o = [c.array(n, np.float32).fill(0) for _ in range(3)]
        p6, fl = c.array((n, 6), np.float32).fill(0), c.array(n, np.uint8).fill(255)
        c.frame(dp, n, *o, p6, None, fl)
        c.sync()
        return [a.download() for a in (*o, p6, fl)]


@pytest.mark.parametrize("interp", [api.INTERP_LUT, api.INTERP_BSPLINE])
def test_created_where_only_the_table_fits(interp):
    hip = C.CDLL("libamdhip64.so")
    rng = np.random.default_rng(3)
    ref = rng.integers(0, 256, (SIZE, SIZE)).astype(np.uint8)
    tar = np.roll(ref, (2, -1), (0, 1))
    poi = rng.integers(60, SIZE - 60, (400, 2)).astype(np.int32)
    want = _results(interp, ref, tar, poi)
    px = (SIZE - 3) ** 2
    before = _free(hip)
    ctx = api.Context(_config(interp))
    need = before - _free(hip) - EXTRA[interp] * px       # what the context takes without the addition
    ctx.close()
    print(f"[gpu-test] mode {interp}: {need} bytes without the layout, {_free(hip)} free", flush=True)
    # all but that and half of the addition, in pieces
    hog, left = [], _free(hip) - need - EXTRA[interp] * px // 2
    try:
        while left > (64 << 20):
            p, b = C.c_void_p(), min(left, 8 << 30)
            assert hip.hipMalloc(C.byref(p), C.c_size_t(b)) == 0
            hog.append(p)
            left = _free(hip) - need - EXTRA[interp] * px // 2
        got = _results(interp, ref, tar, poi)
    finally:
        for p in hog:
            hip.hipFree(p)
    assert (want[4] == 0).mean() > 0.9
    for a, b in zip(got, want):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("interp", [api.INTERP_LUT, api.INTERP_BSPLINE])
def test_given_back_when_the_table_is_handed_out_first(interp):
    hip = C.CDLL("libamdhip64.so")
    with api.Context(_config(interp)) as c:
        held = _free(hip)
        c.buffer(api.BUF_LUT)
        assert _free(hip) - held >= 0.9 * EXTRA[interp] * (SIZE - 3) ** 2
