"""IC-GN's three loops over the row polynomials (cells kept from row to row for
gentle warps, loaded pixel by pixel for steep ones, with the per-pixel tests
near the ROI's border) take the same sums in the same order from the same
values: the same POIs give the same bits whichever runs."""
import numpy as np
import pytest

from tw_amd import api

pytestmark = pytest.mark.gpu

SIZE, X = 220, 110


def _run(pair, rw, S, interp, poi):
    cfg = api.make_config(SIZE, SIZE, 1, 1, rw, SIZE - 2, S, S, 5, 5, 0, 0, 32, interp=interp)
    n = len(poi)
    with api.Context(cfg) as ctx:
        ctx.set_reference(pair[0])
        ctx.set_target(pair[1])
        dp = ctx.array(poi.shape, np.int32).upload(poi)
        u = ctx.array(n, np.float32).upload(np.full(n, 1, np.float32))
        v = ctx.array(n, np.float32).upload(np.full(n, -1, np.float32))
        p6 = ctx.array((n, 6), np.float32).fill(0)
        it, fl = ctx.array(n, np.int32).fill(0), ctx.array(n, np.uint8).fill(255)
        ctx.icgn(dp, n, u, v, p6, it, fl)
        return p6.download(), it.download(), fl.download()


@pytest.mark.parametrize("interp", [api.INTERP_FUSED, api.INTERP_LUT])
@pytest.mark.parametrize("strain", [0.0, 0.003, 0.0055, 0.012, 0.03])
@pytest.mark.parametrize("S", [9, 15, 20])
def test_the_loops_agree_bitwise(S, strain, interp):
    d = api.affine(1.3, -0.8, 0.1 * strain, 0.6 * strain, -0.4 * strain, X, SIZE / 2)
    pair = api.synth_pair(SIZE, SIZE, 700, 31, d)
    poi = np.array([(y, X) for y in range(60, 160, 3)], np.int32)
    print(f"[gpu-test] steep S {S} strain {strain} interp {interp}", flush=True)
    wide = _run(pair, SIZE - 2, S, interp, poi)
    # the right border within a pixel of where the subsets' last columns come to lie
    tight = _run(pair, X + S + 2, S, interp, poi)
    assert (wide[2] == 0).sum() >= 0.9 * len(poi)
    # the ROI's last column reads as zero, so only subsets that keep off it are the same in both
    p = wide[0].astype(np.float64)
    last = X + S + p[:, 0] + S * (np.abs(p[:, 1]) + np.abs(p[:, 2]))
    ok = (tight[2] == 0) & (wide[2] == 0) & (last <= X + S + 1.5)
    assert ok.sum() >= 0.25 * len(poi)
    for a, b in zip(wide, tight):
        assert np.array_equal(a[ok], b[ok])
