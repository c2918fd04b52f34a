"""A server whose device budget is exactly what twdic_serve.h says one request
needs (the reference and its gradients, the POIs and their state, the frame, 16
(w - 2) (h - 1) bytes of row polynomials and 41 bytes per POI, each rounded up
to 256 bytes) takes that request."""
import numpy as np
import pytest

from tw_amd import api

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("w,h", [(256, 256), (333, 257), (700, 130)])
def test_a_request_fits_the_budget_it_is_said_to_need(w, h):
    S, N = 10, 32
    ref, tar = api.synth_pair(w, h, int(0.015 * w * h), 9, api.affine(1.2, -0.6, 0.002, 0.001, -0.001, w / 2, h / 2))
    yy, xx = np.meshgrid(np.arange(30, h - 30, 12), np.arange(30, w - 30, 12), indexing="ij")
    poi = np.stack([yy.ravel(), xx.ravel()], 1).astype(np.int32)
    n = len(poi)
    up = lambda b: (b + 255) // 256 * 256  # noqa: E731
    budget = (up(up(w * h) + 4 * (w - 2) * (h - 2)) + up(8 * n) + up(384 * n)
              + up(up(w * h) + up(16 * (w - 2) * (h - 1)) + 41 * n))
    print(f"[gpu-test] serve budget {w} x {h}: {budget}", flush=True)
    with api.Server(slots=1, queue_capacity=2, hbm_budget=budget, max_width=w, max_height=h, max_pois=n) as srv:
        srv.set_reference(0, ref)
        pid = srv.add_poiset(poi)
        t, out = srv.submit(0, pid, tar, S, N)
        srv.wait(t)
        assert srv.stats().failed == 0 and srv.stats().hbm_peak == budget
    assert (out["flags"] == 0).all()
