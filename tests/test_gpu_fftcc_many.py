"""The DFT FFT-CC engine at 32 < N <= 60 on images that leave it with many shifts
to evaluate exactly (gratings and checkerboards, whose every period ties, ramps,
blocks), beside speckle, so that a wavefront changes between its two ways to the
peak.  The integer engine's outputs, bit for bit; at both ends of each kernel
form and both residues mod 4, where the rows' padding differs."""
import numpy as np
import pytest

from tests import cases
from tests.gpu_helpers import ctx_for, run_fftcc
from tw_amd import api

pytestmark = pytest.mark.gpu

SIZE = 260
y, x = np.mgrid[0:SIZE, 0:SIZE]
SPECKLE = api.synth_pair(SIZE, SIZE, 900, 3, api.affine(2.3, -1.6, 0.01, -0.01, 0.01, SIZE / 2, SIZE / 2))


def _image(kind):
    if kind == "stripes":
        return 100 + 100 * ((x // 2) & 1)
    if kind == "rows":
        return 255 * ((y // 4) & 1)
    if kind == "checker":
        return 60 + 90 * (((x // 4) + (y // 4)) & 1)
    if kind == "ramp":
        return (20 + 0.8 * x).astype(np.int64)
    img = SPECKLE[0].astype(np.int64)                    # speckle and a grating in stripes of windows' width
    return np.where((x // 37) & 1, 128 + 100 * np.sin(2 * np.pi * x / 10), img)


@pytest.mark.parametrize("N", [34, 40, 42, 48, 50, 54, 60])
@pytest.mark.parametrize("kind", ["stripes", "rows", "checker", "ramp", "mixed"])
def test_equals_integer_engine(kind, N, monkeypatch):
    print(f"[gpu-test] {kind} N {N}", flush=True)
    ref = np.clip(_image(kind), 0, 255).astype(np.uint8)
    tar = np.roll(ref, (3, -2), (0, 1)) if kind != "mixed" else np.where((x // 37) & 1, np.roll(ref, 1, 1), SPECKLE[1])
    case = cases.Case(kind, SIZE, 8, 8, 32, (1, 1, SIZE - 2, SIZE - 2), 2, ref, np.ascontiguousarray(tar.astype(np.uint8)), None)
    poi = np.random.default_rng(N).integers(20, SIZE - 20, (20000, 2)).astype(np.int32)
    out = []
    for variant in ("9", "8"):
        monkeypatch.setenv("TWDIC_FFTCC_VARIANT", variant)
        with ctx_for(case, N=N) as ctx:
            out.append(run_fftcc(ctx, poi))
    assert (out[0]["status"] == 0).sum() > 5000
    for f in ("u", "v", "zncc", "status"):
        assert np.array_equal(np.asarray(out[0][f]).view(np.uint8), np.asarray(out[1][f]).view(np.uint8)), f
