"""The fp16 matrix-core DFT FFT-CC engine at the window edges 32 < N <= 60: its
outputs must equal the integer matrix-core engine's bit for bit (both return
the exact integer peak, lowest index on ties) on speckle, exact ties, saturated
and random windows, near-uniform and flat windows and windows that leave the
image; edges at both ends of each kernel form, of both residues mod 4, and N =
62, which the integer engine keeps."""
import numpy as np
import pytest

from tests import cases
from tests.gpu_helpers import ctx_for, run_fftcc
from tw_amd import api

pytestmark = pytest.mark.gpu

SIZE = 200


def _pairs(rng):
    noise = rng.integers(0, 256, (SIZE, SIZE)).astype(np.uint8)
    yield noise, np.roll(noise, (2, -3), (0, 1))
    binary = ((rng.random((SIZE, SIZE)) < 0.5) * 255).astype(np.uint8)
    yield binary, rng.integers(0, 256, (SIZE, SIZE)).astype(np.uint8)
    near = np.full((SIZE, SIZE), 100, np.uint8)                 # a few single pixels: ties, flat windows
    tar = near.copy()
    for y, x in rng.integers(0, SIZE, (40, 2)):
        near[y, x] = 101
    for y, x in rng.integers(0, SIZE, (60, 2)):
        tar[y, x] = 101
    yield near, tar
    yield api.synth_pair(SIZE, SIZE, 600, int(rng.integers(1 << 30)), api.affine(2.3, -1.6, 0.01, -0.01, 0.01, 100, 100))


@pytest.mark.parametrize("N", [34, 40, 46, 48, 50, 56, 58, 60, 62])
def test_equals_integer_engine(N, monkeypatch):
    rng = np.random.default_rng(N)
    poi = rng.integers(0, SIZE, (2300, 2)).astype(np.int32)      # some windows leave the image
    poi[:4] = [[N // 2, N // 2], [SIZE - N // 2, SIZE - N // 2], [N // 2 - 1, 100], [100, SIZE - N // 2 + 1]]
    for k, (ref, tar) in enumerate(_pairs(rng)):
        print(f"[gpu-test] N {N} pair {k}", flush=True)
        case = cases.Case("edge", SIZE, 8, 8, 32, (1, 1, SIZE - 2, SIZE - 2), 2, ref, tar, None)
        out = []
        for variant in ("9", "8"):
            monkeypatch.setenv("TWDIC_FFTCC_VARIANT", variant)
            with ctx_for(case, N=N) as ctx:
                out.append(run_fftcc(ctx, poi))
        assert (out[0]["status"] == 0).any()
        for f in ("u", "v", "zncc", "status"):
            assert np.array_equal(np.asarray(out[0][f]).view(np.uint8), np.asarray(out[1][f]).view(np.uint8)), (k, f)
