"""The error bound behind the fp16 matrix-core DFT FFT-CC engine for the even
window edges 32 < N <= 60, derived as in test_dft_bound.py for N = 64 with that
file's summation model, without the packed DC / Nyquist column (the half
spectrum k = 0 .. N / 2 fits the 32 columns) and with the table the kernel
builds (fp16 of the FP32 twiddles, the upper half of the circle mirrored).

    |C^ - C| <= bound(N) ||r|| ||t|| / N^2 at every shift,

and the kernel allows kDftBoundN N^2 / 4096 for bound(N)."""
import re
from pathlib import Path

import numpy as np
import pytest

ROOT = Path(__file__).resolve().parents[1]
SIZES = list(range(34, 61, 2))


def table(N):
    e = (np.arange(N)[:, None] * np.arange(N)[None, :]) % N
    up = 2 * e > N
    k = np.where(up, N - e, e)
    ang = -2.0 * np.pi * np.arange(N) / N
    c = np.cos(ang).astype(np.float32).astype(np.float16).astype(np.float64)
    s = np.sin(ang).astype(np.float32).astype(np.float16).astype(np.float64)
    return c[k] + 1j * np.where(up, -s[k], s[k]), np.exp(-2j * np.pi * e / N)


def bound(N, flush):
    """N^2 max |C^ - C| / (||r|| ||t||); the passes' fp32 sums have N, 2 N, 2 N
    and (32 columns, re and im, and the row that masks b >= N) 65 terms."""
    Ft, F = table(N)
    D = Ft - F
    delta, dmax = float(np.linalg.norm(D, 2)), float(np.abs(D).max())
    phi = float(max(np.linalg.norm(Ft, axis=0).max(), np.linalg.norm(Ft, axis=1).max()))
    u, v, r2, q, NN = 2.0 ** -11, 2.0 ** -24, np.sqrt(2.0), np.sqrt(N), N * N
    ga, gb, gd = (n * v / (1 - n * v) for n in (N - 1, 2 * N - 1, 64))
    tiny = 2.0 ** -14 if flush else 2.0 ** -25
    g = delta + q * phi * ga + u * (q + delta + q * phi * ga) + N * r2 * tiny
    h = q * g + delta * (q + g) + (q * r2 * phi * gb + v * (q + delta)) * (q + g)
    dP, fp32P = 2 * N * h + h * h, 6 * v * (N + h) ** 2
    sinv = NN / 2.0 ** 13                       # s N^2 ||r|| ||t|| >= 2^13, both norms >= 1
    pi0 = NN + dP + fp32P
    roundP = 2 * u * pi0 + NN * r2 * tiny * sinv
    inv = (pi0 + roundP) * (2 * dmax * (1 + dmax) + 2 * gb * (1 + dmax) ** 2
                            + u * (1 + dmax) ** 2 * (1 + 2 * gb) + gd * (1 + dmax) ** 2 * (1 + u))
    return dP + fp32P + roundP + inv + N * r2 * tiny * 256 * sinv * (1 + dmax)


def kernel_constant():
    src = (ROOT / "tw_amd" / "csrc" / "fftcc.hip").read_text()
    return float(re.search(r"constexpr double kDftBoundN = ([0-9.]+);", src).group(1))


def test_kernel_bound_covers_every_edge():
    worst = max(bound(N, True) * 4096 / N ** 2 for N in SIZES)
    assert worst <= kernel_constant() <= 1.1 * worst, worst


@pytest.mark.parametrize("N", SIZES)
def test_table_identities_and_ranges(N):
    Ft, _ = table(N)
    assert np.array_equal(Ft[(-np.arange(N)) % N, :], np.conj(Ft))
    mags = np.abs(np.concatenate([Ft.real.ravel(), Ft.imag.ravel()]))
    assert mags[mags > 0].min() / 256 > 2.0 ** -14          # times 2^-8 still normal
    assert N * 255 < 65504 and N * 2 ** 14 * np.sqrt(2) * 2 / 256 < 65504
    # |C^| in its units is at most 2^14 / 2^16 (1 + bound / N^2): the mask's -1
    # puts a masked row below every candidate, whose distance from the maximum
    # is at most 2.5 bounds
    rel = kernel_constant() / 4096
    assert -1 + 0.25 * (1 + rel) < -0.25 * (1 + rel) - 2.5 * 0.25 * rel


def _f16(x):
    return np.asarray(x, np.float32).astype(np.float16).astype(np.float32)


@pytest.mark.parametrize("N", [34, 40, 46, 54, 60])
def test_model_within_bound(N):
    """A matrix-level model of the kernel's arithmetic on stress windows."""
    Ft, _ = table(N)
    Fr, Fi, K = Ft.real.astype(np.float32), Ft.imag.astype(np.float32), N // 2 + 1
    rng = np.random.default_rng(N)
    noise, rows, alt = rng.integers(0, 256, (N, N)), rng.integers(0, 256, N), (-1) ** np.arange(N)
    one = np.full((N, N), 100)
    one[N // 3, N // 2] = 101
    for R, T in ((noise, np.roll(noise, (3, -5), (0, 1))), (np.tile(rows[:, None], (1, N)), np.tile(np.roll(rows, 2)[:, None], (1, N))),
                 (128 + (rows[:, None] // 2) * alt, 128 + (np.roll(rows, 4)[:, None] // 2) * alt), (one, np.roll(one, (2, 2), (0, 1)))):
        r, t = (x - (int(x.sum()) + N * N // 2) // (N * N) for x in (R, T))
        rho = float(np.linalg.norm(r) * np.linalg.norm(t))
        s = np.float32(2.0 ** (14 - int(np.frexp(N * N * rho)[1])))

        def forward(x):
            x = x.astype(np.float32)
            yr, yi = _f16(x @ Fr[:, :K]), _f16(x @ Fi[:, :K])
            return Fr @ yr - Fi @ yi, Fr @ yi + Fi @ yr

        (Rr, Ri), (Tr, Ti) = forward(r), forward(t)
        w = np.full(K, 2.0, np.float32)
        w[0] = w[-1] = 1.0
        Pr, Pi = _f16((Rr * Tr + Ri * Ti) * (w * s)), _f16((Rr * Ti - Ri * Tr) * (w * s))
        Qr = _f16((Pr.T @ Fr + Pi.T @ Fi) / 256)
        Qi = _f16((Pi.T @ Fr - Pr.T @ Fi) / 256)
        C = ((Fr[:, :K] @ Qr + Fi[:, :K] @ Qi).T.astype(np.float64)) * 256 / float(s) / (N * N)
        E = np.real(np.fft.ifft2(np.conj(np.fft.fft2(r)) * np.fft.fft2(t)))
        assert np.abs(C - E).max() <= bound(N, False) * rho / (N * N)
