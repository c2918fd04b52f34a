"""Rounding of IC-GN's column walk (CPU emulation in the kernel's order).

Down a column the walk keeps a0 = sum g T and a2 -= STEP a0, and takes the x- and
y-weighted sums from them at the strips' ends (icgn.hip subset_loop), where the
sums weighted pixel by pixel add g T dx and g T dy directly.  Both are in FP64 over
exact FP32 products; each operation rounds by at most 2^-53 of its result.  With
n pixels in a lane's share, |g T| <= c and rows of half height S, the direct sums'
results are at most n c S, so they are off by at most n u n c S (u = 2^-53); the
walk's are at most n c (2 S + 1) and take two operations per pixel and four per
strip end, so the walk is off by at most (2 n + 4 k) u n c (2 S + 1) per lane.  The
test holds the walk to that bound, summed over the lanes, against exact integers,
and the update it leads to to a thousandth of the FP32 rounding of dp that follows
(2^-24 |dp|, here for |dp| = delta_p = 1e-3)."""
import numpy as np
import pytest


def strips(W, H, L, longest):
    """The strips of the fewest rounds: (column, columns, row ranges)."""
    segs = lambda c: min(L // c, H)  # noqa: E731
    rounds = {c: -(-H // segs(c)) for c in range(1, min(L, W) + 1)}
    widest = max(c for c, r in rounds.items() if r <= longest)
    cost, take = [0], [0]
    for w in range(1, W + 1):
        v, c = min((cost[w - c] + rounds[c] + 1, -c) for c in range(1, min(w, widest) + 1))
        cost.append(v)
        take.append(-c)
    out, col, w = [], 0, W
    while w:
        out.append((col, take[w], segs(take[w])))
        col, w = col + take[w], w - take[w]
    return out


def walk(g, T, S, L):
    """sum g T, sum g T dx, sum g T dy over the lanes, in the kernel's order per
    lane; the lanes' results are added exactly."""
    W = 2 * S + 1
    a0, a1, a2 = (np.zeros(L) for _ in range(3))
    plan = strips(W, W, L, W)
    for col, ncol, segs in plan:
        base, rem = divmod(W, segs)
        lane = np.arange(ncol * segs)
        seg, dx = lane // ncol, (col + lane % ncol - S).astype(np.float64)
        y0, rows = seg * base + np.minimum(seg, rem), base + (seg < rem)
        dy = (y0 - S).astype(np.float64)
        a1[lane] -= dx * a0[lane]
        a2[lane] -= dy * a0[lane]
        for r in range(int(rows.max())):
            on = lane[r < rows]
            y, x = y0[on] + r, col + on % ncol
            a0[on] += g[y, x] * T[y, x].astype(np.float64)
            a2[on] -= a0[on]
        a1[lane] += dx * a0[lane]
        a2[lane] += (dy + rows) * a0[lane]
    return [sum(int(round(v * 2.0 ** 40)) for v in a) for a in (a0, a1, a2)], len(plan)


@pytest.mark.parametrize("L", [32, 64])
@pytest.mark.parametrize("S", [10, 15, 20, 28, 60])
def test_the_walk_rounds_no_more_than_its_bound(S, L):
    rng = np.random.default_rng(S + L)
    W, u = 2 * S + 1, 2.0 ** -53
    yy, xx = np.mgrid[0:W + 2, 0:W + 2]
    img = np.clip(128 + 60 * np.sin(0.9 * xx + 0.3 * yy) + 40 * rng.standard_normal((W + 2, W + 2)), 0, 255).round()
    T = (img[1:-1, 1:-1] + rng.uniform(-1, 1, (W, W))).astype(np.float32)       # interpolated: not integers
    gx, gy = img[1:-1, 2:] - img[1:-1, :-2], img[2:, 1:-1] - img[:-2, 1:-1]
    # T in units of 2^-40: exact (|T| < 2^9, 24 bits: multiples of 2^-38 or more from 2^-15 on)
    assert np.all((T == 0) | (np.abs(T) >= 2.0 ** -16))
    Ti = [[int(v * 2.0 ** 40) for v in row] for row in T.astype(np.float64)]
    off, err = np.arange(-S, S + 1), []
    for g in (gx, gy):
        got, k = walk(g, T, S, L)
        gi = g.astype(int)
        want = [0, 0, 0]
        for y in range(W):
            for x in range(W):
                v = int(gi[y, x]) * Ti[y][x]
                want[0] += v
                want[1] += v * int(off[x])
                want[2] += v * int(off[y])
        n, c = -(-W * W // L) + W, float(np.abs(g * T).max())
        bound = L * (2 * n + 4 * k) * u * n * c * W
        err += [abs(a - b) * 2.0 ** -40 for a, b in zip(got, want)]
        assert max(err[-3:]) <= bound + L * 2.0 ** -40, (err, bound)
    # the update from these sums: H dp = sum SD T ..., SD = (gx, gx dx, gx dy, gy, ...)
    dx, dy = np.broadcast_to(off, (W, W)), np.broadcast_to(off[:, None], (W, W))
    sd = np.stack([a.ravel() for g in (gx, gy) for a in (g, g * dx, g * dy)])
    shift = np.abs(np.linalg.inv(sd @ sd.T)) @ (2.0 * np.array(err))     # SD = g / 2, so H is a quarter, sums half
    scale = np.array([1, S, S, 1, S, S])
    assert np.all(shift * scale <= 1e-3 * 2.0 ** -24 * 1e-3), shift
