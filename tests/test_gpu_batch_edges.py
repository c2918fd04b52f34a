"""A batch whose pairs have many FFT-CC window edges: edges that share an integer
kernel's launch, an edge that has one to itself, and edges with enough POIs for
a launch of the DFT engine beside the others.  Every pair's outputs must be the
single context's, bit for bit."""
import numpy as np
import pytest

from tw_amd import api

pytestmark = pytest.mark.gpu

SIZE = 260
OUT = dict(u=np.float32, v=np.float32, zncc=np.float32, p6=np.float32, iters=np.int32, flags=np.uint8)


@pytest.mark.parametrize("edges", [
    [(8, 60), (20, 40), (32, 70), (30, 1)],               # one kernel, four edges
    [(40, 1300), (64, 30)],                               # alone with its kernel: the DFT engine's rule
    [(40, 1300), (34, 50), (48, 3300)],                   # two share it, one leaves it
    [(62, 40), (50, 1199), (60, 1200), (56, 0)],          # at the line; an empty pair
    [(2 * k, 25) for k in range(4, 33)],                  # every edge
])
def test_pairs_equal_single_contexts(edges):
    print(f"[gpu-test] batch edges {edges}", flush=True)
    rng = np.random.default_rng(len(edges))
    ref, tar = api.synth_pair(SIZE, SIZE, 1000, 4, api.affine(1.4, -0.9, 0.003, -0.002, 0.001, SIZE / 2, SIZE / 2))
    cfg = lambda N: api.make_config(SIZE, SIZE, 1, 1, SIZE - 2, SIZE - 2, 10, 10, 8, 8, 30, 30, N)  # noqa: E731
    pois = [rng.integers(45, SIZE - 45, (n, 2)).astype(np.int32) for _, n in edges]
    with api.Context(cfg(32)) as mem, api.Batch() as b:
        dr, dt = (mem.array(x.shape, np.uint8).upload(x) for x in (ref, tar))
        outs, pairs = [], []
        for (N, n), poi in zip(edges, pois):
            dp = mem.array((max(n, 1), 2), np.int32).upload(poi if n else np.zeros((1, 2), np.int32))
            o = {k: mem.array((max(n, 1), 6) if k == "p6" else max(n, 1), d).fill(0) for k, d in OUT.items()}
            outs.append(o)
            pairs.append(api.Pair(dr.ptr, dt.ptr, SIZE, SIZE, SIZE, 1, 1, SIZE - 2, SIZE - 2, 10, 10, N, 20, 0.001,
                                  dp.ptr, n, *(o[k].ptr for k in OUT)))
        mem.sync()
        b.set_pairs(pairs)
        b.run()
        b.sync()
        for (N, n), poi, o in zip(edges, pois, outs):
            if not n:
                continue
            with api.Context(cfg(N)) as c:
                c.set_reference(ref)
                c.set_target(tar)
                dp = c.array(poi.shape, np.int32).upload(poi)
                w = {k: c.array((n, 6) if k == "p6" else n, d).fill(0) for k, d in OUT.items()}
                c.frame(dp, n, *(w[k] for k in OUT))
                c.sync()
                for k in OUT:
                    assert np.array_equal(o[k].download().view(np.uint8), w[k].download().view(np.uint8)), (N, n, k)
