"""Device-to-host copies of twdic_memcpy: the small ones (up to 16 KiB, through
the context's pinned buffer) and the first size beyond, from aligned and
unaligned addresses, to pageable and pinned memory, alone and behind a frame's
work.  Bytes must arrive as they are, and nothing beside them may change."""
import ctypes as C

import numpy as np
import pytest

from tw_amd import api

pytestmark = pytest.mark.gpu

SIZE = 256


def _download(ctx, dst, ptr, nbytes):
    return api.lib().twdic_memcpy(ctx.h, dst, C.c_void_p(ptr), nbytes, 1)


@pytest.fixture(scope="module")
def ctx():
    with api.Context(api.make_config(SIZE, SIZE, 1, 1, SIZE - 2, SIZE - 2, 10, 10, 4, 4, 20, 20, 20)) as c:
        d = api.affine(0.8, -0.4, 0.003, 0.001, -0.002, SIZE / 2, SIZE / 2)
        ref, tar = api.synth_pair(SIZE, SIZE, 900, 77, d)
        c.set_reference(ref)
        c.set_target(tar)
        yield c


@pytest.mark.parametrize("offset", [0, 1, 4, 16])
@pytest.mark.parametrize("nbytes", [1, 3, 4, 63, 64, 600, 4096, 4100, 16380, 16383, 16384, 16385])
def test_bytes_arrive_as_they_are(ctx, nbytes, offset):
    src = np.random.default_rng(nbytes + offset).integers(0, 256, 16384 + 64).astype(np.uint8)
    buf = ctx.array(src.shape, np.uint8).upload(src)
    pinned = C.c_void_p()
    assert api.lib().twdic_host_alloc(C.byref(pinned), 16384 + 64) == api.OK
    try:
        host = np.ctypeslib.as_array((C.c_uint8 * (16384 + 64)).from_address(pinned.value))
        for out in (np.full(nbytes + 32, 0xA5, np.uint8), host[:nbytes + 32]):
            out[:] = 0xA5
            assert _download(ctx, C.c_void_p(out.ctypes.data + 7), buf.ptr + offset, nbytes) == api.OK
            assert np.array_equal(out[7:7 + nbytes], src[offset:offset + nbytes])
            assert np.all(out[:7] == 0xA5) and np.all(out[7 + nbytes:] == 0xA5)
    finally:
        del host
        api.lib().twdic_host_free(pinned)


def test_a_download_follows_the_stream_s_work(ctx):
    dp, n = ctx.poi_grid(), 600
    assert ctx.nx * ctx.ny >= n
    out = dict(u=(n, np.float32), v=(n, np.float32), zncc=(n, np.float32), p6=((n, 6), np.float32),
               iters=(n, np.int32), flags=(n, np.uint8))
    o = {k: ctx.array(*s) for k, s in out.items()}
    got = []
    for _ in range(3):
        for b in o.values():
            b.fill(0)
        ctx.frame(dp, n, o["u"], o["v"], o["zncc"], o["p6"], o["iters"], o["flags"])
        got.append({k: b.download() for k, b in o.items()})       # no synchronisation in between
    ctx.sync()
    for g in got:
        assert (g["flags"] == 0).sum() > n // 2
        for k, b in o.items():
            assert np.array_equal(g[k], b.download())


def test_refused_ranges_stay_refused(ctx):
    buf = ctx.array(100, np.uint8).fill(1)
    have = api.device_span(buf.ptr)
    out = np.zeros(have + 1, np.uint8)
    assert _download(ctx, out.ctypes.data_as(C.c_void_p), buf.ptr, have + 1) != api.OK
    assert _download(ctx, out.ctypes.data_as(C.c_void_p), out.ctypes.data, 64) != api.OK
    assert not out.any()
