"""Downloads from two threads through one context: a small one may find the
context's pinned buffer taken, and then goes the way of large ones.  Every byte
must arrive at its own caller.  (Nothing else of the context is used meanwhile:
a context is one thread's.)"""
import ctypes as C
import threading

import numpy as np
import pytest

from tw_amd import api

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nbytes", [40, 4096, 16384])
def test_each_thread_gets_its_own_bytes(nbytes):
    with api.Context(api.make_config(64, 64, 1, 1, 62, 62, 5, 5, 4, 4, 10, 10, 16)) as ctx:
        rng = np.random.default_rng(nbytes)
        src = [rng.integers(0, 256, nbytes).astype(np.uint8) for _ in range(2)]
        dev = [ctx.array(nbytes, np.uint8).upload(s) for s in src]
        wrong, start = [], threading.Barrier(2)

        def work(k):
            out = np.empty(nbytes, np.uint8)
            start.wait()
            for i in range(300):
                out[:] = 0
                st = api.lib().twdic_memcpy(ctx.h, C.c_void_p(out.ctypes.data), C.c_void_p(dev[k].ptr), nbytes, 1)
                if st != api.OK or not np.array_equal(out, src[k]):
                    wrong.append((k, i, st))

        threads = [threading.Thread(target=work, args=(k,)) for k in range(2)]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
        assert not wrong, wrong[:5]
