"""What the LUT buffer holds when it is handed out (twdic_get_buffer) after IC-GN
has run from the layouts of its own: the table that a context which built the
LUT itself on every call holds at the same point.  A second context whose LUT
was handed out before its first call is that context; both run the same calls,
and every output and every table must be equal bit for bit.

A sequence's calls: A, B set a target; wA, wB write one through the target's
pointer (handed out by `tar`); frame, pre (precompute_target), cap and replay
(the context's captured frame), [ ... ] a graph the caller captures on the
context's stream and `go` launches it; lut reads the LUT."""
import ctypes as C

import numpy as np
import pytest

import oracle
from tests import cases
from tests.gpu_helpers import ctx_for
from tw_amd import api

pytestmark = pytest.mark.gpu

OUT = dict(u=np.float32, v=np.float32, zncc=np.float32, p6=np.float32, iters=np.int32, flags=np.uint8)
SIZE = 160

SEQUENCES = [
    "lut A lut frame lut",                              # nothing built yet: as it was created
    "A frame lut B frame lut",
    "A frame B lut frame lut",                          # the table of the target IC-GN last ran on
    "A frame B lut pre lut",
    "A pre B lut",
    "A pre frame B frame A lut",
    "A tar pre wB frame lut",                           # a target written through its pointer
    "A tar frame pre wB lut frame lut wA frame lut",
    "A frame tar wB lut frame lut",
    "A frame cap B lut replay lut A replay B lut",
    "A frame cap B replay A lut replay lut",
    "A tar pre cap wB replay lut wA replay lut",
    "A frame [ frame ] B go lut A go lut",              # the caller's own graph
    "A frame [ dB frame ] go lut A frame go lut",
    "A frame B [ frame ] lut go lut A go lut",
    "A frame B [ lut frame ] go lut",
    "A frame [ pre ] B lut go lut frame lut",
    "A frame B [ lut ] frame lut",
    "A frame B [ lut ] lut",
    "A frame B [ frame ] lut [ frame ] go lut",
    "A frame cap [ frame ] B replay go lut A go lut replay lut",
]


class Run:
    """One context driven through a sequence; yields what each call left."""

    def __init__(self, case, tars, interp, poi):
        self.ctx, self.case, self.tars = ctx_for(case, interp=interp), case, tars
        c, n = self.ctx, len(poi)
        self.poi = c.array(poi.shape, np.int32).upload(poi)
        self.out = {k: c.array((n, 6) if k == "p6" else n, d).fill(0) for k, d in OUT.items()}
        self.dev = {k: c.array(t.shape, np.uint8).upload(t) for k, t in tars.items()}
        self.hip = C.CDLL("libamdhip64.so")
        self.stream = C.c_void_p(api.lib().twdic_stream(c.h))
        self.graph, self.exec = C.c_void_p(), C.c_void_p()
        self.capturing = False
        self.tar = None

    def lut(self):
        _, _, w, h = self.case.roi
        ptr, nbytes = self.ctx.buffer(api.BUF_LUT)
        assert nbytes == 64 * w * h
        if self.capturing:
            return None
        a = np.empty(16 * w * h, np.float32)
        self.ctx._check(api.lib().twdic_memcpy(self.ctx.h, a.ctypes.data_as(C.c_void_p), ptr, nbytes, 1))
        return {"lut": a}

    def step(self, op):
        c = self.ctx
        if op in self.tars:
            c.set_target(self.tars[op])
        elif op[0] == "d":
            c.set_target_device(self.dev[op[1]], SIZE)
        elif op[0] == "w":
            img = self.tars[op[1]]
            c._check(api.lib().twdic_memcpy(c.h, self.tar, img.ctypes.data_as(C.c_void_p), img.nbytes, 0))
        elif op == "tar":
            self.tar = C.c_void_p(c.buffer(api.BUF_TAR)[0])
        elif op == "pre":
            c.precompute_target()
        elif op == "lut":
            return self.lut()
        elif op == "[":
            self.drop_graph()
            assert self.hip.hipStreamBeginCapture(self.stream, 1) == 0
            self.capturing = True
        elif op == "]":
            assert self.hip.hipStreamEndCapture(self.stream, C.byref(self.graph)) == 0
            self.capturing = False
            assert self.hip.hipGraphInstantiate(C.byref(self.exec), self.graph, None, None, C.c_size_t(0)) == 0
        else:
            args = (self.poi, self.poi.shape[0], *(self.out[k] for k in OUT))
            if op == "cap":
                c.frame_capture(*args)
                return None
            if op == "frame":
                c.frame(*args)
            elif op == "replay":
                c.frame_replay()
            else:
                assert op == "go" and self.hip.hipGraphLaunch(self.exec, self.stream) == 0
            if not self.capturing:
                c.sync()
                return {k: a.download() for k, a in self.out.items()}
        return None

    def drop_graph(self):
        if self.exec:                                  # every launch of it was waited for
            self.hip.hipGraphExecDestroy(self.exec)
            self.hip.hipGraphDestroy(self.graph)
            self.exec = C.c_void_p()

    def close(self):
        if self.capturing:
            self.step("]")
        self.drop_graph()
        self.ctx.close()


@pytest.mark.parametrize("interp", [api.INTERP_LUT, api.INTERP_BSPLINE])
@pytest.mark.parametrize("sequence", SEQUENCES)
def test_the_table_is_the_one_the_calls_left(sequence, interp):
    print(f"[gpu-test] mode {interp}: {sequence}", flush=True)
    ref, a = api.synth_pair(SIZE, SIZE, 400, 21, api.affine(1.3, -0.7, 0.004, -0.002, 0.001, 80, 80))
    _, b = api.synth_pair(SIZE, SIZE, 400, 21, api.affine(-0.6, 1.1, 0.001, 0.003, -0.002, 80, 80))
    case = cases.Case("handout", SIZE, 9, 12, 32, (2, 1, 153, 155), 8, ref, a, None)
    poi = np.random.default_rng(5).integers(40, 120, (90, 2)).astype(np.int32)
    runs = [Run(case, dict(A=a, B=b), interp, poi) for _ in range(2)]
    try:
        runs[1].lut()                                   # handed out before its first call
        for i, op in enumerate(sequence.split()):
            got, want = (r.step(op) for r in runs)
            assert (got is None) == (want is None)
            for k in got or ():
                assert np.array_equal(got[k].view(np.uint8), want[k].view(np.uint8)), (i, op, k)
            if op == "frame" and got:
                assert (got["flags"] == 0).mean() > 0.9
    finally:
        for r in runs:
            r.close()


@pytest.mark.parametrize("interp", [api.INTERP_LUT, api.INTERP_BSPLINE])
def test_the_table_after_a_new_target_is_the_oracle_s(interp):
    ref, a = api.synth_pair(SIZE, SIZE, 400, 22, api.affine(1.3, -0.7, 0.004, -0.002, 0.001, 80, 80))
    case = cases.Case("handout", SIZE, 9, 12, 32, (2, 1, 153, 155), 8, ref, a, None)
    r = Run(case, dict(A=a, B=np.ascontiguousarray(a[::-1])), interp, np.array([[80, 80], [70, 90]], np.int32))
    try:
        for op in "A frame B".split():
            r.step(op)
        _, _, w, h = case.roi
        table = oracle.bspline_lut if interp == api.INTERP_BSPLINE else oracle.bicubic_lut
        assert np.array_equal(r.lut()["lut"].reshape(h, w, 16), table(a, *case.roi))
    finally:
        r.close()
