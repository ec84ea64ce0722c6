# SPDX-License-Identifier: Apache-2.0
"""Caller streams past the 256 that have side streams: k3d_stream_create refuses more, and a call on
a stream made elsewhere gives its result on that stream alone, with both pass lists and after
streams have been given back."""
import ctypes as C

import numpy as np
import pytest

from test_gpu_dense import say

pytestmark = pytest.mark.gpu


def hip():
    """The HIP runtime that the library has loaded."""
    for ln in open("/proc/self/maps"):
        if "libamdhip64" in ln:
            return C.CDLL(ln.split()[-1])
    raise AssertionError("libamdhip64 is not loaded")


class TwoLists:
    """k3d_moe_experts of 64 tokens over 4 experts, two terms: 32 tokens per expert, two pass lists."""
    E, I, N, K, T = 512, 512, 4, 2, 64

    def __init__(self, gpu, k3):
        self.gpu, L = gpu, gpu.lib()
        E, I, N, K, T = self.E, self.I, self.N, self.K, self.T
        rng = np.random.default_rng(5)
        X = rng.standard_normal((T, E)).astype(np.float32)
        idx = np.stack([rng.permutation(N)[:K] for _ in range(T)]).astype(np.int32)
        wt = rng.uniform(0.1, 1.0, (T, K)).astype(np.float32)
        self.bank = gpu.DevBank([k3.gen_expert(E, I, 77, e, 117, 122) for e in range(N)], E, I, gpu.K3D_LAYOUT_TILED)
        self.wsb = L.k3d_moe_ws(T, E, I, N, K, 0)
        self.bufs = [gpu.DevBuf(X.nbytes).upload(X), gpu.DevBuf(idx.nbytes).upload(idx), gpu.DevBuf(wt.nbytes).upload(wt),
                     gpu.DevBuf(T * E * 4), gpu.DevBuf(self.wsb)]

    def clear(self):
        self.bufs[3].upload(np.full((self.T, self.E), np.nan, np.float32))

    def call(self, stream):
        dx, di, dw, out, ws = self.bufs
        gpu, b = self.gpu, self.bank
        gpu.check(gpu.lib().k3d_moe_experts(out.ptr, di.ptr, dw.ptr, dx.ptr, self.T, b.table.ptr, b.layout, self.E, self.I,
                                            self.N, self.K, 0, 4.0, 25.0, 0, ws.ptr, self.wsb, None, None, None, stream),
                  "k3d_moe_experts")

    def result(self, stream):
        self.gpu.check(self.gpu.lib().k3d_sync(stream))
        return self.bufs[3].download(np.empty((self.T, self.E), np.float32)).view(np.uint32).copy()

    def run(self, stream):
        self.clear()
        self.call(stream)
        return self.result(stream)

    def free(self):
        for b in self.bufs:
            b.free()
        self.bank.free()


def test_first_call_under_capture(gpu, k3):
    """A stream made elsewhere whose first call is one that is being captured: its side stream is
    made then, and every replay gives the eager result, with eager work between them."""
    say("case: first call on a stream made elsewhere, under capture")
    L, H = gpu.lib(), hip()
    lay, own, ex = TwoLists(gpu, k3), C.c_void_p(), C.c_void_p()
    try:
        want = lay.run(None)
        assert H.hipStreamCreateWithFlags(C.byref(own), C.c_uint(1)) == 0
        gpu.check(L.k3d_graph_begin(own), "graph_begin")
        lay.call(own)
        gpu.check(L.k3d_graph_end(own, C.byref(ex)), "graph_end")
        for _ in range(4):
            assert np.array_equal(lay.run(None), want)
            lay.clear()
            gpu.check(L.k3d_graph_launch(ex, own), "graph_launch")
            assert np.array_equal(lay.result(own), want)
        assert np.array_equal(lay.run(own), want)
        L.k3d_graph_destroy(ex)
    finally:
        if own:
            L.k3d_stream_destroy(own)
        lay.free()


def test_more_callers_than_side_streams(gpu, k3):
    say("case: 257 caller streams")
    L, H = gpu.lib(), hip()
    lay = TwoLists(gpu, k3)
    run = lay.run
    made, own = [], C.c_void_p()
    try:
        want = run(None)
        assert H.hipStreamCreateWithFlags(C.byref(own), C.c_uint(1)) == 0
        while len(made) < 300:
            s = L.k3d_stream_create()
            if not s:
                break
            made.append(s)
        say(f"  {len(made)} streams made")
        assert len(made) < 256 and b"256" in L.k3d_error()
        assert np.array_equal(run(own.value), want)
        assert np.array_equal(run(made[-1]), want)
        gpu.check(L.k3d_stream_destroy(made.pop()))
        assert np.array_equal(run(own.value), want)   # with a side stream now
        assert not L.k3d_stream_create()
    finally:
        for s in made:
            L.k3d_stream_destroy(s)
        lay.free()
