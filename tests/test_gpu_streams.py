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


def test_more_callers_than_side_streams(gpu, k3):
    E, I, N, K, T = 512, 512, 4, 2, 64               # 32 tokens per expert: two pass lists
    say("case: 257 caller streams")
    L, H = gpu.lib(), hip()
    rng = np.random.default_rng(5)
    X = rng.standard_normal((T, E)).astype(np.float32)
    idx = np.stack([rng.permutation(N)[:K] for _ in range(T)]).astype(np.int32)
    wt = rng.uniform(0.1, 1.0, (T, K)).astype(np.float32)
    bank = gpu.DevBank([k3.gen_expert(E, I, 77, e, 117, 122) for e in range(N)], E, I, gpu.K3D_LAYOUT_TILED)
    wsb = L.k3d_moe_ws(T, E, I, N, K, 0)
    bufs = [gpu.DevBuf(X.nbytes).upload(X), gpu.DevBuf(idx.nbytes).upload(idx), gpu.DevBuf(wt.nbytes).upload(wt),
            gpu.DevBuf(T * E * 4), gpu.DevBuf(wsb)]
    dx, di, dw, out, ws = bufs

    def run(stream):
        out.upload(np.full((T, E), np.nan, np.float32))
        gpu.check(L.k3d_moe_experts(out.ptr, di.ptr, dw.ptr, dx.ptr, T, bank.table.ptr, bank.layout, E, I, N, K, 0, 4.0, 25.0,
                                    0, ws.ptr, wsb, None, None, None, stream), "k3d_moe_experts")
        gpu.check(L.k3d_sync(stream))
        return out.download(np.empty((T, E), np.float32)).view(np.uint32).copy()

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
        for b in bufs:
            b.free()
        bank.free()
