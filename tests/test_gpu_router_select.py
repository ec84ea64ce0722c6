# SPDX-License-Identifier: Apache-2.0
"""The router's selection (k3_select.h; router_final_kernel and, for many tokens,
router_final_wave_kernel in k3_route.hip) where it can go wrong: every group count's edge,
few and many tokens, more equal choices than candidate slots, choices in expert order,
experts that cannot be chosen, fewer than topk of them, and logits whose certification
fails. idx and weight bits equal the oracle's for every token."""
import numpy as np
import pytest

from test_gpu_router_k3 import bits, say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T", [1, 7, 200, 770])
@pytest.mark.parametrize("N,K", [(64, 8), (65, 1), (128, 24), (129, 3), (384, 8), (385, 16), (512, 8), (513, 16), (577, 20), (896, 16),
                                 (897, 64), (1024, 12), (1025, 9)])
def test_router_select_edges(gpu, orc, k3, T, N, K):
    hid = 256
    say(f"case: selection {N} experts top-{K}, {T} tokens")
    W = k3.gen_normal(N * hid, 11 + N).reshape(N, hid) * np.float32(0.1)
    X = k3.gen_normal(T * hid, 12 + T).reshape(T, hid)
    rng = np.random.default_rng(N + T)
    W[1::7] = W[0]                                       # equal logits
    W[3::5, 0], W[3::5, 1] = 1e6, -1e6                   # large prefixes: logits to recompute
    X[:, 1] = X[:, 0]
    if T > 4:
        X[1] = 0.0                                       # all logits 0: every choice equal, or the bias's order
        X[2, 5] = np.nan
    for bias in (None, np.sort(k3.gen_normal(N, 13)).astype(np.float32),
                 np.where(rng.random(N) < 0.5, -np.inf, 0.25).astype(np.float32),
                 np.where(np.arange(N) < K - 1, np.float32(-0.0), np.float32(-np.inf)).astype(np.float32)):
        idx, wt = gpu.router_device(X, W, bias, K, 1, 2.5)
        say(f"  recomputed logits: {int(gpu.router_device.recomputed.sum())}")
        for t in range(T):
            i2, w2 = orc.router(X[t], W, bias, K, 1, 2.5)
            assert np.array_equal(idx[t], i2), (t, idx[t], i2)
            assert np.array_equal(bits(wt[t]), bits(w2)), t


@pytest.mark.parametrize("T,N,K", [(256, 896, 8), (128, 896, 16), (200, 1000, 10), (600, 640, 3), (1024, 384, 2)])
def test_router_int8_partials_with_gather(gpu, orc, k3, T, N, K):
    """The routed layer at sizes whose gather runs in the final kernel's last workgroup, with the
    partials from the fp64 kernels and (1024 tokens) the int8 ones; no expert is in the bank, so the
    layer is routing and gather alone."""
    from test_gpu_moe_device import stable_gather
    hid, inter = 7168, 512
    say(f"case: routing and gather {N} experts top-{K}, {T} tokens")
    W = k3.gen_normal(N * hid, 21 + N).reshape(N, hid) * np.float32(0.02)
    X = k3.gen_normal(T * hid, 22 + T).reshape(T, hid)
    bias = k3.gen_normal(N, 23, 0.0, 0.02)
    b = gpu.DevBank([None] * N, hid, inter)
    try:
        out, idx, wt, perm, off, drops = gpu.moe_routed_device(b, X, W, bias, K, inter=inter)
    finally:
        b.free()
    assert drops == T * K and not out.any()
    p2, off2 = stable_gather(idx, N)
    assert np.array_equal(perm, p2) and np.array_equal(off, off2)
    for t in range(T):
        i2, w2 = orc.router(X[t], W, bias, K, 1, 1.0)
        assert np.array_equal(idx[t], i2) and np.array_equal(bits(wt[t]), bits(w2)), t
