# SPDX-License-Identifier: Apache-2.0
"""k3_moe / k3_moe_prefill with every expert of the layer in the HBM bank (the experts then run
from the bank's device table before the routing is back on the host) against the same calls with
one expert missing from the bank until it is fetched, whose experts wait for the host: outputs,
routing and the bank's counters."""
import numpy as np
import pytest

from test_gpu_dense import say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T", [1, 2, 5, 70, 600])
def test_resident_bank_same_as_fetched(gpu, wl, T):
    say(f"case: resident bank T={T}")
    cfg, W, ex = wl.latent_layer(1024, 512, 512, 24, 4, n_shared=1, tag="host.resident")
    runs = {e: wl.expert_run(ex[e]) for e in ex}
    x = wl.tokens(T, 1024, tag=f"host.resident.{T}")
    keep = {}

    @gpu.GETFN
    def get(self, layer, e, out):
        t = ex[e].t
        keep[e] = t
        q = out.contents
        q.p1, q.s1, q.p3, q.s3, q.p2, q.s2 = [a.ctypes.data for a in t]
        return 0

    up = gpu.K3ExpertSrc(get, gpu.GETMANYFN(), gpu.GETFN(), None)
    import ctypes as C
    full = gpu.HbmBank(1, 24, 512, 512, 24)
    part = gpu.HbmBank(1, 24, 512, 512, 24, upstream_ptr=C.addressof(up))
    try:
        for e in range(24):
            full.put_run(0, e, runs[e])
        for e in range(23):
            part.put_run(0, e, runs[e])          # the last one comes from upstream when routed
        for a in ("gate", "down", "up", "sh1", "sh3", "sh2"):
            gpu.dev_register(W[a])
        want = gpu.moe(x, cfg, W, 1, part.src, int(T > 1))
        h0 = full.stats()
        got = gpu.moe(x, cfg, W, 1, full.src, int(T > 1))
        h1 = full.stats()
        again = gpu.moe(x, cfg, W, 1, full.src, int(T > 1))
        assert np.array_equal(got[0], want[0]) and np.array_equal(again[0], want[0])
        assert np.array_equal(got[1], want[1]) and np.array_equal(got[2], want[2], equal_nan=True)
        assert got[3] == want[3] == 0 and h1["misses"] == h0["misses"] and h1["hits"] > h0["hits"]
        # the table follows the bank: another expert's bytes under id 3, then the right ones again
        if T == 70:
            full.put_run(0, 3, runs[7])
            other = gpu.moe(x, cfg, W, 1, full.src, 1)
            assert not np.array_equal(other[0], want[0])
            full.put_run(0, 3, runs[3])
            assert np.array_equal(gpu.moe(x, cfg, W, 1, full.src, 1)[0], want[0])
    finally:
        for a in ("gate", "down", "up", "sh1", "sh3", "sh2"):
            gpu.dev_unregister(W[a])
        full.destroy()
        part.destroy()


def shared_fp64(x, W):
    """sh2 . situ(sh1 x, sh3 x) of bf16 weights in fp64 (b1 = 4, b2 = 25)."""
    f = {k: (W[k].astype(np.uint32) << 16).view(np.float32).astype(np.float64) for k in ("sh1", "sh3", "sh2")}
    g, u = x.astype(np.float64) @ f["sh1"].T, x.astype(np.float64) @ f["sh3"].T
    return (4.0 * np.tanh(g / 4.0) / (1.0 + np.exp(-g)) * 25.0 * np.tanh(u / 25.0)) @ f["sh2"].T


@pytest.mark.parametrize("resident", [False, True])
@pytest.mark.parametrize("T", [1, 2, 4])
def test_wide_trunk_few_tokens(gpu, wl, T, resident):
    """Up to four tokens keep fp32 activations in the trunk products however wide the matrix is
    (two bf16 terms would show 2.5e-6). Every fetch fails, so the block's output is its shared
    expert alone, whose gate and up have 20480 rows."""
    from oracle import PySource
    say(f"case: wide trunk T={T} resident={resident}")
    cfg, W, _ = wl.latent_layer(512, 64, 10240, 4, 1, tag="host.wide", n_generated=0)
    x = wl.tokens(T, 512, tag=f"host.wide.{T}")
    names = ("gate", "down", "up", "sh1", "sh3", "sh2") if resident else ()
    src = PySource({})                                   # (held while the library calls it)
    try:
        for a in names:
            gpu.dev_register(W[a])
        got = gpu.moe(x, cfg, W, 1, src.ptr, 1)
    finally:
        for a in names:
            gpu.dev_unregister(W[a])
    want = shared_fp64(x, W)
    assert got[3] >= 1 and np.linalg.norm(got[0] - want) <= 1e-6 * np.linalg.norm(want)


def test_overcommitted_bank_layers(gpu, orc, wl):
    """Two layers of 24 experts in 36 slots: each layer's calls evict experts of the other, so a
    layer is whole in one call and not in the next, and the device table is rewritten and left
    alone by turns. Every call against the oracle."""
    import ctypes as C
    from conftest import max_err_rel_inf
    from oracle import PySource, oracle_moe_q
    say("case: two layers in an overcommitted bank")
    cfg, W, ex = wl.latent_layer(1024, 512, 512, 24, 4, n_shared=1, tag="host.over")
    _, _, other = wl.latent_layer(1024, 512, 512, 24, 4, n_shared=1, tag="host.over2")
    layers = [ex, other]

    @gpu.GETFN
    def get(self, layer, e, out):
        q = out.contents
        q.p1, q.s1, q.p3, q.s3, q.p2, q.s2 = [a.ctypes.data for a in layers[layer][e].t]
        return 0

    up = gpu.K3ExpertSrc(get, gpu.GETMANYFN(), gpu.GETFN(), None)
    bank = gpu.HbmBank(2, 24, 512, 512, 36, upstream_ptr=C.addressof(up))
    try:
        for step, (layer, T) in enumerate([(0, 70), (0, 1), (1, 1), (0, 3), (1, 70), (1, 1), (0, 1), (0, 70), (0, 2), (1, 2)]):
            x = wl.tokens(T, 1024, tag=f"host.over.{step}")
            got = gpu.moe(x, cfg, W, 1, bank.src, int(T > 1), layer=layer)
            src = PySource(layers[layer])
            want = oracle_moe_q(orc, x, cfg, W, 1, src, int(T > 1), layer=layer)
            assert max_err_rel_inf(got[0], want[0]) <= 1e-4, step
            assert got[3] == 0 and np.array_equal(got[1], want[1]) and np.array_equal(got[2], want[2], equal_nan=True)
        assert bank.stats()["evictions"] > 0 and bank.stats()["failures"] == 0
    finally:
        bank.destroy()


@pytest.mark.parametrize("T", [1, 40, 333])
def test_resident_shared_expert(gpu, wl, T):
    """The shared expert on resident weights where its products run on the row kernel (one token),
    on the several-token kernel and on the two-term GEMMs (333 tokens fill their tiles both ways):
    every fetch fails, so the block's output is its shared expert alone, against fp64."""
    from oracle import PySource
    say(f"case: resident shared expert T={T}")
    cfg, W, _ = wl.latent_layer(3584, 64, 1792, 4, 1, tag="host.shared", n_generated=0)
    x = wl.tokens(T, 3584, tag=f"host.shared.{T}")
    src = PySource({})
    names = ("gate", "down", "up", "sh1", "sh3", "sh2")
    try:
        for a in names:
            gpu.dev_register(W[a])
        got = gpu.moe(x, cfg, W, 1, src.ptr, 1)[0]
    finally:
        for a in names:
            gpu.dev_unregister(W[a])
    want = shared_fp64(x, W)
    assert np.linalg.norm(got - want) <= (1e-5 if T == 333 else 1e-6) * np.linalg.norm(want)


@pytest.mark.parametrize("T", [1, 333])
def test_resident_block_against_oracle(gpu, orc, wl, T):
    """The whole block with its trunk resident and every expert in the HBM bank, one token and
    enough for the GEMMs and the second pass list, against the oracle token by token."""
    from conftest import max_err_rel_inf
    from oracle import PySource, oracle_moe_q
    say(f"case: resident block T={T}")
    cfg, W, ex = wl.latent_layer(3584, 512, 1536, 24, 4, n_shared=3, tag="host.block")
    x = wl.tokens(T, 3584, tag=f"host.block.{T}")
    bank = gpu.HbmBank(1, 24, 512, 1536, 24)
    names = ("gate", "down", "up", "sh1", "sh3", "sh2")
    try:
        for e in ex:
            bank.put_run(0, e, wl.expert_run(ex[e]))
        for a in names:
            gpu.dev_register(W[a])
        got = gpu.moe(x, cfg, W, 1, bank.src, int(T > 1))
    finally:
        for a in names:
            gpu.dev_unregister(W[a])
        bank.destroy()
    assert got[3] == 0
    for t in sorted({0, 1, 63, 64, 200, T - 1} & set(range(T))):
        src = PySource(ex)
        want = oracle_moe_q(orc, x[t:t + 1], cfg, W, 1, src, 0)
        assert max_err_rel_inf(got[0][t:t + 1], want[0]) <= 1e-4, t


def test_staging_rounds(gpu, orc, wl):
    """x and the output in more than one round of the 32 MiB staging, the last one ragged."""
    from conftest import max_err_rel_inf
    from oracle import PySource, oracle_moe_q
    T, E = 17003, 512
    say(f"case: staging rounds, {T * E * 4 / 2**20:.1f} MiB")
    cfg, W, ex = wl.latent_layer(E, 64, 32, 4, 2, n_shared=1, tag="host.stage")
    x = wl.tokens(T, E, tag="host.stage")
    src = PySource(ex)
    got = gpu.moe(x, cfg, W, 1, src.ptr, 1)
    assert got[3] == 0
    for t in [0, 1, 4095, 4096, 8191, 16383, 16384, 16385, 16999, T - 2, T - 1]:
        one = PySource(ex)
        want = oracle_moe_q(orc, x[t:t + 1], cfg, W, 1, one, 0)
        assert max_err_rel_inf(got[0][t:t + 1], want[0]) <= 1e-4, t
    assert not np.array_equal(got[0][16384], got[0][0])
