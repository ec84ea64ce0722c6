# SPDX-License-Identifier: Apache-2.0
"""Expert passes of more than eight tokens with two activation terms (the prefill kernel's
NS 2 form behind the second pass list): against the oracle at the edges of its token blocks
and passes."""
import numpy as np
import pytest

from conftest import max_err_rel_inf
from test_gpu_dense import say

pytestmark = pytest.mark.gpu
TOL = 1e-4


@pytest.fixture(scope="module")
def layer2(k3):
    E, I, N = 1024, 512, 12
    return E, I, N, [k3.gen_expert(E, I, 4242, e, 117, 122) for e in range(N)]


@pytest.mark.parametrize("counts", [[9, 16, 17, 32, 33, 48, 49, 96, 97, 8, 1, 0], [200, 9, 7, 0, 0, 0, 0, 0, 0, 0, 15, 31]])
@pytest.mark.parametrize("act", [0, 1])
def test_two_term_passes(gpu, orc, layer2, counts, act):
    """One expert per token slot 0, counts[e] tokens of it (slot 1: an index outside the bank),
    so every expert's pass sizes are known."""
    E, I, N, experts = layer2
    T = sum(counts)
    say(f"case: two-term passes {counts} act={act}")
    rng = np.random.default_rng(T + act)
    first = rng.permutation(np.repeat(np.arange(N), counts)).astype(np.int32)
    idx = np.stack([first, np.full(T, -1, np.int32)], 1)
    wt = rng.uniform(0.1, 1.0, (T, 2)).astype(np.float32)
    X = rng.standard_normal((T, E)).astype(np.float32)
    bank = gpu.DevBank(experts, E, I, gpu.K3D_LAYOUT_TILED)
    try:
        out, off, drops = gpu.moe_experts_device(bank, X, idx, wt, N, act=act, prec=0, hidden=E, inter=I)
    finally:
        bank.free()
    assert drops == 0 and np.array_equal(np.diff(off), counts)
    for t in range(T):
        want = wt[t, 0] * orc.expert_ffn(X[t], experts[first[t]], E, I, act=act, wt=1.0)
        assert max_err_rel_inf(out[t], want) <= TOL, (t, first[t])
