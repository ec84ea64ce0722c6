# SPDX-License-Identifier: Apache-2.0
"""Expert passes of many tokens at the edges of their token blocks and passes, against the oracle:
the prefill kernel with two activation terms behind the second pass list (prec 0) and on a
row-major bank, and the row-major streaming passes beside it; one expert has NaN scale bytes."""
import numpy as np
import pytest

from conftest import max_err_rel_inf
from test_gpu_dense import say

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def layer2(k3):
    E, I, N = 1024, 512, 12
    ex = [k3.gen_expert(E, I, 4242, e, 117, 122) for e in range(N)]
    for m in range(3):                       # expert 2: a NaN block in each matrix, rows 0 and last
        s = ex[2].t[2 * m + 1]
        s[0], s[-1] = 255, 255
    return E, I, N, ex


# two lists with 32-token passes / 48-token passes (prec 0), one list; 96-token passes (prec 1)
@pytest.mark.parametrize("counts", [[9, 16, 17, 32, 33, 8, 24, 1, 0, 7, 2, 3], [9, 16, 17, 32, 33, 48, 49, 96, 97, 8, 1, 0],
                                    [200, 9, 7, 0, 0, 0, 0, 0, 0, 0, 15, 31], [1, 9, 8, 2, 0, 3, 0, 1, 0, 0, 4, 1]])
@pytest.mark.parametrize("act,prec", [(0, 0), (1, 0), (1, 1)])
@pytest.mark.parametrize("layout", ["TILED", "ROWS"])
def test_many_token_passes(gpu, orc, layer2, counts, act, prec, layout):
    """One expert per token slot 0, counts[e] tokens of it (slot 1: an index outside the bank),
    so every expert's pass sizes are known."""
    E, I, N, experts = layer2
    T = sum(counts)
    say(f"case: passes {counts} act={act} prec={prec} {layout}")
    rng = np.random.default_rng(T + act)
    first = rng.permutation(np.repeat(np.arange(N), counts)).astype(np.int32)
    idx = np.stack([first, np.full(T, -1, np.int32)], 1)
    wt = rng.uniform(0.1, 1.0, (T, 2)).astype(np.float32)
    X = rng.standard_normal((T, E)).astype(np.float32)
    bank = gpu.DevBank(experts, E, I, getattr(gpu, "K3D_LAYOUT_" + layout))
    try:
        out, off, drops = gpu.moe_experts_device(bank, X, idx, wt, N, act=act, prec=prec, hidden=E, inter=I)
    finally:
        bank.free()
    assert drops == 0 and np.array_equal(np.diff(off), counts)
    tol = 1e-4 if prec == 0 else 2e-2
    for t in range(T):
        want = wt[t, 0] * orc.expert_ffn(X[t], experts[first[t]], E, I, act=act, wt=1.0)
        assert max_err_rel_inf(out[t], want) <= tol, (t, first[t])
