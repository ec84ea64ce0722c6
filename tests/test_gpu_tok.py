# SPDX-License-Identifier: Apache-2.0
"""Products of several tokens on the matrix cores, fp32-accurate (csrc/k3_tok.hip), at the
edges of their tiles: against numpy's fp64 product of the same values. The 2-norm error of
fp32 sums of exact products is 2e-7 to 4e-7 at these widths; activations cut to two bf16
terms would show 2.6e-6, so 1e-6 tells a lost term."""
import numpy as np
import pytest

from test_gpu_dense import dev_matmul, say

pytestmark = pytest.mark.gpu


def bf16_rne(x):
    """Finite fp32 values rounded to bf16, nearest even, as fp64."""
    u = np.ascontiguousarray(x, np.float32).view(np.uint32).astype(np.uint64)
    u = ((u + 0x7FFF + ((u >> 16) & 1)) >> 16 << 16).astype(np.uint32)
    return u.view(np.float32).astype(np.float64)


@pytest.mark.parametrize("bf16", [True, False])
@pytest.mark.parametrize("T,inn,out", [(2, 8, 1), (3, 7168, 12288), (16, 24, 17), (17, 64, 16), (33, 1000, 129), (37, 7168, 3584),
                                       (64, 104, 4100), (65, 264, 300), (130, 2056, 1031), (256, 512, 4099),
                                       (700, 96, 70), (1, 7169, 300), (1, 513, 33), (2, 1001, 999), (5, 9, 17), (8, 33, 4100), (20, 1001, 999),
                                       (33, 63, 50), (64, 7167, 130), (65, 1002, 8200), (100, 1003, 40), (256, 65, 31)])
def test_tok_matmul_edges(gpu, k3, bf16, T, inn, out):
    say(f"case: {T} tokens {inn} -> {out} bf16={bf16}")
    Wb = k3.gen_bf16_normal(inn * out, 5 + T, 0.0, 0.02).reshape(out, inn)
    W = (Wb.astype(np.uint32) << 16).view(np.float32)
    if not bf16:
        W = (W * np.float32(1.0 + 2.0**-13)).astype(np.float32)
    X = k3.gen_normal(T * inn, 6 + T).reshape(T, inn) * (np.float32(10.0) ** (np.arange(T) % 7 - 3))[:, None].astype(np.float32)
    Y = dev_matmul(gpu, X, Wb if bf16 else W, bf16=bf16).astype(np.float64)
    want = X.astype(np.float64) @ W.astype(np.float64).T
    for t in range(T):
        assert np.linalg.norm(Y[t] - want[t]) <= 1e-6 * np.linalg.norm(np.abs(X[t].astype(np.float64)) @ np.abs(W.T.astype(np.float64))), t
    rel = np.linalg.norm(Y - want, axis=1) / np.linalg.norm(want, axis=1)
    if out >= 16:
        assert rel.max() <= 1e-6


# (sizes that between them take every tile shape the products are launched with, the K waves with
# several stages each)
@pytest.mark.parametrize("bf16", [True, False])
@pytest.mark.parametrize("T,inn,out", [(382, 1072, 17), (697, 1080, 38), (2, 1072, 4115), (395, 1032, 316), (677, 1064, 275),
                                       (3, 1056, 8205), (489, 1048, 369), (676, 1032, 372), (389, 1056, 619), (585, 1040, 633),
                                       (675, 1048, 1109), (686, 1072, 81), (674, 1088, 165), (629, 1048, 194), (680, 1048, 244),
                                       (618, 1048, 385), (675, 1056, 81), (682, 1056, 331), (691, 1048, 535), (617, 1032, 770),
                                       (9, 1033, 4200), (17, 1033, 4200), (33, 1033, 4200)])
def test_tok_matmul_shapes(gpu, k3, bf16, T, inn, out):
    test_tok_matmul_edges(gpu, k3, bf16, T, inn, out)


@pytest.mark.parametrize("inn,out", [(136, 40), (137, 40), (136, 2000), (137, 2000)])
@pytest.mark.parametrize("bf16", [True, False])
def test_tok_matmul_nonfinite(gpu, k3, bf16, inn, out):
    """(40 rows: on the vector units; 2000: on the matrix cores.) Infinities and NaN in x and W, the largest finite x, subnormal x: what plain products
    and sums give, element by element."""
    T = 20
    say(f"case: non-finite operands bf16={bf16} in={inn} out={out}")
    Wb = k3.gen_bf16_normal(inn * out, 91, 0.0, 1.0).reshape(out, inn)
    Wb[3, 7], Wb[4, 9], Wb[5, 100] = 0x7F80, 0xFF80, 0x7FC0          # +inf, -inf, NaN
    Wb[6, :] = 0
    W = (Wb.astype(np.uint32) << 16).view(np.float32)
    X = k3.gen_normal(T * inn, 92).reshape(T, inn)
    X[:, 7], X[:, 9] = 2.0, 0.0                                      # inf * 2 (one term only), inf * 0
    X[1, 11], X[2, 13], X[3, 15] = np.inf, -np.inf, np.nan
    X[4, 17] = np.finfo(np.float32).max
    X[5, :] = np.float32(1e-41)
    W[:, 17] = np.where(np.isfinite(W[:, 17]), np.clip(W[:, 17], -0.5, 0.5), W[:, 17])
    Wb[:, 17] = (W[:, 17].view(np.uint32) >> 16).astype(np.uint16)
    W = (Wb.astype(np.uint32) << 16).view(np.float32)
    Y = dev_matmul(gpu, X, Wb if bf16 else W, bf16=bf16)
    with np.errstate(invalid="ignore"):
        want = np.array([[np.sum(X[t].astype(np.float64) * W[o].astype(np.float64)) for o in range(out)] for t in range(T)])
    assert np.array_equal(np.isnan(Y), np.isnan(want))
    inf = np.isinf(want)
    assert np.array_equal(Y[inf], want[inf].astype(np.float32)) and not np.isinf(Y[~inf]).any()
    fin = np.isfinite(want)
    bound = np.abs(np.nan_to_num(X, posinf=0, neginf=0)).astype(np.float64) @ np.abs(np.nan_to_num(W, posinf=0, neginf=0)).astype(np.float64).T
    # the cut's last term ends at 2^-133; fp32 products of subnormals at 2^-149
    tiny = 2.0**-133 * np.abs(np.nan_to_num(W, posinf=0, neginf=0)).astype(np.float64).sum(1)[None, :] + inn * 2.0**-149
    assert (np.abs(Y - want)[fin] <= (1e-6 * bound + tiny)[fin]).all()


@pytest.mark.parametrize("bf16", [True, False])
@pytest.mark.parametrize("T,inn,out", [(40, 7168, 2048), (64, 4099, 1000)])
def test_tok_matmul_nan_tokens_cost(gpu, k3, bf16, T, inn, out):
    """Tokens of NaN (padding) leave the others' results as they are and cost little: their outputs
    need no recomputing. (One dot product after another by single lanes took over 100 times
    the clean call.)"""
    import time
    say(f"case: NaN tokens {T} tokens {inn} -> {out} bf16={bf16}")
    Wb = k3.gen_bf16_normal(inn * out, 95, 0.0, 0.02).reshape(out, inn)
    W = Wb if bf16 else (Wb.astype(np.uint32) << 16).view(np.float32)
    X = k3.gen_normal(T * inn, 96).reshape(T, inn)
    Xn = X.copy()
    Xn[[3, T - 1]] = np.nan
    L = gpu.lib()
    fn = L.k3d_matmul_bf16 if bf16 else L.k3d_matmul_f32
    bufs = [gpu.DevBuf(X.nbytes).upload(X), gpu.DevBuf(X.nbytes).upload(Xn), gpu.DevBuf(W.nbytes).upload(W), gpu.DevBuf(T * out * 4)]
    res, took = [], []
    try:
        for dx in bufs[:2]:
            best = 1e9
            for _ in range(5):
                gpu.check(L.k3d_sync(None))
                t0 = time.perf_counter()
                for _ in range(5):
                    gpu.check(fn(bufs[3].ptr, dx.ptr, T, bufs[2].ptr, inn, out, None), "matmul")
                gpu.check(L.k3d_sync(None))
                best = min(best, time.perf_counter() - t0)
            took.append(best / 5)
            res.append(bufs[3].download(np.empty((T, out), np.float32)))
    finally:
        for b in bufs:
            b.free()
    say(f"  {took[0] * 1e6:.1f} us, with two NaN tokens {took[1] * 1e6:.1f}")
    keep = [t for t in range(T) if t not in (3, T - 1)]
    assert np.isnan(res[1][[3, T - 1]]).all() and np.array_equal(res[0][keep], res[1][keep])
    assert took[1] <= 10 * took[0] + 2e-5


@pytest.mark.parametrize("T,inn,out", [(1, 1, 3), (1, 7, 5), (1, 520, 40), (1, 513, 33), (1, 1001, 999), (1, 4099, 70), (1, 7169, 300),
                                       (2, 520, 65), (5, 512, 40), (33, 1024, 129), (64, 264, 300), (2, 1001, 9), (2, 1, 3), (3, 512, 7),
                                       (4, 9, 8), (5, 7, 8), (5, 2056, 1), (7, 1030, 33), (2, 7168, 1000), (8, 7169, 530),
                                       (9, 520, 680), (9, 520, 690), (2, 1000, 4096), (2, 1000, 4097)])
def test_matmul_any_alignment(gpu, k3, T, inn, out):
    """Any row length, and x, W at any element: against fp64, and for one token bf16 weights give
    the bits of fp32 weights of the same values (the reference's invariant), at every alignment."""
    say(f"case: alignments, {T} tokens {inn} -> {out}")
    Wb = k3.gen_bf16_normal(inn * out, 15 + inn, 0.0, 0.02).reshape(out, inn)
    Wf = (Wb.astype(np.uint32) << 16).view(np.float32)
    X = k3.gen_normal(T * inn, 16 + inn).reshape(T, inn)
    want, bound = X.astype(np.float64) @ Wf.T.astype(np.float64), np.abs(X.astype(np.float64)) @ np.abs(Wf.T.astype(np.float64))
    L = gpu.lib()
    bufs = [gpu.DevBuf(a.nbytes + 64) for a in (X, Wb, Wf)] + [gpu.DevBuf(T * out * 4)]
    dx, db, df, dy = bufs
    first = None
    try:
        for ox, ow in ((0, 0), (1, 0), (0, 1), (3, 5), (2, 8)):
            dx.upload(X, 4 * ox)
            db.upload(Wb, 2 * ow)
            df.upload(Wf, 4 * ow)
            got = []
            for fn, w in ((L.k3d_matmul_bf16, db.ptr + 2 * ow), (L.k3d_matmul_f32, df.ptr + 4 * ow)):
                gpu.check(fn(dy.ptr, dx.ptr + 4 * ox, T, w, inn, out, None), "matmul")
                got.append(dy.download(np.empty((T, out), np.float32)))
                assert (np.abs(got[-1] - want) <= 1e-6 * bound).all(), (ox, ow)
            if T == 1:
                first = got[0] if first is None else first
                assert np.array_equal(got[0].view(np.uint32), got[1].view(np.uint32)), (ox, ow)
                assert np.array_equal(got[0].view(np.uint32), first.view(np.uint32)), (ox, ow)
    finally:
        for b in bufs:
            b.free()

@pytest.mark.parametrize("T,inn,rows", [(3, 128, 1), (3, 7168, 2048), (8, 256, 17), (9, 384, 48), (17, 1152, 130), (33, 3584, 4097),
                                        (64, 896, 300), (65, 512, 4100), (130, 2176, 71), (257, 128, 1031),
                                        (3, 32, 5), (19, 224, 100), (40, 1504, 515), (100, 4128, 70)])
def test_tok_mxfp4_edges(gpu, k3, T, inn, rows):
    """k3d_matmul_mxfp4 from three tokens: the activations are two bf16 terms, off by at most
    2^-17 of each (8 bits a term, rounded, and a sign), or one, rounded to nearest even; a block
    whose scale is NaN is 0."""
    say(f"case: mxfp4 {T} tokens {inn} -> {rows}")
    rng = np.random.default_rng(T)
    codes = rng.integers(0, 256, (rows, inn // 2), dtype=np.uint8)
    scales = rng.integers(118, 127, (rows, inn // 32), dtype=np.uint8)
    scales[rows // 2, inn // 64] = 255
    X = k3.gen_normal(T * inn, 7 + T).reshape(T, inn) * (np.float32(10.0) ** (np.arange(T) % 7 - 3))[:, None].astype(np.float32)
    val = np.array([0, .5, 1, 1.5, 2, 3, 4, 6, -0., -.5, -1, -1.5, -2, -3, -4, -6])
    W = np.stack([val[codes & 15], val[codes >> 4]], axis=2).reshape(rows, inn)
    W *= np.repeat(np.where(scales == 255, 0.0, 2.0 ** (scales.astype(np.float64) - 127)), 32, axis=1)
    want, bound = X.astype(np.float64) @ W.T, np.abs(X.astype(np.float64)) @ np.abs(W.T)
    L = gpu.lib()
    bufs = [gpu.DevBuf(a.nbytes).upload(np.ascontiguousarray(a)) for a in (X, codes, scales)]
    bufs += [gpu.DevBuf(max(L.k3d_matmul_mxfp4_ws(T, inn), 16)), gpu.DevBuf(T * rows * 4)]
    dx, dp, ds, ws, dy = bufs
    try:
        for prec in (0, 1):
            gpu.check(L.k3d_matmul_mxfp4(dy.ptr, dx.ptr, T, dp.ptr, ds.ptr, inn, rows, prec, ws.ptr, ws.nbytes, None), "mxfp4")
            Y = dy.download(np.empty((T, rows), np.float32))
            if prec == 0:
                assert (np.abs(Y - want) <= (2.0**-17 + 1e-6) * bound).all()
            else:                       # the products of the rounded activations, summed in fp32
                one = bf16_rne(X)
                assert (np.abs(Y - one @ W.T) <= 1e-6 * (np.abs(one) @ np.abs(W.T))).all()
    finally:
        for b in bufs:
            b.free()


@pytest.mark.parametrize("T,inn,rows", [(697, 1088, 38), (700, 1024, 129), (682, 1056, 331), (691, 1088, 65), (683, 1056, 170),
                                        (618, 1056, 385), (681, 1120, 104), (680, 1056, 244), (691, 1056, 535), (617, 1024, 770)])
def test_tok_mxfp4_shapes(gpu, k3, T, inn, rows):
    """Every tile shape the MXFP4 products are launched with."""
    test_tok_mxfp4_edges(gpu, k3, T, inn, rows)



@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("T,inn,rows", [(3, 256, 40), (40, 1504, 130), (70, 512, 515)])
def test_mxfp4_codes_off_16_bytes(gpu, k3, T, inn, rows, prec):
    """k3d_matmul_mxfp4 of three tokens and more with codes that do not start at a multiple of 16
    bytes, which the several-token kernel does not take: the expert kernel, at the same
    precision."""
    say(f"case: mxfp4 codes at +8, {T} tokens {inn} -> {rows} prec={prec}")
    rng = np.random.default_rng(T + rows)
    codes = rng.integers(0, 256, (rows, inn // 2), dtype=np.uint8)
    scales = rng.integers(118, 127, (rows, inn // 32), dtype=np.uint8)
    X = k3.gen_normal(T * inn, 8 + T).reshape(T, inn)
    val = np.array([0, .5, 1, 1.5, 2, 3, 4, 6, -0., -.5, -1, -1.5, -2, -3, -4, -6])
    W = np.stack([val[codes & 15], val[codes >> 4]], axis=2).reshape(rows, inn) * np.repeat(2.0 ** (scales.astype(np.float64) - 127), 32, axis=1)
    x = X.astype(np.float64) if prec == 0 else bf16_rne(X)
    L = gpu.lib()
    bufs = [gpu.DevBuf(X.nbytes).upload(X), gpu.DevBuf(codes.nbytes + 16).upload(codes, 8), gpu.DevBuf(scales.nbytes).upload(scales),
            gpu.DevBuf(L.k3d_matmul_mxfp4_ws(T, inn)), gpu.DevBuf(T * rows * 4)]
    dx, dp, ds, ws, dy = bufs
    try:
        gpu.check(L.k3d_matmul_mxfp4(dy.ptr, dx.ptr, T, dp.ptr + 8, ds.ptr, inn, rows, prec, ws.ptr, ws.nbytes, None), "mxfp4")
        Y = dy.download(np.empty((T, rows), np.float32))
    finally:
        for b in bufs:
            b.free()
    assert (np.abs(Y - x @ W.T) <= ((2.0**-17 if prec == 0 else 0.0) + 1e-6) * (np.abs(x) @ np.abs(W.T))).all()

@pytest.mark.parametrize("act", [0, 1])
@pytest.mark.parametrize("T,hidden,inter", [(1, 64, 64), (2, 7168, 192), (8, 128, 4096), (9, 448, 4160), (16, 7168, 2048), (17, 7168, 64),
                                            (32, 4096, 128), (33, 64, 2048), (64, 192, 2048), (65, 320, 1984), (128, 64, 1024)])
def test_shared_expert_few_tokens(gpu, k3, act, T, hidden, inter):
    """The shared expert where it takes this kernel (up to 32 tokens whole, its down product
    up to 128), next to those bounds, written and added: 1e-4 of the largest result with fp32
    or two-term activations, 2e-2 of the norm with one."""
    say(f"case: shared expert {T} tokens {hidden} -> {inter} act={act}")
    W = [k3.gen_bf16_normal(hidden * inter, 31 + i + T, 0.0, 0.03) for i in range(3)]
    F = [(w.astype(np.uint32) << 16).view(np.float32).astype(np.float64) for w in W]
    X = k3.gen_normal(T * hidden, 40 + T).reshape(T, hidden)
    g, u = X.astype(np.float64) @ F[0].reshape(inter, hidden).T, X.astype(np.float64) @ F[1].reshape(inter, hidden).T
    sg = g / (1.0 + np.exp(-g))
    a = sg * u if act == 1 else 4.0 * np.tanh(g / 4.0) / (1.0 + np.exp(-g)) * 25.0 * np.tanh(u / 25.0)
    want = a @ F[2].reshape(hidden, inter).T
    y0 = k3.gen_normal(T * hidden, 41 + T).reshape(T, hidden)
    for prec in (0, 1):
        for add in (None, y0):
            got = gpu.shared_expert_device(X, *[w.reshape(s) for w, s in zip(W, ((inter, hidden), (inter, hidden), (hidden, inter)))],
                                           hidden, inter, act=act, prec=prec, y0=add)
            ref = want if add is None else want + add
            if prec == 0:
                assert np.abs(got - ref).max() <= 1e-4 * np.abs(ref).max()
            else:
                assert np.linalg.norm(got - ref) <= 2e-2 * np.linalg.norm(ref)


@pytest.mark.parametrize("T,hidden,inter", [(1, 256, 512), (3, 4096, 256), (8, 7168, 192), (16, 512, 1024), (17, 1024, 64),
                                            (32, 4096, 128), (33, 4096, 128), (130, 512, 1024)])
def test_shared_expert_one_term(gpu, k3, T, hidden, inter):
    """prec 1 rounds the activations to one bf16 term, x and act(gate, up) alike, whatever kernel
    serves the token count. Against that computed in fp64: what is left is fp32 sums, and act
    values that these carry over a rounding boundary, a few of `inter` at 2^-8 each; products
    of unrounded activations would be off by 2e-3."""
    say(f"case: shared expert, one term, {T} tokens {hidden} -> {inter}")
    W = [k3.gen_bf16_normal(hidden * inter, 51 + i + T, 0.0, 0.03) for i in range(3)]
    F = [(w.astype(np.uint32) << 16).view(np.float32).astype(np.float64) for w in W]
    X = k3.gen_normal(T * hidden, 60 + T).reshape(T, hidden)
    xr = bf16_rne(X)
    g, u = xr @ F[0].reshape(inter, hidden).T, xr @ F[1].reshape(inter, hidden).T
    want = bf16_rne((g / (1.0 + np.exp(-g)) * u).astype(np.float32)) @ F[2].reshape(hidden, inter).T
    got = gpu.shared_expert_device(X, *[w.reshape(s) for w, s in zip(W, ((inter, hidden), (inter, hidden), (hidden, inter)))],
                                   hidden, inter, act=1, prec=1, y0=None)
    assert np.linalg.norm(got - want) <= 5e-4 * np.linalg.norm(want)
