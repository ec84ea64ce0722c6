# SPDX-License-Identifier: Apache-2.0
"""The work that programs have this library do, as measurable cases.

Six kinds, each one call (or the calls of one layer) through the public entry points:

  layer    the routed MoE layer on device-resident data (k3d_moe_routed), with the always-on
           shared expert after it where the model has one (k3d_shared_expert)
  latent   the whole LatentMoE block through the reference-compatible host calls (k3_moe for
           one token, k3_moe_prefill for more), experts from the HBM bank, trunk registered
  dense    a trunk product y = W x, bf16 or fp32 weights (k3d_matmul_bf16 / k3d_matmul_f32)
  mxfp4    a single MXFP4 product (k3d_matmul_mxfp4)
  router   the router alone (k3d_router)
  shared   the shared expert alone (k3d_shared_expert)

Values: activations ~ N(0, 1) (a hidden state after its norm), router rows ~ N(0, 0.02),
uniform E2M1 codes with E8M0 scales 2^-10 .. 2^-5 (weights of standard deviation 0.04, so the
gate's pre-activations have one of 2.5 to 3.7), dense weights ~ N(0, 0.02), a selection bias
~ N(0, 0.01), or, for a skewed routing, 2.5 * rank^-1.2 over a random permutation.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "kimi-k3-in-c_amd"))

import k3amd  # noqa: E402

B1, B2, EPS = 4.0, 25.0, 1e-5
# hidden, inter, experts, topk, act: the 384-expert decode / prefill layer, the routed half of
# the 896-expert latent layer, and a generic small one
LAYERS = ((7168, 2048, 384, 8, "silu"), (3584, 3072, 896, 16, "situ"), (4096, 1536, 128, 8, "silu"))
# hidden, latent, inter, experts, topk, n_shared
LATENTS = ((7168, 3584, 3072, 896, 16, 2), (7168, 3584, 3072, 384, 8, 1), (4096, 2048, 1536, 128, 8, 1))


def _layer(i, **kw):
    h, n, e, k, act = LAYERS[i]
    return dict(kind="layer", hidden=h, inter=n, experts=e, topk=k, act=act, bias="none", shared=False, **kw)


def _latent(i, **kw):
    h, lat, n, e, k, s = LATENTS[i]
    return dict(kind="latent", hidden=h, latent=lat, inter=n, experts=e, topk=k, n_shared=s, **kw)


def listed():
    return [
        # one token of one stream: the smallest layer call, latency of a few launches
        dict(_layer(0, tokens=1, prec=0, layout="tiled"), name="decode_1"),
        # a decode batch of a serving loop
        dict(_layer(0, tokens=64, prec=0, layout="tiled"), name="decode_64"),
        # a ragged decode batch on a bank that keeps the reference's byte order
        dict(_layer(1, tokens=23, prec=0, layout="rows"), bias="normal", name="decode_rows_23"),
        # a long prompt in the bf16 prefill mode
        dict(_layer(0, tokens=4096, prec=1, layout="tiled"), name="prefill_4096"),
        # a shorter prompt with popular experts, and the shared expert
        dict(_layer(0, tokens=512, prec=1, layout="tiled"), bias="skew", shared=True, name="skewed_512_shared"),
        # the block of one layer, as a program relinked from the reference decodes
        dict(_latent(0, tokens=1), name="latent_decode"),
        # the same program's prompt, an odd number of tokens
        dict(_latent(0, tokens=333), name="latent_prefill_333"),
        # the widest trunk product of a decoded token
        dict(kind="dense", dtype="bf16", tokens=1, inn=7168, out=12288, name="trunk_gemv"),
        # the down-projection of a ragged decode batch
        dict(kind="dense", dtype="bf16", tokens=37, inn=7168, out=3584, name="trunk_37"),
        # one expert matrix times one token: the smallest product
        dict(kind="mxfp4", tokens=1, inn=7168, rows=2048, prec=0, name="mxfp4_gemv"),
        # routing of a prompt over the large expert count
        dict(kind="router", tokens=300, hidden=7168, experts=896, topk=16, bias="normal", name="router_300"),
        # the shared expert of a decode batch, fp32-accurate
        dict(kind="shared", tokens=64, hidden=7168, inter=2048, act="silu", prec=0, name="shared_64"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("layer",) * 5 + ("latent",) * 2 + ("dense",) * 2 + ("mxfp4",) * 2 + ("router", "shared"))
    if kind == "layer":
        i = rng.choice((0, 0, 1, 1, 2))
        t = _log(rng, 1, (4096, 2048, 4096)[i])
        prec = 1 if t > 512 else 0 if t < 128 else rng.randint(0, 1)
        c = _layer(i, tokens=t, prec=prec, layout=rng.choice(("tiled", "tiled", "tiled", "rows")))
        c["bias"] = rng.choice(("none", "normal", "skew"))
        c["shared"] = i == 0 and t <= 2048 and rng.random() < 0.25
        return c
    if kind == "latent":
        return _latent(rng.choice((0, 1, 2)), tokens=_log(rng, 1, 512))
    if kind == "dense":
        step = rng.choice((64, 64, 64, 8, 1))
        return dict(kind="dense", dtype=rng.choice(("bf16", "bf16", "bf16", "f32")), tokens=_log(rng, 1, 256),
                    inn=_log(rng, 1024, 12288) // step * step, out=_log(rng, 512, 16384))
    if kind == "mxfp4":
        t = _log(rng, 1, 512)
        return dict(kind="mxfp4", tokens=t, inn=_log(rng, 1024, 12288) // 32 * 32, rows=_log(rng, 512, 16384),
                    prec=rng.randint(0, 1) if t >= 64 else 0)
    if kind == "router":
        e, k = rng.choice(((384, 8), (896, 16), (128, 8), (rng.randint(60, 1500), rng.randint(1, 24))))
        return dict(kind="router", tokens=_log(rng, 1, 4096), hidden=rng.choice((7168, 4096, rng.randint(500, 7168))),
                    experts=e, topk=k, bias=rng.choice(("none", "normal", "skew")))
    h, n = rng.choice(((7168, 2048), (7168, 6144), (4096, 1536), (64 * rng.randint(16, 112), 64 * rng.randint(8, 64))))
    return dict(kind="shared", tokens=_log(rng, 1, 2048), hidden=h, inter=n, act=rng.choice(("silu", "situ")),
                prec=rng.randint(0, 1))


# ------------------------------------------------------------------ inputs ----
def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _normal(g, *shape, sigma=1.0, dtype=torch.float32):
    t = torch.randn(*shape, device="cuda", generator=g)
    return t.mul_(sigma).to(dtype) if sigma != 1.0 or dtype != torch.float32 else t


def _codes(g, rows, inn):
    """A random MXFP4 matrix, rows as the reference stores them: codes [rows][inn/2], scales [rows][inn/32]."""
    n = rows * inn // 2
    p = torch.randint(-2**31, 2**31, ((n + 3) // 4,), device="cuda", generator=g, dtype=torch.int32)
    s = torch.randint(117, 123, (rows * (inn // 32),), device="cuda", generator=g, dtype=torch.uint8)
    return p.view(torch.uint8)[:n].view(rows, inn // 2), s.view(rows, inn // 32)


def _bias(g, kind, experts):
    if kind == "none":
        return None
    if kind == "normal":
        return _normal(g, experts, sigma=0.01)
    rank = torch.randperm(experts, device="cuda", generator=g) + 1
    return (2.5 * rank.double() ** -1.2).float()


def _expert(g, hidden, inter):
    """gate, up, down of one expert."""
    return [_codes(g, r, i) for r, i in ((inter, hidden), (inter, hidden), (hidden, inter))]


def _layer_inputs(c, g):
    h, n = c["hidden"], c["inter"]
    d = {"x": _normal(g, c["tokens"], h), "router": _normal(g, c["experts"], h, sigma=0.02),
         "bias": _bias(g, c["bias"], c["experts"])}
    if c["shared"]:
        d["shared"] = _shared_weights(g, h, n)
    return d


def _shared_weights(g, hidden, inter):
    return [_normal(g, r, i, sigma=0.02, dtype=torch.bfloat16) for r, i in ((inter, hidden), (inter, hidden), (hidden, inter))]


def _latent_inputs(c, g):
    h, lat, si = c["hidden"], c["latent"], c["inter"] * c["n_shared"]
    bf = lambda r, i: _normal(g, r, i, sigma=0.02, dtype=torch.bfloat16)  # noqa: E731
    return {"x": _normal(g, c["tokens"], h), "gate": _normal(g, c["experts"], h, sigma=0.02),
            "bias": _normal(g, c["experts"], sigma=0.01), "latent_norm": 1.0 + _normal(g, lat, sigma=0.1),
            "down": bf(lat, h), "up": bf(h, lat), "sh1": bf(si, h), "sh3": bf(si, h), "sh2": bf(h, si)}


def _bytes(n):
    return torch.empty(max(1, int(n)), dtype=torch.uint8, device="cuda")


def _addr(t):
    return None if t is None else t.data_ptr()


def _stream():
    return torch.cuda.current_stream().cuda_stream or None


def _bank(c, g):
    """The expert bank on the device in the case's layout, and its table of device pointers."""
    L, tiled = k3amd.lib(), c["layout"] == "tiled"
    keep, table = [], []
    for _ in range(c["experts"]):
        row = []
        for p, s in _expert(g, c["hidden"], c["inter"]):
            if tiled:
                rows, inn = p.shape[0], p.shape[1] * 2
                up = -(-rows // 64) * 64        # rows come padded to 64, as k3d_mxfp4_tiled_size says
                tp, ts = _bytes(up * inn // 2), _bytes(up * inn // 32)
                k3amd.check(L.k3d_mxfp4_tile(tp.data_ptr(), ts.data_ptr(), p.data_ptr(), s.data_ptr(), rows, inn, _stream()))
                p, s = tp, ts
            keep += [p, s]
            row += [p.data_ptr(), s.data_ptr()]
        table.append(row)
    return keep, torch.tensor(table, dtype=torch.int64, device="cuda")


class _Latent:
    """Host weights registered resident and the HBM bank of one layer; given back with the state."""

    def __init__(self, c, g):
        d = {k: v.cpu() for k, v in _latent_inputs(c, g).items()}
        self.x = d.pop("x").numpy()
        self.W = {k: (v.view(torch.int16).numpy().view(np.uint16) if v.dtype == torch.bfloat16 else v.numpy())
                  for k, v in d.items()}
        self.cfg = dict(hidden=c["hidden"], latent=c["latent"], inter=c["inter"], n_experts=c["experts"], topk=c["topk"],
                        n_shared=c["n_shared"], renorm=1, latent_norm=1, routed_scale=1.0, rms_eps=EPS, b1=B1, b2=B2)
        self.prefill = 0 if c["tokens"] == 1 else 1
        self.bank, self.registered = None, []
        self.bank = k3amd.HbmBank(1, c["experts"], c["latent"], c["inter"], c["experts"])
        run = torch.empty(k3amd.lib().k3_devbank_run_bytes(c["latent"], c["inter"]), dtype=torch.uint8, pin_memory=True)
        for e in range(c["experts"]):
            (p1, s1), (p3, s3), (p2, s2) = _expert(g, c["latent"], c["inter"])
            run.copy_(torch.cat([t.reshape(-1) for t in (p1, s1, p2, s2, p3, s3)]))
            self.bank.put_run(0, e, run.numpy())
        for a in self.W.values():
            k3amd.dev_register(a)
            self.registered.append(a)

    def __del__(self):
        for a in getattr(self, "registered", ()):
            k3amd.dev_unregister(a)
        if getattr(self, "bank", None) is not None:
            self.bank.destroy()


def prepare(case, seed):
    c, g = case, _gen(seed)
    L = k3amd.lib()
    k3amd.check(L.k3d_init(), "k3d_init")
    kind, T = c["kind"], c.get("tokens")
    s = dict(c)
    f32 = dict(dtype=torch.float32, device="cuda")
    if kind == "layer":
        s.update(_layer_inputs(c, g))
        s["keep"], s["table"] = _bank(c, g)
        s["out"] = torch.empty(T, c["hidden"], **f32)
        s["ws"] = _bytes(L.k3d_moe_ws(T, c["hidden"], c["inter"], c["experts"], c["topk"], c["prec"]))
        if c["shared"]:
            s["shared_ws"] = _bytes(L.k3d_shared_ws(T, c["hidden"], c["inter"], c["prec"]))
    elif kind == "latent":
        s["layer"] = _Latent(c, g)
    elif kind == "dense":
        s["x"] = _normal(g, T, c["inn"])
        s["w"] = _normal(g, c["out"], c["inn"], sigma=0.02, dtype=torch.bfloat16 if c["dtype"] == "bf16" else torch.float32)
        s["y"] = torch.empty(T, c["out"], **f32)
    elif kind == "mxfp4":
        s["x"] = _normal(g, T, c["inn"])
        s["p"], s["s"] = _codes(g, c["rows"], c["inn"])
        s["y"] = torch.empty(T, c["rows"], **f32)
        s["ws"] = _bytes(L.k3d_matmul_mxfp4_ws(T, c["inn"]))
    elif kind == "router":
        s["x"] = _normal(g, T, c["hidden"])
        s["router"] = _normal(g, c["experts"], c["hidden"], sigma=0.02)
        s["bias"] = _bias(g, c["bias"], c["experts"])
        s["ws"] = _bytes(L.k3d_router_ws(T, c["hidden"], c["experts"]))
    else:
        s["x"] = _normal(g, T, c["hidden"])
        s["shared"] = _shared_weights(g, c["hidden"], c["inter"])
        s["out"] = torch.empty(T, c["hidden"], **f32)
        s["shared_ws"] = _bytes(L.k3d_shared_ws(T, c["hidden"], c["inter"], c["prec"]))
    if kind in ("layer", "router"):
        s["idx"] = torch.empty(T, c["topk"], dtype=torch.int32, device="cuda")
        s["wt"] = torch.empty(T, c["topk"], **f32)
    return s


ACT = {"situ": k3amd.K3_ACT_SITU, "silu": k3amd.K3_ACT_SILU}
LAYOUT = {"rows": k3amd.K3D_LAYOUT_ROWS, "tiled": k3amd.K3D_LAYOUT_TILED}


def _run_shared(s, accumulate):
    w1, w3, w2 = s["shared"]
    k3amd.check(k3amd.lib().k3d_shared_expert(
        s["out"].data_ptr(), accumulate, s["x"].data_ptr(), s["tokens"], w1.data_ptr(), w3.data_ptr(), w2.data_ptr(),
        s["hidden"], s["inter"], ACT[s["act"]], B1, B2, s["prec"], s["shared_ws"].data_ptr(), s["shared_ws"].numel(),
        _stream()), "k3d_shared_expert")


def run(state):
    s, L = state, k3amd.lib()
    kind = s["kind"]
    if kind == "layer":
        k3amd.check(L.k3d_moe_routed(
            s["out"].data_ptr(), s["idx"].data_ptr(), s["wt"].data_ptr(), s["x"].data_ptr(), s["tokens"],
            s["router"].data_ptr(), _addr(s["bias"]), s["table"].data_ptr(), LAYOUT[s["layout"]], s["hidden"],
            s["inter"], s["experts"], s["topk"], 1, 1.0, ACT[s["act"]], B1, B2, s["prec"], s["ws"].data_ptr(),
            s["ws"].numel(), None, None, None, _stream()), "k3d_moe_routed")
        if s["shared"]:
            _run_shared(s, 1)
        return {"out": s["out"], "idx": s["idx"], "wt": s["wt"]}
    if kind == "latent":
        y = s["layer"]
        out, idx, wt, drops = k3amd.moe(y.x, y.cfg, y.W, k3amd.K3_WBF16, y.bank.src, y.prefill)
        return {"out": out, "drops": drops} if y.prefill else {"out": out, "drops": drops, "idx": idx, "wt": wt}
    if kind == "dense":
        f = L.k3d_matmul_bf16 if s["dtype"] == "bf16" else L.k3d_matmul_f32
        k3amd.check(f(s["y"].data_ptr(), s["x"].data_ptr(), s["tokens"], s["w"].data_ptr(), s["inn"], s["out"],
                      _stream()), "k3d_matmul")
        return s["y"]
    if kind == "mxfp4":
        k3amd.check(L.k3d_matmul_mxfp4(
            s["y"].data_ptr(), s["x"].data_ptr(), s["tokens"], s["p"].data_ptr(), s["s"].data_ptr(), s["inn"], s["rows"],
            s["prec"], s["ws"].data_ptr(), s["ws"].numel(), _stream()), "k3d_matmul_mxfp4")
        return s["y"]
    if kind == "router":
        k3amd.check(L.k3d_router(
            s["idx"].data_ptr(), s["wt"].data_ptr(), s["x"].data_ptr(), s["tokens"], s["router"].data_ptr(),
            _addr(s["bias"]), s["hidden"], s["experts"], s["topk"], 1, 1.0, s["ws"].data_ptr(), s["ws"].numel(),
            _stream()), "k3d_router")
        return {"idx": s["idx"], "wt": s["wt"]}
    _run_shared(s, 0)
    return s["out"]


# ------------------------------------------------------ the same in 64 bits ----
def _dequant(p, s):
    mag = torch.tensor([0, .5, 1, 1.5, 2, 3, 4, 6, -0., -.5, -1, -1.5, -2, -3, -4, -6], dtype=torch.float64, device="cuda")
    w = torch.stack([mag[(p & 15).int()], mag[(p >> 4).int()]], -1).view(p.shape[0], -1, 32)
    return (w * torch.exp2(s.double() - 127.0).unsqueeze(-1)).view(p.shape[0], -1)


def _glu(g, u, act):
    if act == "silu":
        return g * torch.sigmoid(g) * u
    return B1 * torch.tanh(g / B1) * torch.sigmoid(g) * (B2 * torch.tanh(u / B2))


def _route(x, W, bias, topk):
    """Selection on the fp32 scores (plus the bias), as the router's definition has it; weights in 64 bits."""
    logit = x.double() @ W.double().T
    score = torch.sigmoid(logit.float().double())
    pick = score.float() if bias is None else score.float() + bias
    idx = torch.sort(pick, dim=1, descending=True, stable=True).indices[:, :topk]
    wt = torch.gather(score, 1, idx)
    return idx.to(torch.int32), wt / wt.sum(1, keepdim=True) if topk > 1 else wt


def _routed(z, idx, wt, experts, g, width, inter, act):
    out = torch.zeros(z.shape[0], width, dtype=torch.float64, device="cuda")
    z = z.double()
    for e in range(experts):
        (p1, s1), (p3, s3), (p2, s2) = _expert(g, width, inter)
        t, j = torch.nonzero(idx == e, as_tuple=True)
        if t.numel():
            a = _glu(z[t] @ _dequant(p1, s1).T, z[t] @ _dequant(p3, s3).T, act)
            out.index_add_(0, t, (a @ _dequant(p2, s2).T) * wt[t, j].unsqueeze(1))
    return out


def _dense_ffn(x, w1, w3, w2, act):
    x = x.double()
    return _glu(x @ w1.double().T, x @ w3.double().T, act) @ w2.double().T


def exact(case, seed):
    c, g = case, _gen(seed)
    kind, T = c["kind"], c.get("tokens")
    if kind == "layer":
        d = _layer_inputs(c, g)
        idx, wt = _route(d["x"], d["router"], d["bias"], c["topk"])
        out = _routed(d["x"], idx, wt, c["experts"], g, c["hidden"], c["inter"], c["act"])
        if c["shared"]:
            out += _dense_ffn(d["x"], *d["shared"], c["act"])
        return {"out": out, "idx": idx, "wt": wt}
    if kind == "latent":
        d = _latent_inputs(c, g)
        x = d["x"].double()
        idx, wt = _route(d["x"], d["gate"], d["bias"], c["topk"])
        acc = _routed(x @ d["down"].double().T, idx, wt, c["experts"], g, c["latent"], c["inter"], "situ")
        acc = d["latent_norm"].double() * acc / torch.sqrt((acc * acc).mean(1, keepdim=True) + EPS)
        out = (acc @ d["up"].double().T + _dense_ffn(x, d["sh1"], d["sh3"], d["sh2"], "situ")).cpu().numpy()
        if T > 1:
            return {"out": out, "drops": 0}
        return {"out": out, "drops": 0, "idx": idx[0].cpu().numpy(), "wt": wt[0].cpu().numpy()}
    if kind == "dense":
        x = _normal(g, T, c["inn"])
        w = _normal(g, c["out"], c["inn"], sigma=0.02, dtype=torch.bfloat16 if c["dtype"] == "bf16" else torch.float32)
        return x.double() @ w.double().T
    if kind == "mxfp4":
        x = _normal(g, T, c["inn"])
        return x.double() @ _dequant(*_codes(g, c["rows"], c["inn"])).T
    if kind == "router":
        x, w = _normal(g, T, c["hidden"]), _normal(g, c["experts"], c["hidden"], sigma=0.02)
        idx, wt = _route(x, w, _bias(g, c["bias"], c["experts"]), c["topk"])
        return {"idx": idx, "wt": wt}
    x = _normal(g, T, c["hidden"])
    return _dense_ffn(x, *_shared_weights(g, c["hidden"], c["inter"]), c["act"])


# ------------------------------------------------------------ what it takes ----
def _used(experts, topk, tokens):
    return experts * (1.0 - (1.0 - topk / experts) ** tokens)


def work(case):
    c = case
    kind, T = c["kind"], c["tokens"]
    if kind == "dense":
        size = 2 if c["dtype"] == "bf16" else 4
        return {"bytes": c["inn"] * c["out"] * size + 4 * T * (c["inn"] + c["out"]), "flops": 2 * T * c["inn"] * c["out"]}
    if kind == "mxfp4":
        return {"bytes": c["inn"] * c["rows"] * 17 // 32 + 4 * T * (c["inn"] + c["rows"]), "flops": 2 * T * c["inn"] * c["rows"]}
    h = c["hidden"]
    if kind == "shared":
        return {"bytes": 6 * h * c["inter"] + 8 * T * h, "flops": 6 * T * h * c["inter"]}
    e, k = c["experts"], c["topk"]
    b, f = 4 * e * h + 4 * T * h + 8 * T * k, 2 * T * e * h
    if kind == "router":
        return {"bytes": b, "flops": f}
    w, n = c.get("latent", h), c["inter"]
    b += _used(e, k, T) * 3 * w * n * 17 // 32 + 4 * T * h
    f += 6 * T * k * w * n
    n_shared = c["n_shared"] if kind == "latent" else int(c["shared"])
    b += 6 * h * n * n_shared
    f += 6 * T * h * n * n_shared
    if kind == "latent":
        b += 4 * h * w
        f += 4 * T * h * w
    return {"bytes": b, "flops": f}


def tolerance(case):
    """About four times the error against 64 bits that the path shows at these sizes."""
    kind = case["kind"]
    if kind == "router":
        return "exact"                      # the reference's routing, bit for bit
    if kind == "dense":
        return {"rel": 1e-6}                # fp32 products and sums: 2e-7 measured
    if kind == "mxfp4" and case["prec"] == 0:
        return {"rel": 1e-5}                # activations as two bf16 terms, one product: 2.6e-6
    if kind != "latent" and case["prec"] == 1:
        return {"rel": 1.2e-2}              # activations rounded to bf16: 2.9e-3
    return {"rel": 2e-5}                    # two bf16 terms through a chain of products: 4.9e-6
