"""What this engine is asked to do in use, as cases that can be timed and compared.

One case is one call (or one whole encode) through the public entry points of
``aikit_amd.enchip`` / ``aikit_amd.bert_dev`` on one GPU:

  linear       enchip_w8a8_linear_dev: a W8A8 linear on device buffers
  linear_host  enchip_w8a8_linear: the same linear as the Go seam calls it, host slices
  attention    enchip_attention_f32_dev on the fused [tokens, 3D] QKV rows
  q8w          enchip_matmul_bt_q8_dev: int8 weights, f32 activations (LoadQ8 encoders)
  f32          enchip_matmul_bt_f32_dev: the f32 MatmulBT, one product or a batch
  encode       a whole BERT forward from token ids (DeviceBert): hidden states and pooled
               embeddings
  ann          enchip_ann_topk: top-k of an int8 index for a batch of queries, host to host

A program has one context and keeps its weights registered; so does this file. Calls run on
the context's own stream. Inputs come from the seed alone.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from aikit_amd import enchip
from aikit_amd.bert_dev import LN_EPS, DeviceBert

ACTS = {"none": enchip.ACT_NONE, "gelu": enchip.ACT_GELU}
VOCAB = {"bert": 30522, "xlmr": 250002}

_ctx = None


def context() -> enchip.Context:
    """The process's one context."""
    global _ctx
    if _ctx is None:
        _ctx = enchip.Context(0)
    return _ctx


# ---------------------------------------------------------------------------- the cases


def listed():
    return [
        # a short query, or a handful of them padded together: 16 tokens through one FFN-up.
        # Latency and launches.
        dict(name="linear_m16", kind="linear", M=16, K=768, N=3072, act="none"),
        # one full-length BERT-base sequence through FFN-up with its GELU, what a service
        # that encodes a sequence per request runs
        dict(name="linear_m512_gelu", kind="linear", M=512, K=768, N=3072, act="gelu"),
        # a ragged batch into an odd output width (a token-classification head): nothing is
        # a multiple of a tile, and N is not a multiple of 4
        dict(name="linear_m1500_odd", kind="linear", M=1500, K=1000, N=1001, act="none"),
        # a full batch (64 x 512 tokens) through BERT-base's FFN-down
        dict(name="linear_m32768", kind="linear", M=32768, K=3072, N=768, act="none"),
        # the seam as the Go encoder uses it: host slices in, host slices out, one sequence
        dict(name="linear_host_m512", kind="linear_host", M=512, K=768, N=3072, act="gelu"),
        # short ragged texts (queries, titles) through a MiniLM-width attention
        dict(name="attention_short", kind="attention", S=32, L=77, heads=12, hd=32),
        # two long documents, past the two-pass kernels' 512 tokens
        dict(name="attention_long", kind="attention", S=2, L=2000, heads=16, hd=64),
        # a weight-only int8 encoder's fused QKV on one 512-token sequence
        dict(name="q8w_m512", kind="q8w", M=512, K=768, N=2304),
        # an f32 encoder's FFN-up on one 512-token sequence
        dict(name="f32_m512", kind="f32", M=512, K=768, N=3072, batch=1, layout="nk"),
        # a small embedding model on a small batch: many short launches
        dict(name="encode_minilm_b8s128", kind="encode", family="bert", layers=6, hidden=384, heads=12, ffn=1536,
             S=8, L=128),
        # bulk embedding: the benchmark's workload
        dict(name="encode_bert_b64s512", kind="encode", family="bert", layers=12, hidden=768, heads=12, ffn=3072,
             S=64, L=512),
        # retrieval: a batch of queries against a million-row index
        dict(name="ann_q256_k10", kind="ann", rows=1 << 20, dim=384, M=256, k=10),
    ]


def _log(rng, lo, hi):
    """A whole number between lo and hi, spread over its logarithm."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _width(rng, lo, hi):
    """A layer width: one a model has, or any multiple of 4, or (rarely) an odd one."""
    t = rng.random()
    if t < 0.5:
        return rng.choice([w for w in (384, 768, 1024, 1536, 2304, 3072, 4096) if lo <= w <= hi])
    w = _log(rng, lo, hi)
    return w if t > 0.85 else max(4, w // 4 * 4)


def draw(rng):
    kind = rng.choice(["linear", "linear", "linear_host", "attention", "q8w", "f32", "encode", "ann"])
    if kind in ("linear", "linear_host"):
        return dict(kind=kind, M=_log(rng, 1, 32768 if kind == "linear" else 2048), K=_width(rng, 256, 4096),
                    N=_width(rng, 256, 4096), act=rng.choice(["none", "gelu"]))
    if kind == "q8w":
        return dict(kind=kind, M=_log(rng, 1, 8192), K=_width(rng, 256, 4096), N=_width(rng, 256, 4096))
    if kind == "f32":
        if rng.random() < 0.5:
            return dict(kind=kind, M=_log(rng, 1, 4096), K=_width(rng, 256, 3072), N=_width(rng, 256, 3072), batch=1,
                        layout="nk")
        # attention products of every head of some sequences: Q . K^T, or scores . V
        L, hd = _log(rng, 16, 512), rng.choice([32, 64])
        layout = rng.choice(["nk", "kn"])
        return dict(kind=kind, M=L, K=hd if layout == "nk" else L, N=L if layout == "nk" else hd,
                    batch=12 * _log(rng, 1, 32), layout=layout)
    if kind == "attention":
        L = _log(rng, 16, 2048)
        return dict(kind=kind, S=_log(rng, 1, max(1, min(64, 32768 // L))), L=L, heads=rng.choice([12, 16]),
                    hd=rng.choice([32, 64]))
    if kind == "ann":
        dim = rng.choice([128, 256, 384, 512, 768])
        return dict(kind=kind, rows=_log(rng, 1 << 15, (1 << 20) * 384 // max(384, dim)), dim=dim, M=_log(rng, 1, 256),
                    k=_log(rng, 1, 100))
    family, hidden, heads, ffn, layers = rng.choice(
        [("bert", 384, 12, 1536, 6), ("bert", 768, 12, 3072, 12), ("xlmr", 1024, 16, 4096, 6)])
    L = _log(rng, 16, 512)
    return dict(kind=kind, family=family, layers=layers, hidden=hidden, heads=heads, ffn=ffn,
                S=_log(rng, 1, min(64, 16384 // L)), L=L)


# ---------------------------------------------------------------------------- inputs


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed) * 7919 + 17)


def _randn(g, *shape, std=1.0):
    x = torch.randn(shape, device="cuda", generator=g)
    return x if std == 1.0 else x * std


def _activations(g, M, K):
    """N(0, 1) with 1% of the elements 20 times larger: an encoder's outlier channels."""
    a = _randn(g, M, K)
    return torch.where(torch.rand((M, K), device="cuda", generator=g) < 0.01, a * 20.0, a)


def _rows_i8(x):
    """Symmetric int8 rows: codes and f32 scales (QuantizeRowsInt8)."""
    m = x.abs().amax(dim=1)
    s = torch.where(m == 0, torch.ones_like(m), m / 127.0)
    v = x * (1.0 / s)[:, None]
    q = torch.trunc(v.double() + torch.copysign(torch.full_like(v, 0.5), v).double()).clamp(-127, 127).to(torch.int8)
    return q, s


def _weight(g, N, K, std=0.02):
    """A trained linear's int8 weight: codes of normal rows, per-channel scales, and a bias."""
    q, s = _rows_i8(_randn(g, N, K, std=std))
    return q, s, _randn(g, N, std=std)


def _encoder(case, g):
    D, I, V = case["hidden"], case["ffn"], VOCAB[case["family"]]
    xlmr = case["family"] == "xlmr"
    off = 2 if xlmr else 0  # XLM-R's positions start at pad_token_id + 1, and it has no token types
    npos = max(case["L"], 512) + off
    e = dict(word=_randn(g, V, D, std=0.02), pos=_randn(g, npos, D, std=0.02), off=off,
             typ=None if xlmr else _randn(g, 2, D, std=0.02),
             ln=(1 + _randn(g, D, std=0.02), _randn(g, D, std=0.02)))
    layers = []
    for _ in range(case["layers"]):
        lw = {n: _weight(g, N, K) for n, K, N in (("qkv", D, 3 * D), ("o", D, D), ("ffn_up", D, I), ("ffn_down", I, D))}
        for n in ("attn_ln", "out_ln"):
            lw[n] = (1 + _randn(g, D, std=0.02), _randn(g, D, std=0.02))
        layers.append(lw)
    ids = torch.randint(0, V, (case["S"] * case["L"],), device="cuda", dtype=torch.int32, generator=g)
    return e, layers, ids


def _inputs(case, seed):
    """The case's inputs as GPU tensors, from the seed alone."""
    g, kind = _gen(seed), case["kind"]
    if kind in ("linear", "linear_host"):
        return (_activations(g, case["M"], case["K"]), *_weight(g, case["N"], case["K"]))
    if kind == "q8w":
        return (_activations(g, case["M"], case["K"]), *_weight(g, case["N"], case["K"])[:2])
    if kind == "f32":
        B, M, K, N = case["batch"], case["M"], case["K"], case["N"]
        a = _randn(g, B, M, K)
        if case["layout"] == "kn":  # attention weights: rows that sum to one
            a = torch.softmax(a, dim=-1)
        return a, _randn(g, B, *((N, K) if case["layout"] == "nk" else (K, N)))
    if kind == "attention":
        return (_randn(g, case["S"] * case["L"], 3 * case["heads"] * case["hd"]),)
    if kind == "ann":
        x = torch.nn.functional.normalize(_randn(g, case["rows"], case["dim"]))
        return (torch.nn.functional.normalize(_randn(g, case["M"], case["dim"])), *_rows_i8(x))
    return _encoder(case, g)


class _Registered:
    """A registered weight, released with the state that holds it."""

    def __init__(self, q, s):
        self.w = context().register_weight(q.cpu().numpy(), s.cpu().numpy())

    def __del__(self):
        try:
            context().release_weight(self.w)
        except Exception:
            pass


class _Model:
    def __init__(self, case, e, layers):
        acts = {"qkv": "none", "o": "none", "ffn_up": "gelu", "ffn_down": "none"}
        host = [{n: tuple(t.cpu().numpy() for t in lw[n]) + ((ACTS[acts[n]],) if n in acts else ()) for n in lw}
                for lw in layers]
        self.model = DeviceBert(context(), host, case["hidden"], case["heads"], case["ffn"])
        self.model.set_embeddings(e["word"], e["pos"], e["ln"], typ=e["typ"], pos_off=e["off"])

    def __del__(self):
        try:
            self.model.close()
        except Exception:
            pass


def prepare(case, seed):
    kind, x = case["kind"], _inputs(case, seed)
    empty = lambda *shape: torch.empty(shape, device="cuda")  # noqa: E731
    st = dict(case=case)
    if kind == "linear":
        st.update(a=x[0], w=_Registered(x[1], x[2]), b=x[3], out=empty(case["M"], case["N"]))
    elif kind == "linear_host":
        st.update(a=x[0].cpu().numpy(), w=_Registered(x[1], x[2]), b=x[3].cpu().numpy())
    elif kind == "q8w":
        st.update(a=x[0], w=_Registered(x[1], x[2]), out=empty(case["M"], case["N"]))
    elif kind == "f32":
        st.update(a=x[0], b=x[1], out=empty(case["batch"], case["M"], case["N"]))
    elif kind == "attention":
        st.update(qkv=x[0], out=empty(case["S"] * case["L"], case["heads"] * case["hd"]))
    elif kind == "ann":
        st.update(q=x[0].cpu().numpy(), w=_Registered(x[1], x[2]))
    else:
        e, layers, ids = x
        st.update(m=_Model(case, e, layers), ids=ids, h=empty(case["S"] * case["L"], case["hidden"]),
                  out=empty(case["S"], case["hidden"]))
    context()
    torch.cuda.synchronize()  # the context's stream does not wait for torch's
    return st


def run(st):
    c, case, kind = context(), st["case"], st["case"]["kind"]
    if kind == "linear":
        c.linear_dev(st["w"].w, st["a"].data_ptr(), case["M"], st["b"].data_ptr(), ACTS[case["act"]], st["out"].data_ptr())
        return st["out"]
    if kind == "linear_host":
        return c.linear(st["w"].w, st["a"], bias=st["b"], act=ACTS[case["act"]])
    if kind == "q8w":
        c.matmul_bt_q8_dev(st["w"].w, st["a"].data_ptr(), case["K"], case["M"], st["out"].data_ptr(), case["N"])
        return st["out"]
    if kind == "f32":
        M, K, N, nk = case["M"], case["K"], case["N"], case["layout"] == "nk"
        c.matmul_bt_f32_dev(st["a"].data_ptr(), K, st["b"].data_ptr(), K if nk else N, enchip.B_NK if nk else enchip.B_KN,
                            st["out"].data_ptr(), N, M, K, N,
                            inner=None if case["batch"] == 1 else (case["batch"], M * K, N * K, M * N))
        return st["out"]
    if kind == "attention":
        D, p = case["heads"] * case["hd"], st["qkv"].data_ptr()
        c.attention_f32_dev(p, p + 4 * D, p + 8 * D, 3 * D, st["out"].data_ptr(), D, case["S"], case["L"], case["heads"],
                            case["hd"], 1.0 / math.sqrt(case["hd"]))
        return st["out"]
    if kind == "ann":
        index, score = c.ann_topk(st["w"].w, st["q"], case["k"])
        return {"index": index, "score": score}
    m, S, L = st["m"].model, case["S"], case["L"]
    m.embeddings(st["ids"], S, L, st["h"])
    m.embed(st["h"], S, L, st["out"])
    return {"hidden": st["h"], "pooled": st["out"]}


# ---------------------------------------------------------------------------- accounting


def work(case):
    kind = case["kind"]
    if kind in ("linear", "linear_host", "q8w"):
        M, K, N = case["M"], case["K"], case["N"]
        return {"bytes": 4 * M * K + N * K + 8 * N + 4 * M * N, "flops": 2 * M * N * K}
    if kind == "f32":
        B, M, K, N = case["batch"], case["M"], case["K"], case["N"]
        return {"bytes": 4 * B * (M * K + N * K + M * N), "flops": 2 * B * M * N * K}
    if kind == "attention":
        rows, D = case["S"] * case["L"], case["heads"] * case["hd"]
        return {"bytes": 16 * rows * D, "flops": 4 * rows * case["L"] * D}
    if kind == "ann":
        n, d, M = case["rows"], case["dim"], case["M"]
        return {"bytes": n * d + 4 * n + 4 * M * d + 8 * M * case["k"], "flops": 2 * n * d * M}
    T, D, I, n = case["S"] * case["L"], case["hidden"], case["ffn"], case["layers"]
    params = n * (4 * D * D + 2 * D * I)
    return {"bytes": params + 4 * T + 8 * T * D + 4 * case["S"] * D, "flops": 2 * T * params + n * 4 * T * case["L"] * D}


def tolerance(case):
    kind = case["kind"]
    if kind in ("linear", "linear_host", "ann"):
        return "exact"  # the int32 dot is exact and the epilogue's roundings are the contract's
    if kind in ("q8w", "f32"):  # against 64 bits: 2.6e-7 at K = 768, 1e-6 at K = 3072
        return {"rel": 4e-6, "max": 1e-4}
    if kind == "attention":  # against 64 bits: up to 6e-7 (split f16 products, online softmax)
        return {"rel": 4e-6, "max": 1e-4}
    # The last bits of one layer's attention move int8 codes of the linears after it: the
    # library's three attention modes, each within 2e-4 of exact, give hidden states that
    # differ by 0.3% to 2.2% after 6 or 12 layers (at most 0.12 of the rms at one value).
    return {"rel": 3e-2, "max": 0.5}


# ---------------------------------------------------------------------------- 64-bit results


def _codes(x):
    """Activation codes and scales as the format defines them (f32 operations), of x[M, K]."""
    x = x.float()
    m = x.abs().amax(dim=1)
    zero = m == 0
    # f32 quotients, rounded once (torch divides by a number with its reciprocal)
    s = torch.where(zero, torch.ones_like(m), (m.double() / torch.full_like(m, 127.0).double()).float())
    v = (x * (torch.ones_like(m).double() / s.double()).float()[:, None]).double()
    q = torch.trunc(v + torch.copysign(torch.full_like(v, 0.5), v)).clamp(-127, 127)
    return q, torch.where(zero, torch.zeros_like(s), s).double()


def _linear64(x, wq, ws, b, act):
    out = []
    wd, ws, b = wq.double().t().contiguous(), ws.double(), b.double()
    for r in range(0, x.shape[0], 8192):
        q, s = _codes(x[r:r + 8192])
        y = (q @ wd) * s[:, None] * ws + b
        out.append(y * 0.5 * (1 + torch.erf(y / math.sqrt(2.0))) if act == "gelu" else y)
    return torch.cat(out)


def _attention64(qkv, S, L, heads, hd):
    D, out = heads * hd, []
    for z in range(S):
        t = qkv[z * L:(z + 1) * L].double().reshape(L, 3, heads, hd).permute(1, 2, 0, 3).contiguous()
        p = torch.softmax(torch.matmul(t[0], t[1].transpose(1, 2).contiguous()) / math.sqrt(hd), dim=-1)
        out.append(torch.matmul(p, t[2]).permute(1, 0, 2).reshape(L, D))
    return torch.cat(out)


def _ln64(x, ln):
    x = x.double()
    v = x - x.mean(dim=1, keepdim=True)
    return v / torch.sqrt((v * v).mean(dim=1, keepdim=True) + LN_EPS) * ln[0].double() + ln[1].double()


def _encode64(case, x):
    (e, layers, ids), S, L = x, case["S"], case["L"]
    h = e["word"][ids.long()].double() + e["pos"][e["off"]:e["off"] + L].double().repeat(S, 1)
    if e["typ"] is not None:
        h = h + e["typ"][0].double()
    h = _ln64(h, e["ln"])
    for lw in layers:
        c = _attention64(_linear64(h, *lw["qkv"], "none"), S, L, case["heads"], case["hidden"] // case["heads"])
        h = _ln64(h + _linear64(c, *lw["o"], "none"), lw["attn_ln"])
        h = _ln64(h + _linear64(_linear64(h, *lw["ffn_up"], "gelu"), *lw["ffn_down"], "none"), lw["out_ln"])
    return {"hidden": h, "pooled": torch.nn.functional.normalize(h.reshape(S, L, -1).mean(dim=1))}


def exact(case, seed):
    kind, x = case["kind"], _inputs(case, seed)
    if kind in ("linear", "linear_host"):
        y = _linear64(*x, case["act"])
        return y if kind == "linear" else y.cpu().numpy()
    if kind == "q8w":
        return x[0].double() @ (x[1].double() * x[2].double()[:, None]).t()
    if kind == "f32":
        a, b = x[0].double(), x[1].double()
        return torch.matmul(a, b.transpose(1, 2).contiguous() if case["layout"] == "nk" else b)
    if kind == "attention":
        return _attention64(x[0], case["S"], case["L"], case["heads"], case["hd"])
    if kind == "ann":
        q, s = _codes(x[0])
        best = []
        for r in range(0, case["rows"], 1 << 17):
            y = (q @ x[1][r:r + (1 << 17)].double().t()) * s[:, None] * x[2][r:r + (1 << 17)].double()
            best.append(torch.topk(y, min(case["k"], y.shape[1]), dim=1).values)
        return {"index": None, "score": torch.topk(torch.cat(best, dim=1), case["k"], dim=1).values.cpu().numpy()}
    return _encode64(case, x)
