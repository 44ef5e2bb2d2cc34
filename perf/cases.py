"""The work this framework is used for, as timed cases over its public entry points.

One model, Qwen3-VL-2B, as it runs on this library: the text decoder's
projections (hidden 2048, 16 query and 8 key/value heads of 128, intermediate
6144, vocabulary 151936) and the vision encoder's (hidden 1024, intermediate
4096, merger 4096 -> 4096 -> 2048), int8 weights with one fp32 scale per group
of 64 (the exporter also writes groups of 32 and 128). The activations are
N(0, 1) fp32, the weights int8 U[-127, 127] with U(0.001, 0.02) scales, the
caches N(0, 1) fp16.

A case is {"kind", sizes ...}. Kinds and what they stand for:

  linear    one linear() call: C = A W^T
  multi     q, k and v over one activation
  mlp       the MLP block: gate|up, SwiGLU, down
  vit       the four linears of one vision block (qkv, proj, fc1, fc2)
  merger    the vision merger's two linears (4096 -> 4096 -> 2048)
  lm_head   logits over the vocabulary and the greedy token of each row
  decode    one greedy decode step of the whole text model, a replay of the
            HIP graph that the caller captured, as a serving loop runs it

The entry points reproduce their reference bit for bit, so the tolerance is
"exact" throughout.
"""
from __future__ import annotations

import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                                "qwen3-vl-2b-inference_amd"))
import q3vl_int8 as q  # noqa: E402
from q3vl_int8 import model as qm  # noqa: E402

HIDDEN, INTER, VOCAB, LAYERS, HEADS, KV_HEADS, HEAD_DIM = 2048, 6144, 151936, 28, 16, 8, 128
VIS, VIS_INTER = 1024, 4096
EPS, THETA = 1e-6, 5e6
DECODE_ROOM = 8  # cache rows beyond the context, in whole rows of 8


def listed():
    return [
        # one token through one projection: the smallest call there is
        {"name": "linear_up_m1", "kind": "linear", "M": 1, "N": INTER, "K": HIDDEN, "gs": 64},
        # a handful of sequences decoded together
        {"name": "qkv_m4", "kind": "multi", "M": 4, "K": HIDDEN, "gs": 64},
        # a serving batch, or the prompt of a short question
        {"name": "mlp_m16", "kind": "mlp", "M": 16, "gs": 64},
        # prefill of an image and its question
        {"name": "mlp_m512", "kind": "mlp", "M": 512, "gs": 64},
        # prefill of a long prompt, with a ragged number of rows
        {"name": "mlp_m1501", "kind": "mlp", "M": 1501, "gs": 64},
        # one block of the vision encoder on a 448 x 448 image
        {"name": "vit_block_m784", "kind": "vit", "M": 784, "gs": 64},
        # the merger behind it (a quarter of the rows)
        {"name": "merger_m196", "kind": "merger", "M": 196, "gs": 64},
        # a checkpoint exported with groups of 128, a mid-sized prompt
        {"name": "mlp_g128_m300", "kind": "mlp", "M": 300, "gs": 128},
        # the next token's logits and greedy choice, one sequence and a batch
        {"name": "lm_head_m1", "kind": "lm_head", "M": 1, "gs": 64},
        {"name": "lm_head_m8", "kind": "lm_head", "M": 8, "gs": 64},
        # one generated token, in the reference's attention order and in the
        # chunked one, which long contexts use
        {"name": "decode_1024", "kind": "decode", "ctx": 1024, "order": 0},
        {"name": "decode_chunked_3000", "kind": "decode", "ctx": 3000, "order": 1},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["linear", "linear", "multi", "mlp", "mlp", "vit", "merger", "lm_head", "decode"])
    gs = rng.choice([64, 64, 64, 32, 128])
    if kind == "linear":
        N, K = rng.choice([(HIDDEN, HIDDEN), (INTER, HIDDEN), (HIDDEN, INTER), (KV_HEADS * HEAD_DIM, HIDDEN),
                           (VIS, 1536), (3 * VIS, VIS), (VIS_INTER, VIS), (VIS, VIS_INTER)])
        if rng.random() < 0.25:
            N -= rng.randrange(1, 64)  # a ragged slice of the rows
        return {"kind": kind, "M": _log(rng, 1, 2048), "N": N, "K": K, "gs": gs}
    if kind == "lm_head":
        return {"kind": kind, "M": rng.randint(1, 16), "gs": gs}
    if kind == "decode":
        return {"kind": kind, "ctx": _log(rng, 16, 3000), "order": rng.choice([0, 1])}
    hi = {"multi": 2048, "mlp": 1500, "vit": 2304, "merger": 576}[kind]
    return {"kind": kind, "M": _log(rng, 196 if kind == "vit" else 49 if kind == "merger" else 1, hi), "gs": gs}


# ------------------------------------------------------------------- inputs
def _rows(case):
    """(N, K) of the weights a case holds, in call order."""
    kind = case["kind"]
    if kind == "linear":
        return [(case["N"], case["K"])]
    if kind == "multi":
        return [(HEADS * HEAD_DIM, HIDDEN), (KV_HEADS * HEAD_DIM, HIDDEN), (KV_HEADS * HEAD_DIM, HIDDEN)]
    if kind == "mlp":
        return [(INTER, HIDDEN), (INTER, HIDDEN), (HIDDEN, INTER)]
    if kind == "vit":
        return [(3 * VIS, VIS), (VIS, VIS), (VIS_INTER, VIS), (VIS, VIS_INTER)]
    if kind == "merger":
        return [(VIS_INTER, VIS_INTER), (HIDDEN, VIS_INTER)]
    return [(VOCAB, HIDDEN)]  # lm_head


def _acts(case):
    """K of the activations a case is handed: one of its own for each vision
    and merger linear (norm, attention and GELU lie between them)."""
    rows = _rows(case)
    return [k for _, k in rows] if case["kind"] in ("vit", "merger") else [rows[0][1]]


def _weight(g, gs, *shape):
    w = torch.randint(-127, 128, shape, dtype=torch.int8, device="cuda", generator=g)
    s = torch.empty(shape[:-1] + (shape[-1] // gs,), device="cuda").uniform_(0.001, 0.02, generator=g)
    return w, s


def _make(case, seed):
    g = torch.Generator(device="cuda").manual_seed(int(seed))
    if case["kind"] == "decode":
        return _make_decode(case, g)
    w = [_weight(g, case["gs"], n, k) for n, k in _rows(case)]
    a = [torch.randn((case["M"], k), device="cuda", generator=g) for k in _acts(case)]
    return w, a


def _dims(case):
    S = (case["ctx"] + DECODE_ROOM) // 8 * 8 + 8
    return dict(vocab=VOCAB, hidden=HIDDEN, inter=INTER, layers=LAYERS, heads=HEADS, kv_heads=KV_HEADS,
                head_dim=HEAD_DIM, max_seq=S, gs=64, eps=EPS, attn_order=case["order"])


def _make_decode(case, g):
    d = _dims(case)
    L, H, I, D, S, gs = LAYERS, HIDDEN, INTER, HEAD_DIM, d["max_seq"], 64
    t = {}
    t["emb_w"], t["emb_s"] = _weight(g, gs, VOCAB, H)
    for n, shape in (("fnorm", (H,)), ("anorm", (L, H)), ("mnorm", (L, H)), ("qnorm", (L, D)), ("knorm", (L, D))):
        # weights U(0.9, 1.1) under the exporter's group scale
        w = torch.empty(shape, device="cuda").uniform_(0.9, 1.1, generator=g)
        s = w.reshape(-1, gs).abs().amax(1) / 127
        t[n + "_w"] = (w.reshape(-1, gs) / s[:, None]).round().clamp(-127, 127).to(torch.int8).reshape(shape)
        t[n + "_s"] = s.reshape(shape[:-1] + (shape[-1] // gs,)).contiguous()
    for n, N, K in (("q", HEADS * D, H), ("k", KV_HEADS * D, H), ("v", KV_HEADS * D, H), ("o", H, HEADS * D),
                    ("g", I, H), ("u", I, H), ("d", H, I)):
        t["w" + n], t["s" + n] = _weight(g, gs, L, N, K)
    inv = THETA ** (-torch.arange(0, D, 2, dtype=torch.float64) / D)
    ang = torch.arange(S, dtype=torch.float64)[:, None] * inv
    t["rope_cos"], t["rope_sin"] = ang.cos().float().cuda(), ang.sin().float().cuda()
    kv = []
    for _ in range(2):
        c = torch.zeros((L, KV_HEADS, S, D), dtype=torch.float16, device="cuda")
        c[:, :, : case["ctx"]] = torch.randn((L, KV_HEADS, case["ctx"], D), dtype=torch.float16, device="cuda", generator=g)
        kv.append(c)
    token = torch.randint(0, VOCAB, (1,), dtype=torch.int32, device="cuda", generator=g)
    return d, t, kv, token


# ------------------------------------------------------------------ the path
def prepare(case, seed):
    kind = case["kind"]
    if kind == "decode":
        d, t, (k, v), token = _make_decode(case, torch.Generator(device="cuda").manual_seed(int(seed)))
        st = {"kind": kind, "model": qm.DeviceTextModel.from_device(d, t), "k": k, "v": v, "first": token,
              "at": torch.tensor([case["ctx"]], dtype=torch.int32, device="cuda")}
        st["ws"] = qm.alloc_decode_workspace(st["model"])
        st["token"], st["pos"] = token.clone(), st["at"].clone()
        st["logits"] = torch.zeros(VOCAB, device="cuda")
        step = lambda: qm.decode_step(st["model"], k, v, st["token"], st["pos"], st["logits"], st["ws"])  # noqa: E731
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            step()  # first use of every kernel, outside the capture
        torch.cuda.current_stream().wait_stream(side)
        torch.cuda.synchronize()
        st["graph"] = torch.cuda.CUDAGraph()
        with torch.cuda.graph(st["graph"]):
            step()
        return st
    w, a = _make(case, seed)
    M, gs = case["M"], case["gs"]
    if kind == "mlp":
        need = q.mlp_workspace_bytes(M, HIDDEN, INTER, gs)
    else:
        need = max(q.workspace_bytes(M, n, k, gs) for n, k in _rows(case))
    out = [torch.empty((M, n), device="cuda") for n, _ in (_rows(case)[2:] if kind == "mlp" else _rows(case))]
    return {"kind": kind, "w": w, "a": a, "gs": gs, "out": out, "ws": torch.zeros(need, dtype=torch.uint8, device="cuda"),
            "ids": torch.zeros(M, dtype=torch.int32, device="cuda")}


def run(st):
    kind = st["kind"]
    if kind == "decode":
        # the sequence's last token and its position, then one step
        st["token"].copy_(st["first"])
        st["pos"].copy_(st["at"])
        st["graph"].replay()
        return {"logits": st["logits"], "token": st["token"], "k": st["k"], "v": st["v"]}
    w, a, gs, out, ws = st["w"], st["a"], st["gs"], st["out"], st["ws"]
    if kind == "multi":
        return q.linear_i8_multi(a[0], [x for x, _ in w], [s for _, s in w], gs, outs=out, workspace=ws)
    if kind == "mlp":
        (wg, sg), (wu, su), (wd, sd) = w
        return q.mlp_i8(a[0], wg, sg, wu, su, wd, sd, gs, out=out[0], workspace=ws)
    if kind == "lm_head":
        ids = q.lm_head_argmax(a[0], w[0][0], w[0][1], gs, logits=out[0], ids=st["ids"], workspace=ws)
        return {"logits": out[0], "ids": ids}
    return [q.linear_i8(x, wi, si, gs, out=o, workspace=ws) for x, (wi, si), o in zip(a, w, out)]


def work(case):
    if case["kind"] == "decode":
        per_layer = sum(n * k * (1 + 4 / 64) for n, k in (
            (2 * KV_HEADS * HEAD_DIM + HEADS * HEAD_DIM, HIDDEN), (HIDDEN, HEADS * HEAD_DIM), (2 * INTER, HIDDEN), (HIDDEN, INTER)))
        n_w = LAYERS * per_layer + VOCAB * HIDDEN * (1 + 4 / 64)
        kv = LAYERS * 2 * (case["ctx"] + 2) * KV_HEADS * HEAD_DIM
        return {"bytes": n_w + 2 * kv + 4 * VOCAB, "flops": 2 * n_w / (1 + 4 / 64) + LAYERS * 4 * (case["ctx"] + 1) * HEADS * HEAD_DIM}
    rows, M, gs = _rows(case), case["M"], case["gs"]
    outs = rows[2:] if case["kind"] == "mlp" else rows
    nbytes = sum(n * k + 4 * n * (k // gs) for n, k in rows) + 4 * M * (sum(_acts(case)) + sum(n for n, _ in outs))
    return {"bytes": nbytes, "flops": 2 * M * sum(n * k for n, k in rows)}


def tolerance(case):
    # every entry point promises the reference's bits: its orders of fp32
    # operations are fixed, and whole numbers are exact
    return "exact"


# ----------------------------------------------- the same in 64 bits, plainly
def _quant(x, gs):
    """int16 activations under a group scale of rms / 127, as the values they stand for."""
    g = x.double().reshape(x.shape[0], -1, gs)
    s = (g.square().mean(2, keepdim=True) + 1e-6).sqrt() / 127
    return ((g / s).round() * s).reshape(x.shape)


def _lin(x, w, s, gs):
    xq, out = _quant(x, gs), []
    for i in range(0, w.shape[0], 16384):  # the weight in 64 bits, some rows at a time
        wi = w[i:i + 16384].double().reshape(-1, w.shape[1] // gs, gs) * s[i:i + 16384].double()[..., None]
        out.append(xq @ wi.reshape(-1, w.shape[1]).t().contiguous())
    return torch.cat(out, 1)


def _norm(x, w, s, gs=64):
    wd = (w.double().reshape(-1, gs) * s.double().reshape(-1, 1)).reshape(-1)
    return x / (x.square().mean(-1, keepdim=True) + EPS).sqrt() * wd


def _rope(x, cos, sin):
    a, b = x[..., : HEAD_DIM // 2], x[..., HEAD_DIM // 2:]
    return torch.cat([a * cos - b * sin, b * cos + a * sin], -1)


def exact(case, seed):
    if case["kind"] == "decode":
        return _exact_decode(case, seed)
    w, a = _make(case, seed)
    gs, kind = case["gs"], case["kind"]
    if kind == "multi":
        return [_lin(a[0], wi, si, gs) for wi, si in w]
    if kind == "mlp":
        gate, up = (_lin(a[0], wi, si, gs) for wi, si in w[:2])
        return _lin(gate * torch.sigmoid(gate) * up, *w[2], gs)
    if kind == "lm_head":
        return {"logits": _lin(a[0], *w[0], gs), "ids": None}
    return [_lin(x, wi, si, gs) for x, (wi, si) in zip(a, w)]


def _exact_decode(case, seed):
    d, t, (kc, vc), token = _make_decode(case, torch.Generator(device="cuda").manual_seed(int(seed)))
    gs, p = 64, case["ctx"]
    tok = int(token.item())
    x = (t["emb_w"][tok].double().reshape(-1, gs) * t["emb_s"][tok].double()[:, None]).reshape(1, -1)
    cos, sin = t["rope_cos"][p].double(), t["rope_sin"][p].double()
    kd, vd = kc.double(), vc.double()
    for l in range(LAYERS):
        lin = lambda y, n: _lin(y, t["w" + n][l], t["s" + n][l], gs)  # noqa: E731
        y = _norm(x, t["anorm_w"][l], t["anorm_s"][l])
        qh = _rope(_norm(lin(y, "q").reshape(HEADS, HEAD_DIM), t["qnorm_w"][l], t["qnorm_s"][l]), cos, sin)
        kh = _rope(_norm(lin(y, "k").reshape(KV_HEADS, HEAD_DIM), t["knorm_w"][l], t["knorm_s"][l]), cos, sin)
        kd[l, :, p], vd[l, :, p] = kh.half().double(), lin(y, "v").reshape(KV_HEADS, HEAD_DIM).half().double()
        rep = HEADS // KV_HEADS
        ks, vs = kd[l, :, : p + 1].repeat_interleave(rep, 0), vd[l, :, : p + 1].repeat_interleave(rep, 0)
        pr = torch.softmax((ks * qh[:, None, :]).sum(2) / math.sqrt(HEAD_DIM), 1)
        x = x + lin((pr[..., None] * vs).sum(1).reshape(1, -1), "o")
        y = _norm(x, t["mnorm_w"][l], t["mnorm_s"][l])
        gate = lin(y, "g")
        x = x + lin(gate * torch.sigmoid(gate) * lin(y, "u"), "d")
    y = _norm(x, t["fnorm_w"], t["fnorm_s"])
    return {"logits": _lin(y, t["emb_w"], t["emb_s"], gs)[0], "token": None, "k": kd, "v": vd}
