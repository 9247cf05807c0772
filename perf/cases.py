"""Timing cases of the RT4 path: what a runtime has this library do, through rt4_amd's public functions.

Four kinds of call, at the 27B layer shapes of rt4_amd/workload.py (hidden 5120, feed-forward 17408, vocabulary 248320,
24 query heads over 4 KV heads) and around them:

* ``linear``:    one decode linear (1-4 activation rows), called eagerly: quantize the activations, then the GEMV.
* ``mlp``:       the gate, up and down linears of a few layers as one HIP graph that the program captured once and replays
                 for every token, as a serving loop does.
* ``prefill``:   one prompt linear: the row quantizer, then the GEMM.  ``entry`` is "i8" (int8 codes, any number of rows),
                 "dropin" (the h/l digit planes of the reference's calls, rows padded to 128) or "a4" (W4A4).
* ``attention``: one layer's attention over a chunk of new tokens: quantize Q, append K and V, causal prefill.

Inputs follow rt4_amd/workload.py: int4 codes uniform in [-8, 7], |N(0,1)|*0.01 + 1e-3 fp16 weight scales, fp16-valued N(0,1)
activations with 1% outliers (x20) in prompts, N(0,1) Q/K/V with Q scaled by 1/sqrt(256).
"""
from __future__ import annotations

import math
import pathlib
import sys

import torch

_ROOT = pathlib.Path(__file__).resolve().parents[1]
if str(_ROOT / "k100lc-rt4_amd") not in sys.path:
    sys.path.insert(0, str(_ROOT / "k100lc-rt4_amd"))
import rt4_amd  # noqa: E402

DEV = "cuda"
G = 128
D = 256


def listed():
    return [
        # The smallest call: one token through one square projection; latency and launches are what counts.
        {"name": "linear_m1_5120", "kind": "linear", "bits": 8, "M": 1, "N": 5120, "K": 5120},
        # W4A4 option, two rows, the down projection's deep K.
        {"name": "linear_a4_m2_down", "kind": "linear", "bits": 4, "M": 2, "N": 5120, "K": 17408},
        # The LM head over a draft of three tokens and the one they follow: the largest weight stream.
        {"name": "lm_head_m4", "kind": "linear", "bits": 8, "M": 4, "N": 248320, "K": 5120},
        # Decode of one token, and of a four-token verify step: the MLP of two layers, replayed from a graph.
        {"name": "mlp_m1", "kind": "mlp", "M": 1, "H": 5120, "F": 17408, "layers": 2},
        {"name": "mlp_m4", "kind": "mlp", "M": 4, "H": 5120, "F": 17408, "layers": 2},
        # A short prompt of an odd length; a medium one on the W4A4 path; a full chunk through the int8 entry and the
        # reference's own benchmark size through the drop-in entry.
        {"name": "prefill_i8_m37", "kind": "prefill", "entry": "i8", "M": 37, "N": 17408, "K": 5120},
        {"name": "prefill_a4_m384_down", "kind": "prefill", "entry": "a4", "M": 384, "N": 5120, "K": 17408},
        {"name": "prefill_i8_m1024", "kind": "prefill", "entry": "i8", "M": 1024, "N": 17408, "K": 5120},
        {"name": "prefill_dropin_m2048", "kind": "prefill", "entry": "dropin", "M": 2048, "N": 17408, "K": 5120},
        # A follow-up turn of 43 tokens over a 4096-token cache; a first prompt of 1000 tokens; a 1024-token chunk over
        # a 32768-token cache.
        {"name": "attn_turn43_ctx4k", "kind": "attention", "T": 43, "ctx": 4096, "QH": 24, "KVH": 4},
        {"name": "attn_first1000", "kind": "attention", "T": 1000, "ctx": 0, "QH": 24, "KVH": 4},
        {"name": "attn_1024_ctx32k", "kind": "attention", "T": 1024, "ctx": 32768, "QH": 24, "KVH": 4},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["linear", "mlp", "prefill", "prefill", "attention"])
    if kind == "linear":
        return {"kind": kind, "bits": rng.choice([8, 8, 4]), "M": rng.randint(1, 4), "N": _log(rng, 256, 100000),
                "K": 128 * _log(rng, 4, 136)}
    if kind == "mlp":
        return {"kind": kind, "M": rng.randint(1, 4), "H": 128 * _log(rng, 8, 64), "F": 128 * _log(rng, 16, 224),
                "layers": rng.randint(1, 2)}
    if kind == "prefill":
        entry = rng.choice(["i8", "i8", "dropin", "a4"])
        M = _log(rng, 5, 2048) if entry == "i8" else 128 * _log(rng, 1, 16)
        N = _log(rng, 256, 17408) if entry == "i8" else 64 * _log(rng, 4, 272)
        K = 128 * _log(rng, 4, 136)
        while M * N * K > 2048 * 17408 * 5120:
            K = 128 * (K // 256)
        return {"kind": kind, "entry": entry, "M": M, "N": N, "K": K}
    kvh = rng.choice([1, 2, 4, 8])
    qh = kvh * rng.choice([1, 4, 6, 8])
    T = _log(rng, 5, 1024)
    ctx = 64 * (_log(rng, 1, 513) - 1)
    while T * (ctx + T) * qh > 1024 * 33792 * 24:
        ctx = 64 * (ctx // 128)
    return {"kind": kind, "T": T, "ctx": ctx, "QH": qh, "KVH": kvh}


# ------------------------------------------------------------------ inputs --
def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(1 + seed)
    return g


def _weights(N, K, g):
    """RT4 weights: (wq int32 [N, K/8], ws int16 [N, K/128], the bits of the fp16 scales)."""
    wq = torch.randint(0, 256, (N, K // 2), dtype=torch.uint8, device=DEV, generator=g).view(torch.int32)
    s = torch.randn((N, K // G), device=DEV, generator=g).abs() * 0.01 + 1e-3
    return wq, s.to(torch.float16).view(torch.int16)


def _acts(M, K, g, outliers=False):
    x = torch.randn((M, K), device=DEV, generator=g).to(torch.float16).to(torch.float32)
    if outliers:
        x = torch.where(torch.rand((M, K), device=DEV, generator=g) < 0.01, x * 20.0, x)
    return x


def _padded(T):
    return (T + 63) // 64 * 64


def prepare(case, seed):
    g = _gen(seed)
    k = case["kind"]
    st = {"case": case}
    if k == "linear":
        M, N, K = case["M"], case["N"], case["K"]
        st["wq"], st["ws"] = _weights(N, K, g)
        st["x"] = _acts(M, K, g)
        st["y"] = torch.empty((M, N), device=DEV)
    elif k == "mlp":
        M, H, F = case["M"], case["H"], case["F"]
        st["layers"] = [{"gate": _weights(F, H, g), "up": _weights(F, H, g), "down": _weights(H, F, g)}
                        for _ in range(case["layers"])]
        st["x"] = [_acts(M, H, g) for _ in range(case["layers"])]
        st["h"] = [_acts(M, F, g) for _ in range(case["layers"])]   # the activated gate*up of each layer
        st["y"] = [{"gate": torch.empty((M, F), device=DEV), "up": torch.empty((M, F), device=DEV),
                    "down": torch.empty((M, H), device=DEV)} for _ in range(case["layers"])]
        _mlp(st)                                # one eager step sizes the library's scratch
        torch.cuda.synchronize()
        st["graph"] = torch.cuda.CUDAGraph()
        with torch.cuda.graph(st["graph"]):
            _mlp(st)
    elif k == "prefill":
        M, N, K = case["M"], case["N"], case["K"]
        st["wq"], st["ws"] = _weights(N, K, g)
        st["wsc"] = rt4_amd.make_group_major(st["ws"], K)     # laid out once, at load time
        st["x"] = _acts(M, K, g, outliers=True)
        st["c"] = torch.empty((M, N), device=DEV)
        if case["entry"] == "dropin":
            st["c2"] = torch.empty((M, N), device=DEV)
    else:
        T, ctx, QH, KVH = case["T"], case["ctx"], case["QH"], case["KVH"]
        TP, cap = _padded(T), _padded(ctx + T)
        st["kc"] = torch.zeros((KVH, cap, D // 8), dtype=torch.int32, device=DEV)
        st["ksc"] = torch.ones((KVH, D // G, cap), device=DEV)
        st["vc"] = torch.zeros((KVH, cap // 8, D), dtype=torch.int32, device=DEV)
        st["vsc"] = torch.ones((KVH, cap // 64, D), device=DEV)
        st["stage"] = torch.zeros((KVH, 64, D), device=DEV)
        if ctx:
            rt4_amd.kv_append_k(st["kc"], st["ksc"], _acts(ctx * KVH, D, g).view(ctx, KVH, D), 0)
            rt4_amd.kv_append_v(st["vc"], st["vsc"], st["stage"], _acts(ctx * KVH, D, g).view(ctx, KVH, D), 0)
        st["q"] = (_acts(T * QH, D, g) * (D ** -0.5)).view(T, QH, D)
        st["k"] = _acts(T * KVH, D, g).view(T, KVH, D)
        st["v"] = _acts(T * KVH, D, g).view(T, KVH, D)
        st["qq"] = torch.zeros((QH, TP, D // 8), dtype=torch.int32, device=DEV)
        st["qs"] = torch.ones((QH, D // G, TP), device=DEV)
        st["out"] = torch.empty((QH, TP, D), device=DEV)
    return st


# -------------------------------------------------------------------- runs --
def _mlp(st):
    for w, x, h, y in zip(st["layers"], st["x"], st["h"], st["y"]):
        rt4_amd.gemv_w4a8(*w["gate"], x, out=y["gate"])
        rt4_amd.gemv_w4a8(*w["up"], x, out=y["up"])
        rt4_amd.gemv_w4a8(*w["down"], h, out=y["down"])


def run(st):
    case = st["case"]
    k = case["kind"]
    if k == "linear":
        f = rt4_amd.gemv_w4a8 if case["bits"] == 8 else rt4_amd.gemv_w4a4
        return f(st["wq"], st["ws"], st["x"], out=st["y"])
    if k == "mlp":
        st["graph"].replay()
        return st["y"]
    if k == "prefill":
        if case["entry"] == "i8":
            xq, sc = rt4_amd.quant_rows_i8(st["x"])
            return {"c": rt4_amd.gemm_w4a8_i8(st["wq"], st["wsc"], xq, sc, out=st["c"]), "xq": xq, "sc": sc}
        if case["entry"] == "a4":
            q, sc = rt4_amd.quant_rows_a4(st["x"])
            return {"c": rt4_amd.gemm_w4a4(st["wq"], st["wsc"], q, sc, out=st["c"]), "q": q, "sc": sc}
        qh, ql, sc, sc16 = rt4_amd.quant_rows_a8(st["x"])
        c = rt4_amd.gemm_w4a8(st["wq"], st["wsc"], qh, ql, sc, sc16, out=st["c"], c2=st["c2"])
        return {"c": c, "qh": qh, "ql": ql, "sc": sc, "sc16": sc16}
    T, ctx = case["T"], case["ctx"]
    rt4_amd.attn_q_quant(st["q"], st["out"].shape[1], qq=st["qq"], qs=st["qs"])
    rt4_amd.kv_append_k(st["kc"], st["ksc"], st["k"], ctx)
    rt4_amd.kv_append_v(st["vc"], st["vsc"], st["stage"], st["v"], ctx)
    out = rt4_amd.attention_prefill(st["qq"], st["qs"], st["kc"], st["ksc"], st["vc"], st["vsc"], n_kv=ctx + T, off=ctx,
                                    ratio=case["QH"] // case["KVH"], out=st["out"])
    return {"out": out, "qq": st["qq"], "qs": st["qs"], "kc": st["kc"], "ksc": st["ksc"], "vc": st["vc"], "vsc": st["vsc"]}


# -------------------------------------------------------------------- work --
def _linear_bytes(M, N, K):
    return N * K // 2 + N * K // 64 + 4 * M * K + 4 * M * N   # codes, fp16 scales, fp32 activations in and outputs out


def work(case):
    k = case["kind"]
    if k == "linear":
        M, N, K = case["M"], case["N"], case["K"]
        return {"bytes": _linear_bytes(M, N, K), "flops": 2 * M * N * K}
    if k == "mlp":
        M, H, F, L = case["M"], case["H"], case["F"], case["layers"]
        return {"bytes": L * (2 * _linear_bytes(M, F, H) + _linear_bytes(M, H, F)), "flops": L * 6 * M * H * F}
    if k == "prefill":
        M, N, K = case["M"], case["N"], case["K"]
        # codes, fp32 scales, activations; the quantized activations are outputs too (1 byte an element, 1/2 for a4)
        out = M * K // 2 if case["entry"] == "a4" else M * K
        return {"bytes": N * K // 2 + N * K // 32 + 4 * M * K + out + M * K // 32 + 4 * M * N, "flops": 2 * M * N * K}
    T, ctx, QH, KVH = case["T"], case["ctx"], case["QH"], case["KVH"]
    n_kv = ctx + T
    cache = KVH * (n_kv * D + 8 * n_kv + n_kv * D // 16)             # K and V codes, K scales, V scales
    return {"bytes": cache + 4 * D * T * (QH + 2 * KVH) + 4 * D * QH * _padded(T) + T * D * (QH + 2 * KVH) // 2,
            "flops": 4 * D * QH * (T * ctx + T * (T + 1) // 2)}


def tolerance(case):
    if case["kind"] == "attention":
        # The 3-bit P codes: an S that differs in its last bits can flip a code, which moves one row by up to a seventh
        # of a key's weight (two correct kernels differ by 2.4e-4 over the 32k case, and by more on a short row).
        return {"rel": 2e-3, "max": 0.5}
    return {"rel": 1e-6, "max": 1e-5}    # fp32 sums over the K groups, in any order


# ------------------------------------------------------------------- exact --
def _codes(x, div, lo, hi, group):
    """Per-group quantization as the formats define it (fp32 scale and quotient, half to even): codes, scales in float64."""
    v = x.reshape(-1, group)
    # (divided tensor by tensor: torch multiplies by the reciprocal of a plain number)
    amax = v.abs().amax(1, keepdim=True)
    s = torch.where(amax > 0, amax / torch.full_like(amax, div), torch.ones_like(amax))
    c = torch.round(v / s).clamp(lo, hi).double()
    return c.reshape(x.shape), s.double().reshape(*x.shape[:-1], x.shape[-1] // group)


def _nibbles(w):
    """int32 [..., n] -> signed codes float64 [..., 8n], low nibble first."""
    sh = 4 * torch.arange(8, device=w.device, dtype=torch.int32)
    c = (w.unsqueeze(-1) >> sh) & 15
    return torch.where(c > 7, c - 16, c).reshape(*w.shape[:-1], -1).double()


def _times_w(a, wq, ws):
    """a [M, K] float64 times the dequantized weights."""
    outs, step = [], max(1, (1 << 27) // (wq.shape[1] * 8))
    for n in range(0, wq.shape[0], step):
        w = _nibbles(wq[n:n + step])
        w = w.view(w.shape[0], -1, G) * ws[n:n + step].view(torch.float16).double().unsqueeze(-1)
        outs.append(a @ w.view(w.shape[0], -1).T)
    return torch.cat(outs, 1)


def _dequant(x, div, lo, hi, group):
    c, s = _codes(x, div, lo, hi, group)
    return (c.reshape(*s.shape, group) * s.unsqueeze(-1)).reshape(x.shape), s


def exact(case, seed):
    st = prepare(case, seed)
    k = case["kind"]
    if k == "linear":
        a, _ = _dequant(st["x"], 127.0, -128, 127, G) if case["bits"] == 8 else _dequant(st["x"], 7.0, -8, 7, 32)
        return _times_w(a, st["wq"], st["ws"])
    if k == "mlp":
        got = []
        for w, x, h in zip(st["layers"], st["x"], st["h"]):
            ax, ah = (_dequant(v, 127.0, -128, 127, G)[0] for v in (x, h))
            got.append({"gate": _times_w(ax, *w["gate"]), "up": _times_w(ax, *w["up"]), "down": _times_w(ah, *w["down"])})
        return got
    if k == "prefill":
        a, s = _dequant(st["x"], 7.0, -8, 7, G) if case["entry"] == "a4" else _dequant(st["x"], 119.0, -128, 119, G)
        r = {"c": _times_w(a, st["wq"], st["ws"]), "sc": s.T.contiguous()}
        if case["entry"] == "dropin":
            r.update(qh=None, ql=None, sc16=16 * r["sc"])
        else:
            r["q" if case["entry"] == "a4" else "xq"] = None
        return r
    return _exact_attention(st)


def _exact_attention(st):
    """The fixed-point tile algorithm in float64: per 64-key tile P = int(7 exp(S - tile max) + 1/2), tiles weighted by
    exp(tile max - row max) / 7."""
    c = st["case"]
    T, ctx, QH, KVH = c["T"], c["ctx"], c["QH"], c["KVH"]
    n_kv, TP = ctx + T, _padded(T)
    cap = st["kc"].shape[1]
    # the cache before the call holds ctx keys; the new ones are quantized here
    kq, ks = _codes(st["k"], 7.0, -8, 7, G)
    K = torch.zeros((KVH, cap, D), dtype=torch.float64, device=DEV)
    ksc = st["ksc"].double()
    if ctx:
        K[:, :ctx] = _nibbles(st["kc"][:, :ctx])
    K[:, ctx:n_kv] = kq.permute(1, 0, 2)
    ksc[:, :, ctx:n_kv] = ks.permute(1, 2, 0)
    K = (K.view(KVH, cap, D // G, G) * ksc.permute(0, 2, 1).unsqueeze(-1)).view(KVH, cap, D)
    nt = cap // 64
    vf = torch.zeros((cap - ctx, KVH, D), device=DEV)
    vf[:T] = st["v"]
    vt = vf.view(-1, 64, KVH, D).permute(2, 0, 3, 1).contiguous()                       # [KVH, new tiles, D, 64]
    vq, vs = _codes(vt, 7.0, -8, 7, 64)
    V = torch.zeros((KVH, cap, D), dtype=torch.float64, device=DEV)
    if ctx:
        V[:, :ctx] = _nibbles(st["vc"][:, :ctx // 8].transpose(1, 2).contiguous()).transpose(1, 2)
    V[:, ctx:] = vq.permute(0, 1, 3, 2).reshape(KVH, -1, D)
    V[:, n_kv // 8 * 8:] = 0                                # a last partial group of 8 keys is not read
    vsc = st["vsc"].double()
    vsc[:, ctx // 64:] = vs.squeeze(-1)
    V = (V.view(KVH, nt, 64, D) * vsc.unsqueeze(2)).view(KVH, cap, D)
    Q = torch.zeros((TP, QH, D), dtype=torch.float64, device=DEV)
    Q[:T], qs = _dequant(st["q"], 7.0, -8, 7, G)
    qsf = torch.ones((QH, D // G, TP), dtype=torch.float64, device=DEV)
    qsf[:, :, :T] = qs.permute(1, 2, 0)
    out = torch.empty((QH, TP, D), dtype=torch.float64, device=DEV)
    key, row = torch.arange(cap, device=DEV), ctx + torch.arange(TP, device=DEV)
    hidden = key[None, :] > row[:, None]
    for h in range(QH):
        S = Q[:, h] @ K[h * KVH // QH].T
        S[hidden] = -math.inf
        S = S.view(TP, nt, 64)
        mt = S.amax(2, keepdim=True)
        p = torch.floor(7.0 * torch.exp(S - torch.where(mt.isfinite(), mt, torch.zeros_like(mt))) + 0.5)
        p = p * torch.exp(mt - mt.amax(1, keepdim=True))
        p = p.view(TP, cap)
        out[h] = (p @ V[h * KVH // QH]) / p.sum(1, keepdim=True)
    return {"out": out, "qq": None, "qs": qsf, "kc": None, "ksc": ksc, "vc": None, "vsc": vsc}
