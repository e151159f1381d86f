"""Workloads of the fused attention / normalisation path, timed through the
package's public entry points: the ctypes binding of the kernel C ABI
(`jax_mlx_amd.native`) and, for whole modules, the PJRT client
(`jax_mlx_amd.pjrt`).

Each case is a dict of plain values.  `kind` picks the operation:

  norm        LayerNorm / RMSNorm forward over rows (every block of a model
              runs two of them)
  softmax     log-softmax over a vocabulary-sized axis (the loss / sampling
              head); such axes are rarely a multiple of anything
  norm_bwd    LayerNorm backward (training)
  attention   prefill / encoder / training-forward attention, with the masks
              models use: none, causal, a padding mask, an additive bias per
              (head, query, key), a 0 / -inf band (sliding window)
  decode      one new token per sequence against a KV cache of ragged
              lengths, with grouped-query heads and a fused q RMSNorm
  attention_bwd   the gradients of attention, from the forward's residuals
              (a training step in one module) or recomputing (custom_call)
  dense       a dense layer's forward, input gradient and weight gradient
  transformer a whole pre-LN transformer forward compiled from StableHLO
"""
from __future__ import annotations

import math
import sys
from pathlib import Path

import torch

REPO = Path(__file__).resolve().parent.parent
if str(REPO / "jax-mlx-plugin_amd") not in sys.path:
    sys.path.insert(0, str(REPO / "jax-mlx-plugin_amd"))

from jax_mlx_amd import native, pjrt  # noqa: E402

DT = {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16}
SIZE = {"f32": 4, "bf16": 2, "f16": 2}


# ---- the cases -----------------------------------------------------------------

def listed():
    return [
        # One sequence batch's LayerNorm in a small encoder: shorter than a launch.
        dict(name="layer_norm_small", kind="norm", op="layer", dtype="f32", rows=1024, n=512),
        # The same operation where it streams HBM: a long-sequence training batch.
        dict(name="layer_norm_large", kind="norm", op="layer", dtype="f32", rows=65536, n=4096),
        # The head of a language model: an odd vocabulary, so no row but the first is aligned.
        dict(name="log_softmax_vocab", kind="softmax", dtype="f32", rows=4096, n=32003),
        # The backward of a training step's LayerNorm.
        dict(name="layer_norm_bwd", kind="norm_bwd", dtype="f32", rows=65536, n=4096),
        # A short f32 attention: latency.
        dict(name="attention_f32_small", kind="attention", dtype="f32", B=8, Hq=8, Hkv=8, Tq=128, Tk=128, D=64,
             mask="none", layout="bhtd"),
        # Causal prefill / training forward, the ordinary large call.
        dict(name="attention_causal", kind="attention", dtype="bf16", B=4, Hq=32, Hkv=32, Tq=2048, Tk=2048, D=128,
             mask="causal", layout="bhtd"),
        # Attention with a learned or distance bias per head, ragged length, grouped-query heads, BTNH.
        dict(name="attention_bias", kind="attention", dtype="bf16", B=4, Hq=16, Hkv=4, Tq=1999, Tk=1999, D=128,
             mask="bias", layout="bthd"),
        # Serving: one token for each of 16 sequences of 1024..8192 cached keys.
        dict(name="decode", kind="decode", dtype="bf16", B=16, Hq=32, Hkv=8, Tk=8192, D=128),
        # Training step of the causal attention in bf16.
        dict(name="attention_bwd_bf16", kind="attention_bwd", dtype="bf16", B=4, Hq=32, Hkv=32, Tq=2048, Tk=2048,
             D=128, mask="causal", layout="bhtd", residuals=True),
        # The f32 transformer's attention in training, as the custom_call runs it (nothing kept from the forward).
        dict(name="attention_bwd_f32", kind="attention_bwd", dtype="f32", B=32, Hq=8, Hkv=8, Tq=256, Tk=256, D=64,
             mask="none", layout="bthd", residuals=False),
        # A bf16 MLP layer in training: x W, dy W^T and x^T dy.
        dict(name="dense_bf16", kind="dense", dtype="bf16", M=8192, K=512, N=2048),
        # The f32 transformer end to end through PJRT.
        dict(name="transformer_f32", kind="transformer", layers=4, B=32, T=256, d=512, heads=8, mlp=2048,
             causal=False),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["norm", "softmax", "norm_bwd", "attention", "attention", "decode", "attention_bwd",
                       "attention_bwd", "dense", "transformer"])
    if kind in ("norm", "norm_bwd"):
        # Widths of models: mostly multiples of 64, some odd.
        n = 64 * _log(rng, 2, 128) if rng.random() < 0.75 else _log(rng, 100, 8192)
        rows = min(_log(rng, 1, 1 << 18), (1 << 28) // n)
        c = dict(kind=kind, dtype=rng.choice(["f32", "f32", "bf16", "f16"]), rows=rows, n=n)
        return dict(c, op=rng.choice(["layer", "rms"])) if kind == "norm" else c
    if kind == "softmax":
        n = _log(rng, 1000, 65536)
        return dict(kind=kind, dtype=rng.choice(["f32", "f32", "bf16"]), rows=min(_log(rng, 1, 16384), (1 << 27) // n), n=n)
    if kind == "decode":
        group = rng.choice([1, 4, 8])
        Hkv = rng.choice([2, 4, 8])
        Tk = _log(rng, 128, 16384)
        B = min(_log(rng, 1, 64), max(1, (1 << 20) // (Tk * Hkv)))
        return dict(kind=kind, dtype=rng.choice(["bf16", "bf16", "f16"]), B=B, Hq=Hkv * group, Hkv=Hkv, Tk=Tk,
                    D=rng.choice([64, 128, 128]))
    if kind == "dense":
        # Features are multiples of 8 in nearly every model; token counts are anything.
        step = 8 if rng.random() < 0.85 else 1
        K = step * (_log(rng, 128, 4096) // step)
        N = step * (_log(rng, 128, 4096) // step)
        M = min(_log(rng, 16, 16384), int(3e11 / (6 * K * N)))
        if rng.random() < 0.6:
            M = max(16, M // 16 * 16)
        return dict(kind=kind, dtype=rng.choice(["bf16", "bf16", "f16", "f32"]), M=M, K=K, N=N)
    if kind == "transformer":
        heads = rng.choice([2, 4, 8, 12])
        T = _log(rng, 16, 512)
        B = max(1, min(_log(rng, 1, 32), 8192 // T))
        return dict(kind=kind, layers=rng.randint(1, 4), B=B, T=T, d=heads * 64, heads=heads, mlp=heads * 256,
                    causal=rng.random() < 0.5)
    dtype = rng.choice(["f32", "bf16", "bf16", "f16"])
    D = rng.choice([32, 64, 64, 96, 128, 128])
    group = rng.choice([1, 1, 2, 4])
    mask = rng.choice(["none", "causal", "causal", "padding", "bias", "band"])
    T = _log(rng, 17, 4096) if dtype != "f32" else _log(rng, 17, 1024)
    Tk = T if mask in ("causal", "band") or rng.random() < 0.7 else _log(rng, 17, 4096 if dtype != "f32" else 1024)
    # Heads and batch up to what the largest listed case of the direction and type costs.
    bwd = kind == "attention_bwd"
    cap = (1.0e10 if bwd else 6.0e10) if dtype == "f32" else 1.3e11
    most = max(1, int(cap / ((10 if bwd else 4) * T * Tk * D)))
    pairs = max(1, min(most, _log(rng, 4, 512)))
    Hq = max(1, min(pairs, rng.choice([2, 8, 12, 16, 32])) // group) * group
    c = dict(kind=kind, dtype=dtype, B=max(1, pairs // Hq), Hq=Hq, Hkv=Hq // group, Tq=T, Tk=Tk, D=D, mask=mask,
             layout=rng.choice(["bhtd", "bthd"]))
    return dict(c, residuals=rng.random() < 0.5) if bwd else c


# ---- inputs --------------------------------------------------------------------

class _Draws:
    """Device tensors from one seeded generator."""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda")
        self.g.manual_seed(seed)

    def normal(self, *shape, dtype=torch.float32, std=1.0, mean=0.0):
        t = torch.randn(shape, generator=self.g, device="cuda")
        if std != 1.0:
            t.mul_(std)
        if mean:
            t.add_(mean)
        return t if dtype == torch.float32 else t.to(dtype)

    def uniform(self, *shape, lo=0.0, hi=1.0, dtype=torch.float32):
        return torch.rand(shape, generator=self.g, device="cuda").mul_(hi - lo).add_(lo).to(dtype)

    def ints(self, lo, hi, *shape):
        return torch.randint(lo, hi + 1, shape, generator=self.g, device="cuda")


def _heads(d, c, H, T, dt):
    shape = (c["B"], H, T, c["D"]) if c["layout"] == "bhtd" else (c["B"], T, H, c["D"])
    return d.normal(*shape, dtype=dt)


def _length_mask(lengths, Tk):
    """Additive [B, 1, 1, Tk]: 0 before each sequence's length, -inf after."""
    keep = torch.arange(Tk, device="cuda")[None] < lengths[:, None]
    return torch.zeros(lengths.numel(), Tk, device="cuda").masked_fill_(~keep, -math.inf)[:, None, None]


def _mask(d, c):
    """The additive mask tensor of an attention case, or None."""
    Tq, Tk = c["Tq"], c["Tk"]
    if c["mask"] == "padding":
        return _length_mask(d.ints(max(1, Tk // 2), Tk, c["B"]), Tk)
    if c["mask"] == "bias":  # one [Tq, Tk] bias per head, shared by the batch, of the model's type
        return d.normal(1, c["Hq"], Tq, Tk, dtype=DT[c["dtype"]])
    if c["mask"] == "band":  # the predicate of a causal sliding window, as jnp.where(pred, 0, -inf)
        i = torch.arange(Tq, device="cuda")[:, None]
        j = torch.arange(Tk, device="cuda")[None]
        w = max(1, Tk // 4)
        return torch.zeros(1, 1, Tq, Tk, device="cuda").masked_fill_((j > i) | (j <= i - w), -math.inf)
    return None


def prepare(case, seed):
    c, d = case, _Draws(seed)
    kind = c["kind"]
    dt = DT[c.get("dtype", "f32")]
    s = {"case": c}
    if kind in ("norm", "norm_bwd", "softmax"):
        s["x"] = d.normal(c["rows"], c["n"], dtype=dt, std=3.0 if kind == "softmax" else 1.0)
        if kind == "softmax":
            return s
        s["gamma"] = d.normal(c["n"], dtype=dt, std=0.1, mean=1.0)
        if kind == "norm_bwd":
            s["dy"] = d.normal(c["rows"], c["n"], dtype=dt)
        else:
            s["beta"] = d.normal(c["n"], dtype=dt, std=0.1)
    elif kind == "decode":
        s["q"] = d.normal(c["B"], c["Hq"], 1, c["D"], dtype=dt)
        s["k"], s["v"] = (d.normal(c["B"], c["Hkv"], c["Tk"], c["D"], dtype=dt) for _ in range(2))
        s["weight"] = d.normal(c["D"], dtype=dt, std=0.1, mean=1.0)
        s["mask"] = _length_mask(d.ints(max(1, c["Tk"] // 8), c["Tk"], c["B"]), c["Tk"])
    elif kind in ("attention", "attention_bwd"):
        s["q"] = _heads(d, c, c["Hq"], c["Tq"], dt)
        s["k"], s["v"] = (_heads(d, c, c["Hkv"], c["Tk"], dt) for _ in range(2))
        s["mask"] = _mask(d, c)
        s["opts"] = dict(causal=c["mask"] == "causal", mask=s["mask"], layout=c["layout"])
        if kind == "attention_bwd":
            s["dout"] = _heads(d, c, c["Hq"], c["Tq"], dt)
            if c["residuals"]:
                s["lse"] = torch.empty(c["B"] * c["Hq"] * c["Tq"], device="cuda")
                s["out"] = native.sdpa(s["q"], s["k"], s["v"], lse=s["lse"], **s["opts"])
    elif kind == "dense":
        a = math.sqrt(6.0 / (c["K"] + c["N"]))
        s["x"] = d.normal(c["M"], c["K"], dtype=dt)
        s["w"] = d.uniform(c["K"], c["N"], lo=-a, hi=a, dtype=dt)
        s["dy"] = d.normal(c["M"], c["N"], dtype=dt)
    else:
        s["tensors"] = _transformer_inputs(c, d)
        s["exe"] = _client().compile(_transformer_text(c))
        s["bufs"] = [_client().buffer_view(t) for t in s["tensors"]]
    return s


# ---- one pass ------------------------------------------------------------------

def run(state):
    s, c = state, state["case"]
    kind = c["kind"]
    if kind == "norm":
        if c["op"] == "layer":
            return native.layer_norm(s["x"], s["gamma"], s["beta"], eps=1e-5)
        return native.rms_norm(s["x"], s["gamma"], eps=1e-6)
    if kind == "softmax":
        return native.log_softmax(s["x"])
    if kind == "norm_bwd":
        return native.layer_norm_bwd(s["x"], s["dy"], s["gamma"], eps=1e-5)
    if kind == "attention":
        return native.sdpa(s["q"], s["k"], s["v"], **s["opts"])
    if kind == "decode":
        return native.sdpa(s["q"], s["k"], s["v"], mask=s["mask"], q_rms_eps=1e-6, q_rms_weight=s["weight"])
    if kind == "attention_bwd":
        return native.sdpa_bwd(s["q"], s["k"], s["v"], s["dout"], fwd_out=s.get("out"), fwd_lse=s.get("lse"),
                               **s["opts"])
    if kind == "dense":
        dt = s["x"].dtype
        return (native.gemm(s["x"], s["w"], out_dtype=dt),
                native.gemm(s["dy"], s["w"], trans_b=True, out_dtype=dt),
                native.gemm(s["x"], s["dy"], trans_a=True, out_dtype=torch.float32))
    return torch.as_tensor(_DeviceArray(s["exe"].execute(s["bufs"], wait=False)[0], (c["B"], c["T"], c["d"])),
                           device="cuda")


# ---- what a pass cannot do without ---------------------------------------------

def work(case):
    c = case
    kind, e = c["kind"], SIZE[c.get("dtype", "f32")]
    if kind in ("norm", "softmax"):
        return {"bytes": 2 * c["rows"] * c["n"] * e + 2 * c["n"] * e, "flops": 8 * c["rows"] * c["n"]}
    if kind == "norm_bwd":
        return {"bytes": 3 * c["rows"] * c["n"] * e + 3 * c["n"] * e, "flops": 16 * c["rows"] * c["n"]}
    if kind == "decode":
        keys = c["B"] * c["Tk"] * 9 / 16  # mean visible length
        return {"bytes": 2 * keys * c["Hkv"] * c["D"] * e + 2 * c["B"] * c["Hq"] * c["D"] * e + 4 * c["B"] * c["Tk"],
                "flops": 4 * keys * c["Hq"] * c["D"]}
    if kind in ("attention", "attention_bwd"):
        Tq, Tk = c["Tq"], c["Tk"]
        pairs = Tq * Tk
        if c["mask"] == "causal":
            pairs = Tq * (Tq + 1) / 2
        elif c["mask"] == "band":
            w = max(1, Tk // 4)
            pairs = Tq * w - w * (w - 1) / 2
        elif c["mask"] == "padding":
            pairs = Tq * Tk * 0.75
        q, kv = c["B"] * c["Hq"] * Tq * c["D"], c["B"] * c["Hkv"] * Tk * c["D"]
        mask = {"padding": 4 * c["B"] * Tk, "bias": c["Hq"] * Tq * Tk * e, "band": 4 * Tq * Tk}.get(c["mask"], 0)
        if kind == "attention":
            return {"bytes": (2 * q + 2 * kv) * e + mask, "flops": 4 * c["B"] * c["Hq"] * pairs * c["D"]}
        extra = q * e + 4 * c["B"] * c["Hq"] * Tq if c["residuals"] else 0
        return {"bytes": (3 * q + 4 * kv) * e + mask + extra, "flops": 10 * c["B"] * c["Hq"] * pairs * c["D"]}
    if kind == "dense":
        M, K, N = c["M"], c["K"], c["N"]
        return {"bytes": (3 * M * K + 2 * K * N + 3 * M * N - M * N) * e + 4 * K * N, "flops": 6 * M * K * N}
    tok, dm, mlp = c["B"] * c["T"], c["d"], c["mlp"]
    pairs = c["T"] * (c["T"] + 1) / 2 if c["causal"] else c["T"] * c["T"]
    per = 2 * tok * dm * 4 * dm + 4 * tok * dm * mlp + 4 * c["B"] * pairs * dm
    return {"bytes": 4 * (2 * tok * dm + c["layers"] * (4 * dm * dm + 2 * dm * mlp + 9 * dm + mlp)),
            "flops": c["layers"] * per}


def tolerance(case):
    """About four times what each path differs from its value in 64 bits."""
    dt = case.get("dtype", "f32")
    kind = case["kind"]
    if dt != "f32":
        # Outputs rounded to 16 bits; probabilities and dS in 16 bits inside attention.
        return {"rel": {"bf16": 1.0e-2, "f16": 1.5e-3}[dt]}
    return {"rel": {"norm": 5e-7, "softmax": 5e-7, "norm_bwd": 2e-6, "attention": 3e-6, "attention_bwd": 6e-6,
                    "dense": 3e-6, "transformer": 6e-6}[kind]}


# ---- 64-bit values -------------------------------------------------------------

def exact(case, seed):
    c, s = case, prepare(case, seed)
    kind = c["kind"]
    f = lambda t: t.double()  # noqa: E731
    if kind in ("norm", "softmax", "norm_bwd"):
        return _exact_rows(c, s)
    if kind == "decode":
        q = f(s["q"])
        q = q * torch.rsqrt((q * q).mean(-1, keepdim=True) + 1e-6) * f(s["weight"])
        return _exact_attention(q, f(s["k"]), f(s["v"]), f(s["mask"]), False)
    if kind in ("attention", "attention_bwd"):
        bhtd = lambda t: f(t if c["layout"] == "bhtd" else t.transpose(1, 2)).contiguous()  # noqa: E731
        back = lambda t: t if c["layout"] == "bhtd" else t.transpose(1, 2)  # noqa: E731
        q, k, v = bhtd(s["q"]), bhtd(s["k"]), bhtd(s["v"])
        m = None if s["mask"] is None else f(s["mask"])
        if kind == "attention":
            return back(_exact_attention(q, k, v, m, c["mask"] == "causal"))
        return tuple(back(t) for t in _exact_attention(q, k, v, m, c["mask"] == "causal", bhtd(s["dout"])))
    if kind == "dense":
        x, w, dy = f(s["x"]), f(s["w"]), f(s["dy"])
        return x @ w, dy @ w.t().contiguous(), x.t().contiguous() @ dy
    return _exact_transformer(c, [f(t) for t in s["tensors"]])


def _exact_rows(c, s):
    n, parts = c["n"], []
    dg = db = 0.0
    for lo in range(0, c["rows"], max(1, (1 << 26) // n)):
        x = s["x"][lo:lo + max(1, (1 << 26) // n)].double()
        if c["kind"] == "softmax":
            parts.append(torch.log_softmax(x, -1))
            continue
        g = s["gamma"].double()
        if c["kind"] == "norm" and c["op"] == "rms":
            parts.append(x * torch.rsqrt((x * x).mean(-1, keepdim=True) + 1e-6) * g)
            continue
        xc = x - x.mean(-1, keepdim=True)
        r = torch.rsqrt((xc * xc).mean(-1, keepdim=True) + 1e-5)
        if c["kind"] == "norm":
            parts.append(xc * r * g + s["beta"].double())
            continue
        dy = s["dy"][lo:lo + x.shape[0]].double()
        xh, dxh = xc * r, dy * g
        parts.append((dxh - dxh.mean(-1, keepdim=True) - xh * (dxh * xh).mean(-1, keepdim=True)) * r)
        dg, db = dg + (dy * xh).sum(0), db + dy.sum(0)
    out = torch.cat(parts)
    return (out, dg, db) if c["kind"] == "norm_bwd" else out


def _exact_attention(q, k, v, mask, causal, dout=None):
    """softmax(q k^T / sqrt(D) + mask) v over [B, H, T, D] in 64 bits, or with
    dout its (dq, dk, dv); a few heads at a time."""
    B, Hq, Tq, D = q.shape
    Hkv, Tk = k.shape[1], k.shape[2]
    g = Hq // Hkv
    out = torch.empty_like(q)
    dk, dv = torch.zeros_like(k), torch.zeros_like(v)
    for b in range(B):
        for h in range(Hkv):
            hs = slice(h * g, (h + 1) * g)
            S = (q[b, hs].reshape(-1, D) @ k[b, h].t().contiguous()).view(g, Tq, Tk) / math.sqrt(D)
            if mask is not None:
                mb = mask[b if mask.shape[0] > 1 else 0]
                S += mb[hs] if mb.shape[0] > 1 else mb
            if causal:
                S.masked_fill_(torch.ones(Tq, Tk, dtype=torch.bool, device="cuda").triu_(1), -math.inf)
            P = torch.softmax(S, -1)
            o = (P.view(-1, Tk) @ v[b, h]).view(g, Tq, D)
            if dout is None:
                out[b, hs] = o
                continue
            do = dout[b, hs]
            dP = (do.reshape(-1, D) @ v[b, h].t().contiguous()).view(g, Tq, Tk)
            dS = P * (dP - (do * o).sum(-1, keepdim=True)) / math.sqrt(D)
            out[b, hs] = (dS.view(-1, Tk) @ k[b, h]).view(g, Tq, D)
            dk[b, h] = dS.view(-1, Tk).t().contiguous() @ q[b, hs].reshape(-1, D)
            dv[b, h] = P.view(-1, Tk).t().contiguous() @ do.reshape(-1, D)
    return out if dout is None else (out, dk, dv)


# ---- the transformer through PJRT ----------------------------------------------

_CLIENT = None


def _client():
    """The process's PJRT client: a program keeps one."""
    global _CLIENT
    if _CLIENT is None:
        _CLIENT = pjrt.Client()
    return _CLIENT


class _DeviceArray:
    """An output buffer's device memory, for torch (f32, dense row-major)."""

    def __init__(self, buf, shape):
        self.buf = buf
        self.__cuda_array_interface__ = {"shape": shape, "typestr": "<f4", "version": 2, "strides": None,
                                         "data": (buf.device_pointer(), False)}


def _transformer_inputs(c, d):
    """x and, per layer: ln1 scale / bias, qkv w / b, out w / b, ln2 scale /
    bias, mlp-in w / b, mlp-out w / b (Xavier-uniform matrices)."""
    dm, mlp = c["d"], c["mlp"]

    def xavier(fi, fo):
        a = math.sqrt(6.0 / (fi + fo))
        return d.uniform(fi, fo, lo=-a, hi=a)

    def small(n, mean=0.0):
        return d.normal(n, std=0.02, mean=mean)

    out = [d.normal(c["B"], c["T"], dm)]
    for _ in range(c["layers"]):
        out += [small(dm, 1.0), small(dm), xavier(dm, 3 * dm), small(3 * dm), xavier(dm, dm), small(dm),
                small(dm, 1.0), small(dm), xavier(dm, mlp), small(mlp), xavier(mlp, dm), small(dm)]
    return out


def _exact_transformer(c, t):
    B, T, dm, H = c["B"], c["T"], c["d"], c["heads"]

    def ln(x, g, b):
        xc = x - x.mean(-1, keepdim=True)
        return xc * torch.rsqrt((xc * xc).mean(-1, keepdim=True) + 1e-5) * g + b

    x = t[0].reshape(B * T, dm)
    for i in range(c["layers"]):
        g1, b1, wqkv, bqkv, wo, bo, g2, b2, w1, bm1, w2, bm2 = t[1 + 12 * i:13 + 12 * i]
        q, k, v = ((ln(x, g1, b1) @ wqkv + bqkv).view(B, T, 3, H, dm // H).permute(2, 0, 3, 1, 4).contiguous())
        o = _exact_attention(q, k, v, None, c["causal"])
        x = x + o.transpose(1, 2).reshape(B * T, dm) @ wo + bo
        u = ln(x, g2, b2) @ w1 + bm1
        x = x + 0.5 * u * (1 + torch.tanh(math.sqrt(2 / math.pi) * (u + 0.044715 * u ** 3))) @ w2 + bm2
    return x.view(B, T, dm)


class _Hlo:
    """Writes the body of one StableHLO function; a value is (name, shape, type)."""

    def __init__(self):
        self.lines = []

    @staticmethod
    def ty(shape, dt="f32"):
        return "tensor<" + "".join(f"{n}x" for n in shape) + dt + ">"

    def put(self, text, shape, dt="f32"):
        v = f"%{len(self.lines)}"
        self.lines.append(f"    {v} = stablehlo.{text}")
        return v, tuple(shape), dt

    def const(self, lit, dt="f32"):
        return self.put(f"constant dense<{lit}> : {self.ty((), dt)}", (), dt)

    def bcast(self, a, dims, shape):
        return self.put(f"broadcast_in_dim {a[0]}, dims = [{', '.join(map(str, dims))}] : "
                        f"({self.ty(a[1], a[2])}) -> {self.ty(shape, a[2])}", shape, a[2])

    def fill(self, x, shape):
        return self.bcast(self.const(x if isinstance(x, str) else f"{x:.8E}"), [], shape)

    def op(self, name, *a):
        return self.put(f"{name} {', '.join(v[0] for v in a)} : {self.ty(a[0][1], a[0][2])}", a[0][1], a[0][2])

    def reduce(self, a, kind):
        """Over the last axis, kept as size 1."""
        init = self.const("0xFF800000" if kind == "maximum" else "0.0")
        last = len(a[1]) - 1
        r = self.put(f"reduce({a[0]} init: {init[0]}) applies stablehlo.{kind} across dimensions = [{last}] : "
                     f"({self.ty(a[1])}, {self.ty(())}) -> {self.ty(a[1][:-1])}", a[1][:-1])
        return self.bcast(r, range(last), a[1][:-1] + (1,))

    def wide(self, a, shape):
        return self.bcast(a, range(len(shape)), shape)

    def mean(self, a):
        s = self.reduce(a, "add")
        return self.op("divide", s, self.fill(float(a[1][-1]), s[1]))

    def dot(self, a, b, batch, contract, shape):
        bt = f"batching_dims = [{', '.join(map(str, batch[0]))}] x [{', '.join(map(str, batch[1]))}], " if batch[0] else ""
        return self.put(f"dot_general {a[0]}, {b[0]}, {bt}contracting_dims = [{contract[0]}] x [{contract[1]}], "
                        f"precision = [DEFAULT, DEFAULT] : ({self.ty(a[1])}, {self.ty(b[1])}) -> {self.ty(shape)}", shape)

    def move(self, name, a, shape, more=""):
        return self.put(f"{name} {a[0]}{more} : ({self.ty(a[1])}) -> {self.ty(shape)}", shape)

    def layer_norm(self, x, g, b):
        last = [len(x[1]) - 1]
        xc = self.op("subtract", x, self.wide(self.mean(x), x[1]))
        var = self.mean(self.op("multiply", xc, xc))
        inv = self.op("rsqrt", self.op("add", var, self.fill(1e-5, var[1])))
        y = self.op("multiply", xc, self.wide(inv, x[1]))
        y = self.op("multiply", y, self.bcast(g, last, x[1]))
        return self.op("add", y, self.bcast(b, last, x[1]))

    def softmax(self, s):
        m = self.reduce(s, "maximum")
        e = self.op("exponential", self.op("subtract", s, self.wide(m, s[1])))
        return self.op("divide", e, self.wide(self.reduce(e, "add"), s[1]))

    def dense(self, x, w, b):
        shape = x[1][:-1] + (w[1][1],)
        y = self.dot(x, w, ([], []), (len(shape) - 1, 0), shape)
        return self.op("add", y, self.bcast(b, [len(shape) - 1], shape))


def _transformer_text(c):
    B, T, dm, H, mlp = c["B"], c["T"], c["d"], c["heads"], c["mlp"]
    hd = dm // H
    shapes = [(B, T, dm)]
    for _ in range(c["layers"]):
        shapes += [(dm,), (dm,), (dm, 3 * dm), (3 * dm,), (dm, dm), (dm,), (dm,), (dm,), (dm, mlp), (mlp,), (mlp, dm), (dm,)]
    args = [(f"%arg{i}", s, "f32") for i, s in enumerate(shapes)]
    f, x = _Hlo(), args[0]
    for i in range(c["layers"]):
        g1, b1, wqkv, bqkv, wo, bo, g2, b2, w1, bm1, w2, bm2 = args[1 + 12 * i:13 + 12 * i]
        qkv = f.dense(f.layer_norm(x, g1, b1), wqkv, bqkv)
        q, k, v = (f.move("reshape", f.move("slice", qkv, (B, T, dm), f" [0:{B}, 0:{T}, {j * dm}:{(j + 1) * dm}]"),
                          (B, T, H, hd)) for j in range(3))
        s = f.dot(q, k, ([0, 2], [0, 2]), (3, 3), (B, H, T, T))
        s = f.op("multiply", s, f.fill(1.0 / math.sqrt(hd), s[1]))
        if c["causal"]:
            at = [f.put(f"iota dim = {n} : {f.ty((T, T), 'i32')}", (T, T), "i32") for n in (0, 1)]
            pred = f.put(f"compare GE, {at[0][0]}, {at[1][0]}, SIGNED : ({f.ty((T, T), 'i32')}, {f.ty((T, T), 'i32')}) -> "
                         f"{f.ty((T, T), 'i1')}", (T, T), "i1")
            pred = f.bcast(pred, [2, 3], s[1])
            s = f.put(f"select {pred[0]}, {s[0]}, {f.fill('0xFF800000', s[1])[0]} : {f.ty(s[1], 'i1')}, {f.ty(s[1])}", s[1])
        o = f.dot(f.softmax(s), v, ([0, 1], [0, 2]), (3, 1), (B, H, T, hd))
        o = f.move("reshape", f.move("transpose", o, (B, T, H, hd), ", dims = [0, 2, 1, 3]"), (B, T, dm))
        x = f.op("add", x, f.dense(o, wo, bo))
        u = f.dense(f.layer_norm(x, g2, b2), w1, bm1)
        x3 = f.op("multiply", f.op("multiply", u, u), u)
        inner = f.op("add", u, f.op("multiply", f.fill(0.044715, u[1]), x3))
        t = f.op("tanh", f.op("multiply", f.fill(math.sqrt(2.0 / math.pi), u[1]), inner))
        u = f.op("multiply", f.op("multiply", f.fill(0.5, u[1]), u), f.op("add", f.fill(1.0, u[1]), t))
        x = f.op("add", x, f.dense(u, w2, bm2))
    ins = ", ".join(f"{n}: {f.ty(s)}" for n, s, _ in args)
    body = "\n".join(f.lines)
    return ("module @jit_transformer attributes {mhlo.num_partitions = 1 : i32, mhlo.num_replicas = 1 : i32} {\n"
            f"  func.func public @main({ins}) -> ({f.ty(x[1])} {{jax.result_info = \"result\"}}) {{\n{body}\n"
            f"    return {x[0]} : {f.ty(x[1])}\n  }}\n}}\n")
