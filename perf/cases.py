"""Performance cases of the WKV7 operators: what they are, how one pass of
each runs through the public entry points, and what it should return.

``listed()`` gives the fixed cases and ``draw(rng)`` more of the same ranges;
``prepare`` makes a case's inputs on the GPU, ``run`` does one pass,
``work`` counts the bytes and operations a pass cannot do without, and
``exact`` is the same result in fp64 by plain torch.

Token distributions are those of ``flashrwkv_amd.workloads``: r, k, v ~
N(0, 1), a = -kk, b = kk g with a unit kk per head and g = sigmoid(N(0, 1)).
The operators take decay logits x (retention exp(-e^{-1/2} sigmoid(x))), drawn
over the range a trained model has: a per-channel base in [-6, 1] plus
token-dependent noise.
"""

from __future__ import annotations

import math
import random

import torch

import flashrwkv_amd
from flashrwkv_amd.rl_infctx.wkv7 import rl_infctx_chunk_fp32io16
from flashrwkv_amd.tmix.gates import (
    infer_tmix_kk_a_gate_forward_varlen,
    infer_tmix_lnx_rkvres_xg_forward_varlen,
)
from flashrwkv_amd.tmix.lnx_rkvres_xg.pretrain import pretrain_tmix_lnx_rkvres_xg_bf16
from flashrwkv_amd.tmix.wkv7.fused import infer_tmix_wkv7_fused_forward_varlen

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16}
SPARE_SLOTS = 3  # state pools hold a few sequences that a call does not touch
EPS = 64.0e-5    # the TMix output norm


# ------------------------------------------------------------------- cases
def listed() -> list[dict]:
    return [
        # One user generating: a single token through one layer. Latency.
        dict(name="decode-one", kind="decode", batch=1, heads=32, head_size=64, dtype="bf16"),
        # The serving batch of benchmark config 1, the largest decode step.
        dict(name="decode-batch", kind="decode", batch=256, heads=40, head_size=64,
             dtype="bf16"),
        # Serving with the fp16 state pool: a mid-size batch, the step and its
        # phase advance.
        dict(name="decode-fp16-state", kind="decode_fp16", batch=61, heads=40, head_size=64),
        # The layer's producer, recurrence and consumer as one operator.
        dict(name="decode-fused", kind="decode_fused", batch=96, heads=32, dtype="fp16"),
        # An fp16 model reading a ragged batch of short prompts: the three
        # operators of the layer, one after the other.
        dict(name="layer-prompts", kind="layer", batch=9, low=17, high=384, heads=32,
             head_size=64),
        # One bf16 prompt through the fp32-state operator (the default route
        # of a chat request).
        dict(name="prompt-one", kind="prompt", batch=1, low=1531, high=1531, heads=32),
        # Benchmark config 3's ragged prefill batch: the largest forward.
        dict(name="prefill-batch", kind="prefill", batch=64, low=128, high=4096, heads=32,
             bias=False),
        # A few long documents, ragged, with a decay bias.
        dict(name="prefill-few", kind="prefill", batch=3, low=500, high=3000, heads=40,
             bias=True),
        # Benchmark config 4: training at full size, forward and backward.
        dict(name="statetune-batch", kind="statetune", batch=8, low=4096, high=4096, heads=64,
             head_size=64, dtype="bf16"),
        # State tuning on a couple of short documents, fp16, ragged.
        dict(name="statetune-few", kind="statetune", batch=2, low=400, high=1100, heads=32,
             head_size=64, dtype="fp16"),
        # The reference benchmark's pretraining shape: the layer's recurrence and
        # its output norm, each forward and backward on its own inputs.
        dict(name="pretrain-block", kind="pretrain", batch=2, tokens=512, heads=12,
             head_size=64),
        # Pretraining with wide heads.
        dict(name="pretrain-wide-head", kind="pretrain", batch=2, tokens=512, heads=8,
             head_size=256),
    ]


def _log_int(rng: random.Random, low: int, high: int) -> int:
    return max(low, min(high, round(math.exp(rng.uniform(math.log(low), math.log(high))))))


def draw(rng: random.Random) -> dict:
    kind = rng.choice(["decode", "decode", "decode_fp16", "decode_fused", "layer", "prompt",
                       "prompt", "prefill", "prefill", "rl", "statetune", "statetune",
                       "pretrain", "pretrain"])
    heads = rng.choice([12, 16, 24, 32, 40])
    head_size = rng.choice([64, 64, 64, 128, 256])
    if kind == "decode":
        wide = 1 if head_size == 64 else 4 if head_size == 128 else 16
        return dict(kind=kind, batch=_log_int(rng, 1, 256 // wide), heads=heads,
                    head_size=head_size, dtype=rng.choice(["bf16", "fp16"]))
    if kind == "decode_fp16":
        return dict(kind=kind, batch=_log_int(rng, 1, 256), heads=heads, head_size=64)
    if kind == "decode_fused":
        return dict(kind=kind, batch=_log_int(rng, 1, 256), heads=heads,
                    dtype=rng.choice(["bf16", "fp16"]))
    if kind == "layer":
        low = _log_int(rng, 2, 64)
        return dict(kind=kind, batch=_log_int(rng, 1, 32), low=low,
                    high=low + _log_int(rng, 1, 500), heads=heads, head_size=64)
    if kind in ("prompt", "prefill", "rl"):
        low = _log_int(rng, 64, 1500)
        case = dict(kind=kind, batch=_log_int(rng, 1, 16), low=low,
                    high=low + _log_int(rng, 1, 2500), heads=heads)
        if kind == "prefill":
            case["bias"] = rng.choice([False, True])
        if kind == "rl":
            case["dtype"] = rng.choice(["bf16", "fp16"])
        return case
    if kind == "statetune":
        wide = head_size // 64
        low = _log_int(rng, 60, 1500 // wide)
        return dict(kind=kind, batch=_log_int(rng, 1, 8 // wide), low=low,
                    high=low + _log_int(rng, 1, 2000 // wide), heads=heads // wide,
                    head_size=head_size, dtype=rng.choice(["bf16", "fp16"]))
    wide = head_size // 64
    return dict(kind=kind, batch=_log_int(rng, 1, 8 // wide),
                tokens=16 * _log_int(rng, 4, 128 // wide), heads=heads // wide,
                head_size=head_size)


def _lengths(case: dict) -> list[int]:
    """The case's sequence lengths: a fixed ragged batch in [low, high]."""
    if "low" not in case:
        return [case.get("tokens", 1)] * case["batch"]
    rng = random.Random(f"{case['batch']}.{case['low']}.{case['high']}")
    return [rng.randint(case["low"], case["high"]) for _ in range(case["batch"])]


def _shape(case: dict) -> tuple[int, int, int]:
    """Total tokens, heads, head size."""
    return sum(_lengths(case)), case["heads"], case.get("head_size", 64)


# ------------------------------------------------------------------ inputs
class _Maker:
    """Seeded random tensors on the GPU."""

    def __init__(self, seed: int):
        self.dev = torch.device("cuda")
        self.gen = torch.Generator(device=self.dev).manual_seed(seed)

    def normal(self, *shape, scale=1.0, mean=0.0, dtype=torch.float32):
        x = torch.randn(shape, generator=self.gen, device=self.dev)
        return x.mul_(scale).add_(mean).to(dtype)

    def uniform(self, *shape, low=0.0, high=1.0, dtype=torch.float32):
        x = torch.rand(shape, generator=self.gen, device=self.dev)
        return x.mul_(high - low).add_(low).to(dtype)

    def logits(self, *shape, dtype):
        base = self.uniform(*shape[-2:], low=-6.0, high=1.0)
        return self.normal(*shape, scale=0.7).add_(base).to(dtype)

    def tokens(self, *shape, dtype):
        """r, decay logits, k, v, a, b."""
        r, k, v = (self.normal(*shape, dtype=dtype) for _ in range(3))
        kk = self.normal(*shape)
        kk /= kk.norm(dim=-1, keepdim=True)
        gate = torch.sigmoid(self.normal(*shape))
        return dict(r=r, w=self.logits(*shape, dtype=dtype), k=k, v=v, a=(-kk).to(dtype),
                    b=(kk * gate).to(dtype))


def _metadata(case: dict, seed: int, dev, ticket=True) -> dict:
    lengths = _lengths(case)
    offsets = [0]
    for n in lengths:
        offsets.append(offsets[-1] + n)
    slots = list(range(len(lengths) + SPARE_SLOTS))
    random.Random(seed).shuffle(slots)
    s = dict(cu=torch.tensor(offsets, dtype=torch.int32, device=dev),
             idx=torch.tensor(slots[:len(lengths)], dtype=torch.int32, device=dev),
             max_len=max(lengths), total=offsets[-1])
    if ticket:  # a serving loop validates a batch's metadata once
        s["ticket"] = flashrwkv_amd.prepare_recurrent_metadata(
            s["cu"], s["idx"], total_tokens=s["total"], state_pool_size=len(slots),
            max_seqlen=s["max_len"])
    return s


def _gate_vectors(m: _Maker, c: int, dtype) -> dict:
    return dict(k_k=m.normal(c, scale=0.3, mean=1.0, dtype=dtype),
                a0=m.normal(c, scale=0.5, dtype=dtype), k_a=m.uniform(c, dtype=dtype),
                r_k=m.normal(c, scale=0.5, dtype=dtype),
                ln_w=m.normal(c, scale=0.2, mean=1.0, dtype=dtype),
                ln_b=m.normal(c, scale=0.1, dtype=dtype))


def prepare(case: dict, seed: int) -> dict:
    kind = case["kind"]
    n, h, d = _shape(case)
    m = _Maker(seed)
    dtype = DTYPES[case.get("dtype", "bf16" if kind in ("prompt", "prefill", "pretrain")
                            else "fp16")]
    s = dict(case=case)
    if kind == "pretrain":
        b, t, c = case["batch"], case["tokens"], h * d
        tok = m.tokens(b, t, h, d, dtype=dtype)
        s["tok"] = {x: v.view(b, t, c).requires_grad_() for x, v in tok.items()}
        s["vec"] = dict(residual_scale=m.normal(h, d, scale=0.1, dtype=dtype),
                        weight=m.normal(c, scale=0.2, mean=1.0, dtype=dtype),
                        bias=m.normal(c, scale=0.1, dtype=dtype))
        s["vec"] = {x: v.requires_grad_() for x, v in s["vec"].items()}
        s["x"] = m.normal(b, t, c, dtype=dtype).requires_grad_()
        s["g"] = torch.sigmoid(m.normal(b, t, c)).to(dtype).requires_grad_()
        s["dy"], s["dout"] = (m.normal(b, t, c, dtype=dtype) for _ in range(2))
        return s
    s.update(_metadata(case, seed, m.dev, ticket=kind not in ("statetune", "rl")))
    slots = case["batch"] + SPARE_SLOTS
    if kind == "statetune":
        starts, ends, offsets = [], [], [0]
        begin = 0
        for length in _lengths(case):
            cuts = list(range(begin, begin + length, 64))
            starts += cuts
            ends += cuts[1:] + [begin + length]
            begin += length
            offsets.append(len(starts))
        s["meta"] = [torch.tensor(x, dtype=torch.int32, device=m.dev)
                     for x in (offsets, starts, ends)]
        s["tok"] = {x: v.requires_grad_() for x, v in m.tokens(n, h, d, dtype=dtype).items()}
        s["state"] = m.normal(case["batch"], h, d, d, scale=0.1).requires_grad_()
        s["dy"] = m.normal(n, h, d, dtype=dtype)
        s["ds"] = m.normal(case["batch"], h, d, d, scale=0.01)
        return s
    pool_dtype = {"decode_fp16": torch.float16, "prefill": torch.bfloat16}.get(
        kind, torch.float32)
    s["pool"] = m.normal(slots, h, d, d, scale=0.1, dtype=pool_dtype)
    if kind in ("layer", "decode_fused"):
        s["tok"] = dict(r=m.normal(n, h, d, dtype=dtype), w=m.logits(n, h, d, dtype=dtype),
                        k=m.normal(n, h, d, dtype=dtype), v=m.normal(n, h, d, dtype=dtype),
                        a12=m.normal(n, h, d, dtype=dtype),
                        g=torch.sigmoid(m.normal(n, h, d)).to(dtype))
        s["vec"] = _gate_vectors(m, h * d, dtype)
        return s
    s["tok"] = m.tokens(n, h, d, dtype=dtype)
    if kind == "decode_fp16":
        s["elapsed"] = torch.arange(slots, dtype=torch.int32, device=m.dev) * 37
    if kind == "prefill":
        s["bias"] = m.normal(h, d, scale=0.3, dtype=dtype) if case["bias"] else None
    return s


# --------------------------------------------------------------- one pass
_ORDER = ("r", "w", "k", "v", "a", "b")


def run(s: dict):
    case, tok = s["case"], s["tok"]
    kind = case["kind"]
    if kind == "pretrain":
        h, d = case["heads"], case["head_size"]
        y = flashrwkv_amd.pretrain_recurrent_bf16(*(tok[x] for x in _ORDER), head_size=d)
        grads = torch.autograd.grad(y, [tok[x] for x in _ORDER], s["dy"])
        leaves = [s["x"], tok["r"], tok["k"], tok["v"], *s["vec"].values(), s["g"]]
        out = pretrain_tmix_lnx_rkvres_xg_bf16(*leaves, head_size=d)
        return [y.detach(), out.detach(), *grads,
                *torch.autograd.grad(out, leaves, s["dout"])]
    if kind == "statetune":
        y, final, boundary, sda = flashrwkv_amd.statetune_recurrent_fp32io16(
            s["state"], *s["meta"], *(tok[x] for x in _ORDER))
        grads = torch.autograd.grad((y, final), [tok[x] for x in _ORDER] + [s["state"]],
                                    (s["dy"], s["ds"]))
        return [y.detach(), final.detach(), boundary, sda, *grads]
    if kind == "rl":
        return list(rl_infctx_chunk_fp32io16(
            *(tok[x] for x in _ORDER), state_pool=s["pool"], cu_seqlens=s["cu"],
            state_indices=s["idx"], chunk_size=64))
    common = dict(state_pool=s["pool"], cu_seqlens=s["cu"], state_indices=s["idx"],
                  validated_metadata=s["ticket"])
    if kind == "decode_fp16":
        y = flashrwkv_amd.infer_recurrent_fp16_forward_varlen(
            *(tok[x] for x in _ORDER), elapsed_state_pool=s["elapsed"], **common)
        flashrwkv_amd.infer_recurrent_fp16_advance_i32_varlen(
            s["elapsed"], s["cu"], s["idx"], total_tokens=s["total"],
            validated_metadata=s["ticket"])
        return [y, s["pool"], s["elapsed"]]
    if kind == "decode_fused":
        vec = s["vec"]
        y = infer_tmix_wkv7_fused_forward_varlen(
            *(tok[x] for x in ("r", "w", "k", "v", "a12", "g")), vec["k_k"], vec["a0"],
            vec["k_a"], vec["r_k"], vec["ln_w"], vec["ln_b"], **common)
        return [y, s["pool"]]
    if kind == "layer":
        vec, (n, h, d) = s["vec"], _shape(case)
        flat = {x: t.view(n, h * d) for x, t in tok.items()}
        hints = dict(head_size=d, batch_size=case["batch"], max_seqlen=s["max_len"])
        k, a, b = infer_tmix_kk_a_gate_forward_varlen(flat["k"], vec["k_k"], vec["a0"],
                                                      flat["a12"], vec["k_a"], **hints)
        y = flashrwkv_amd.infer_recurrent_fp32io16_forward_varlen(
            tok["r"], tok["w"], k.view(n, h, d), tok["v"], a.view(n, h, d), b.view(n, h, d),
            **common)
        out = infer_tmix_lnx_rkvres_xg_forward_varlen(
            y.view(n, h * d), flat["r"], k, flat["v"], vec["r_k"], vec["ln_w"], vec["ln_b"],
            flat["g"], **hints)
        return [out, y, s["pool"]]
    if kind == "prefill":
        y = flashrwkv_amd.infer_chunk_bf16_forward_varlen(
            *(tok[x] for x in _ORDER), chunk_size=64, max_seqlen=s["max_len"],
            decay_bias=s["bias"], **common)
        return [y, s["pool"]]
    y = flashrwkv_amd.infer_recurrent_fp32io16_forward_varlen(*(tok[x] for x in _ORDER),
                                                              **common)
    return [y, s["pool"]]


def work(case: dict) -> dict:
    """Each input read once, each output written once; 8 D^2 operations per
    token and head for the recurrence, three times that with the backward."""
    kind, lengths = case["kind"], _lengths(case)
    n, h, d = _shape(case)
    row, tokens = h * d, n
    state = case["batch"] * h * d * d
    flops = 8.0 * tokens * h * d * d
    if kind == "decode_fp16":
        return dict(bytes=2 * 2 * state + 7 * 2 * tokens * row, flops=flops)
    if kind == "decode_fused":
        return dict(bytes=2 * 4 * state + 7 * 2 * tokens * row + 6 * 2 * row, flops=flops)
    if kind == "layer":  # r, w, k, v, a12, g in; y and the layer's output out
        return dict(bytes=2 * 4 * state + 8 * 2 * tokens * row + 6 * 2 * row, flops=flops)
    if kind == "prefill":
        return dict(bytes=2 * 2 * state + 7 * 2 * tokens * row, flops=flops)
    if kind == "rl":  # the whole pool is copied
        pool = (case["batch"] + SPARE_SLOTS) * h * d * d
        return dict(bytes=2 * 4 * pool + 7 * 2 * tokens * row, flops=flops)
    if kind == "pretrain":  # 6 + 5 tokens, dy, dout in; y, out and 6 + 5 gradients out
        return dict(bytes=26 * 2 * tokens * row + 6 * 2 * row, flops=3 * flops)
    if kind == "statetune":  # tokens, dy, S0, dS in; y, S, boundary, a^T S, gradients out
        chunks = sum(-(-x // 64) for x in lengths)
        return dict(bytes=14 * 2 * tokens * row + 4 * tokens * row + 4 * chunks * h * d * d
                    + 4 * 4 * state, flops=3 * flops)
    return dict(bytes=2 * 4 * state + 7 * 2 * tokens * row, flops=flops)


def tolerance(case: dict) -> dict:
    """About four times the error against ``exact`` that each path was measured
    to have (2-norm): 5.5e-3 for the gradients, 3.6e-3 for bf16 products, 2.1e-3
    and 1.7e-3 for bf16 outputs of wider sums, 2e-4 to 3e-4 for fp16 outputs."""
    kind = case["kind"]
    if kind in ("statetune", "pretrain"):
        return dict(rel=2.2e-2)
    if kind in ("prefill", "rl"):
        return dict(rel=1.45e-2)
    if kind == "prompt":
        return dict(rel=8.4e-3)
    if kind == "decode_fp16":  # the pool's own fp16 steps are part of the contract
        return dict(rel=1.2e-3)
    if case.get("dtype", "fp16") == "fp16":
        return dict(rel=1e-3, **({"max": 0.25} if kind in ("layer", "decode_fused") else {}))
    return dict(rel=6.8e-3)


# ------------------------------------------------------------------- exact
def _retention(x: torch.Tensor) -> torch.Tensor:
    return torch.exp(-math.exp(-0.5) * torch.sigmoid(x))


def _steps(S, r, w, k, v, a, b):
    """The recurrence over [B, T, H, D] tokens from S [B, H, K, V]."""
    ys, sas = [], []
    for t in range(r.shape[1]):
        sa = (S * a[:, t, :, :, None]).sum(-2)
        S = S * w[:, t, :, :, None] + b[:, t, :, :, None] * sa[..., None, :] \
            + k[:, t, :, :, None] * v[:, t, :, None, :]
        ys.append((S * r[:, t, :, :, None]).sum(-2))
        sas.append(sa)
    return torch.stack(ys, 1), S, torch.stack(sas, 1)


_BLOCK = 64


class _Padded:
    """A ragged packed batch as [B, T, ...], padded with tokens that leave the
    state as it is (w = 1, the rest 0)."""

    def __init__(self, lengths, dev):
        self.lengths, self.longest = lengths, max(lengths)
        starts = torch.tensor([sum(lengths[:i]) for i in range(len(lengths))], device=dev)
        t = torch.arange(self.longest, device=dev)
        self.inside = t[None] < torch.tensor(lengths, device=dev)[:, None]
        self.index = torch.where(self.inside, starts[:, None] + t[None], 0)

    def pad(self, x, fill=0.0):
        return x[self.index].masked_fill(~self.inside[..., None, None], fill)

    def pack(self, x):
        return x[self.inside]


def _forward(p: _Padded, tok: dict, S):
    """y, final state, a^T S (padded) and the state at every 64th token."""
    ys, sas, saved = [], [], []
    x = [p.pad(tok[n], 1.0 if n == "w" else 0.0) for n in _ORDER]
    with torch.no_grad():
        for t in range(0, p.longest, _BLOCK):
            saved.append(S)
            y, S, sa = _steps(S, *(q[:, t:t + _BLOCK] for q in x))
            ys.append(y)
            sas.append(sa)
    return torch.cat(ys, 1), S, torch.cat(sas, 1), saved, x


def _backward(p: _Padded, x, saved, dy, dS):
    """Gradients of the padded tokens (dw with respect to w) and of S0."""
    grads = [torch.zeros_like(q) for q in x]
    dy = p.pad(dy)
    for i in reversed(range(len(saved))):
        cut = slice(i * _BLOCK, (i + 1) * _BLOCK)
        leaves = [saved[i].detach().requires_grad_()] + [q[:, cut].detach().requires_grad_()
                                                         for q in x]
        with torch.enable_grad():
            y, S, _ = _steps(*leaves)
            got = torch.autograd.grad((y, S), leaves, (dy[:, cut], dS))
        dS = got[0]
        for g, q in zip(grads, got[1:]):
            g[:, cut] = q
    return grads, dS


def _logit_gradient(dw, w, x):
    sig = torch.sigmoid(x)
    return dw * w * (-math.exp(-0.5)) * sig * (1.0 - sig)


def _lnx(x, r, k, v, r_k, weight, bias, g, h, d):
    shape = x.shape[:-1] + (h, d)
    x, r, k, v = (t.reshape(shape) for t in (x, r, k, v))
    mean = x.mean(-1, keepdim=True)
    var = ((x - mean) ** 2).mean(-1, keepdim=True)
    rkv = (r * k * r_k.reshape(h, d)).sum(-1, keepdim=True)
    out = (x - mean) / torch.sqrt(var + EPS) * weight.reshape(h, d) + bias.reshape(h, d) + rkv * v
    return out.reshape(g.shape) * g


def _gates(k, k_k, a0, a12, k_a, h, d):
    """new_k, -kk, kk gate of [N, H, D] keys."""
    u = k * k_k.reshape(h, d)
    kk = u / u.norm(dim=-1, keepdim=True).clamp_min(1e-12)
    gate = torch.sigmoid(a0.reshape(h, d) + a12)
    ka = k_a.reshape(h, d)
    return k * (gate * ka + 1.0 - ka), -kk, kk * gate


def exact(case: dict, seed: int):
    s = prepare(case, seed)
    kind = case["kind"]
    n, h, d = _shape(case)
    f64 = {x: t.detach().double() for x, t in s["tok"].items()}
    p = _Padded(_lengths(case), next(iter(f64.values())).device)
    vec = {x: t.detach().double() for x, t in s.get("vec", {}).items()}
    if kind == "pretrain":
        shape = s["g"].shape
        logits = f64["w"].reshape(n, h, d)
        tok = {x: t.reshape(n, h, d) for x, t in f64.items()}
        tok["w"] = _retention(logits)
        zero = torch.zeros(case["batch"], h, d, d, dtype=torch.float64, device=logits.device)
        y, _, _, saved, x = _forward(p, tok, zero)
        grads, _ = _backward(p, x, saved, s["dy"].double().reshape(n, h, d), zero)
        grads = [p.pack(g).reshape(shape) for g in grads]
        grads[1] = _logit_gradient(grads[1], tok["w"].reshape(shape), f64["w"])
        leaves = [s["x"].detach().double(), f64["r"], f64["k"], f64["v"], *vec.values(),
                  s["g"].detach().double()]
        leaves = [t.detach().requires_grad_() for t in leaves]
        with torch.enable_grad():
            out = _lnx(*leaves, h, d)
            more = torch.autograd.grad(out, leaves, s["dout"].double())
        return [p.pack(y).reshape(shape), out.detach(), *grads, *more]
    if kind == "statetune":
        logits = f64["w"]
        f64["w"] = _retention(logits)
        y, final, sda, saved, x = _forward(p, f64, s["state"].detach().double())
        boundary = torch.cat([torch.stack(saved[:-(-length // 64)])[:, i]
                              for i, length in enumerate(p.lengths)])
        grads, dS = _backward(p, x, saved, s["dy"].double(), s["ds"].double())
        grads = [p.pack(g) for g in grads]
        grads[1] = _logit_gradient(grads[1], f64["w"], logits)
        return [p.pack(y), final, boundary, p.pack(sda), *grads, dS]
    pool = s["pool"].double()
    idx = s["idx"].long()
    if s.get("bias") is not None:
        f64["w"] = f64["w"] + s["bias"].double()
    f64["w"] = _retention(f64["w"])
    if kind in ("layer", "decode_fused"):
        raw_k = f64["k"]
        f64["k"], f64["a"], f64["b"] = _gates(raw_k, vec["k_k"], vec["a0"], f64["a12"],
                                              vec["k_a"], h, d)
        if kind == "layer":  # the producer's tensors are fp16
            for x in ("k", "a", "b"):
                f64[x] = f64[x].half().double()
    y, final, *_ = _forward(p, f64, pool[idx])
    y = p.pack(y)
    pool = pool.index_copy(0, idx, final)
    if kind == "decode_fp16":
        return [y, pool, None]
    if kind in ("layer", "decode_fused"):
        x = y.half().double() if kind == "layer" else y
        out = _lnx(x.reshape(n, h * d), *(f64[t].reshape(n, h * d) for t in ("r", "k", "v")),
                   vec["r_k"], vec["ln_w"], vec["ln_b"], f64["g"].reshape(n, h * d), h, d)
        return [out, y, pool] if kind == "layer" else [out.reshape(n, h, d), pool]
    return [y, pool]
