"""Similar and repeated keys, as a prompt of one repeated token has them: with a
rate near 1 the intra-chunk matrix L of every chunk kernel has entries near -1
all over, powers of L grow to binomials and only their sum, (I - L)^{-1}, stays
near 1. Bounds are those of the operators on independent keys: bf16 operands
2e-2 normwise (the split-precision state 2e-3), fp32 arithmetic 1e-6 for states
and 1e-5 for sums over a whole gradient.
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

import flashrwkv_amd
from oracle import oracle
from tests import parity

pytestmark = pytest.mark.gpu

DEV = torch.device("cuda")
NAMES = ("r", "w", "k", "v", "a", "b")
HEADS = 2
# Spread of the keys around one direction, and the rate.
KEYS = [(0.0, 1.0), (0.0, 0.9), (0.2, 1.0)]


@pytest.fixture(scope="module", autouse=True)
def _require_native():
    if flashrwkv_amd._C is None:
        pytest.fail("flashrwkv_amd native library is not built (no fallback exists)")


def _tokens(n, d, dtype, spread, rate):
    """Tokens with decay logits (slow decay, so that states reach far)."""
    g = torch.Generator().manual_seed(41)
    kk = torch.randn(1, HEADS, d, generator=g)
    kk = kk + spread * torch.randn(n, HEADS, d, generator=g)
    kk /= kk.norm(dim=-1, keepdim=True)
    tok = {x: torch.randn(n, HEADS, d, generator=g) for x in "rkv"}
    tok["w"] = torch.randn(n, HEADS, d, generator=g) - 6.0
    tok["a"], tok["b"] = -kk, rate * kk
    return {x: tok[x].to(dtype) for x in NAMES}


def _reference(tok):
    x64 = {x: t.double().numpy() for x, t in tok.items()}
    x64["w"] = oracle.retention_from_logits(x64["w"])
    return x64


# bf16 chunks (whole and cut into parts), the split-precision route (the same),
# and the fp32 matrix form.
@pytest.mark.parametrize("spread,rate", KEYS)
@pytest.mark.parametrize("entry,dtype,d,lengths,tol_y,tol_state", [
    ("chunk", torch.bfloat16, 64, (130, 70), 2e-2, 2e-2),
    ("chunk", torch.bfloat16, 64, (700,), 2e-2, 2e-2),
    ("recurrent", torch.bfloat16, 64, (130, 70), 2e-2, 2e-3),
    ("recurrent", torch.bfloat16, 64, (700,), 2e-2, 2e-3),
    ("recurrent", torch.float16, 64, (130, 70), 1e-3, 1e-6),
    ("recurrent", torch.float16, 128, (256,), 1e-3, 1e-6),
    ("recurrent", torch.bfloat16, 256, (130, 70), 4e-3, 1e-6),
])
def test_forward(entry, dtype, d, lengths, tol_y, tol_state, spread, rate):
    n = sum(lengths)
    tok = _tokens(n, d, dtype, spread, rate)
    cu = torch.tensor(np.concatenate([[0], np.cumsum(lengths)]), dtype=torch.int32)
    idx = torch.arange(len(lengths), dtype=torch.int32)
    pool = torch.randn(len(lengths), HEADS, d, d,
                       generator=torch.Generator().manual_seed(42)) * 0.1
    if entry == "chunk":  # its pool is bf16
        pool = pool.to(dtype)
    dev = [tok[x].to(DEV) for x in NAMES]
    dev_pool = pool.to(DEV)
    kw = dict(state_pool=dev_pool, cu_seqlens=cu.to(DEV), state_indices=idx.to(DEV))
    if entry == "chunk":
        y = flashrwkv_amd.infer_chunk_bf16_forward_varlen(*dev, chunk_size=64,
                                                          max_seqlen=max(lengths), **kw)
    else:
        y = flashrwkv_amd.infer_recurrent_fp32io16_forward_varlen(*dev, **kw)
    torch.cuda.synchronize()
    x64 = _reference(tok)
    y_ref, pool_ref = oracle.forward_varlen(*(x64[x] for x in NAMES), pool.double().numpy(),
                                            cu.numpy(), idx.numpy())
    parity.check("y", y, y_ref, tol_y)
    parity.check("state", dev_pool, pool_ref, tol_state)


@pytest.mark.parametrize("spread,rate", KEYS)
@pytest.mark.parametrize("d,lengths,dtype,tol,tol_state", [
    (64, (130, 70), torch.bfloat16, 2e-2, 2e-2),
    (64, (640,), torch.bfloat16, 2e-2, 2e-2),
    (128, (130, 70), torch.bfloat16, 2e-2, 2e-2),
    (256, (130, 70), torch.float16, 1e-3, 1e-6),
])
def test_training(d, lengths, dtype, tol, tol_state, spread, rate):
    n = sum(lengths)
    tok = _tokens(n, d, dtype, spread, rate)
    g = torch.Generator().manual_seed(43)
    starts, ends, offsets = [], [], [0]
    for begin, length in zip(np.cumsum((0, *lengths[:-1])).tolist(), lengths):
        cuts = list(range(begin, begin + length, 64))
        starts += cuts
        ends += cuts[1:] + [begin + length]
        offsets.append(len(starts))
    meta = [np.asarray(x, dtype=np.int32) for x in (offsets, starts, ends)]
    s0 = torch.randn(len(lengths), HEADS, d, d, generator=g) * 0.1
    dy = torch.randn(n, HEADS, d, generator=g).to(dtype)
    ds = torch.randn(s0.shape, generator=g) * 0.05
    leaves = [tok[x].to(DEV).requires_grad_() for x in NAMES]
    state = s0.to(DEV).requires_grad_()
    y, final, _, _ = flashrwkv_amd.statetune_recurrent_fp32io16(
        state, *(torch.from_numpy(x).to(DEV) for x in meta), *leaves)
    grads = torch.autograd.grad((y, final), [*leaves, state], (dy.to(DEV), ds.to(DEV)))
    torch.cuda.synchronize()
    x64 = _reference(tok)
    kw = dict(seg_offsets=meta[0], seg_starts=meta[1], seg_ends=meta[2],
              state_slots=np.arange(len(lengths), dtype=np.int32))
    args = [x64[x] for x in NAMES] + [s0.double().numpy()]
    y_ref, final_ref, _, _ = oracle.forward(*args, **kw, want_boundary=True,
                                            want_state_dot_a=True)
    ref = oracle.backward(*args, dy=dy.double().numpy(), dstate_final=ds.double().numpy(), **kw)
    logits = tok["w"].double().numpy()
    ref["dw"] = ref["dw"] * x64["w"] * oracle.retention_log_derivative(logits)
    parity.check("y", y, y_ref, tol)
    parity.check("final", final, final_ref, tol_state)
    for name, got in zip(NAMES, grads):
        # With one key, T^T dSA and T (At S + ..) are differences of neighbouring
        # rows: two roundings of 2^-9 of the rows where other gradients have one,
        # on a result smaller than either (measured up to 2.1e-2).
        parity.check("d" + name, got, ref["d" + name], 2 * tol if name in "ab" else tol)
    parity.check("dS0", grads[-1], ref["dstate0"], tol_state)
