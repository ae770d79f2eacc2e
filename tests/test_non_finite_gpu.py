"""An infinity or NaN in one token reaches that token and later ones only (in
the backward: that token and earlier ones, from dy), in the columns and heads
that the recurrence couples, on the calls of the fp32 matrix form too, whose
matrix products would spread it over 16 tokens: finite and non-finite entries
are those of the fp64 oracle, and the finite ones are as close to it as ever.
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

import flashrwkv_amd
from flashrwkv_amd import workloads
from oracle import oracle
from tests import parity

pytestmark = pytest.mark.gpu

DEV = torch.device("cuda")
NAMES = ("r", "w", "k", "v", "a", "b")
NAN, INF = float("nan"), float("inf")


@pytest.fixture(scope="module", autouse=True)
def _require_native():
    if flashrwkv_amd._C is None:
        pytest.fail("flashrwkv_amd native library is not built (no fallback exists)")


def _check(name, got, ref, tol):
    got, ref = parity.as_f64(got), parity.as_f64(ref)
    assert np.array_equal(np.isfinite(got), np.isfinite(ref)), name
    ok = np.isfinite(ref)
    assert ok.any(), name
    parity.check(name, got[ok], ref[ok], tol)


def _tokens(n, heads, d, dtype, seed):
    case = workloads.make_case(lengths=(n,), heads=heads, head_size=d, dtype=dtype, seed=seed,
                               state_std=0.1)
    g = torch.Generator().manual_seed(seed)
    tok = {x: case[x].clone() for x in NAMES}
    tok["w"] = (torch.randn(tok["r"].shape, generator=g) * 2.0).to(dtype)
    return tok, g


def _reference(tok):
    x64 = {x: t.double().numpy() for x, t in tok.items()}
    x64["w"] = oracle.retention_from_logits(x64["w"])
    return x64


# The token is in the middle of a piece of the second sequence, once in its last
# piece, which is short.
@pytest.mark.parametrize("dtype,d", [(torch.float16, 64), (torch.bfloat16, 128),
                                     (torch.float16, 256)])
@pytest.mark.parametrize("where,value,token", [
    ("v", NAN, 45), ("v", INF, 107), ("k", INF, 45), ("a", NAN, 45), ("b", INF, 45),
    ("r", NAN, 45), ("w", NAN, 45), ("w", INF, 45), ("w", -INF, 45),
])
def test_forward(dtype, d, where, value, token):
    lengths, heads = (40, 70, 33), 2
    tok, g = _tokens(sum(lengths), heads, d, dtype, 51)
    tok[where][token, 1, 3] = value
    cu = torch.tensor([0, 40, 110, 143], dtype=torch.int32)
    idx = torch.tensor([2, 0, 1], dtype=torch.int32)
    pool = torch.randn(4, heads, d, d, generator=g) * 0.1
    dev_pool = pool.to(DEV)
    y = flashrwkv_amd.infer_recurrent_fp32io16_forward_varlen(
        *(tok[x].to(DEV) for x in NAMES), state_pool=dev_pool, cu_seqlens=cu.to(DEV),
        state_indices=idx.to(DEV), scale=0.5)
    torch.cuda.synchronize()
    with np.errstate(all="ignore"):
        x64 = _reference(tok)
        y_ref, pool_ref = oracle.forward_varlen(*(x64[x] for x in NAMES), pool.double().numpy(),
                                                cu.numpy(), idx.numpy(), scale=0.5)
    if where != "w" or np.isnan(value):
        assert not np.isfinite(y_ref).all() and np.isfinite(y_ref[:token]).all()
    _check("y", y, y_ref, 4e-3 if dtype == torch.bfloat16 else 1e-3)
    _check("state", dev_pool, pool_ref, 1e-5)


@pytest.mark.parametrize("where,value,token", [
    ("v", NAN, 45), ("k", INF, 45), ("a", NAN, 50), ("b", NAN, 45), ("r", INF, 45),
    ("w", NAN, 45), ("dy", NAN, 45), ("dy", INF, 3),
])
def test_training_wide_head(where, value, token):
    heads, d, dtype = 2, 256, torch.bfloat16
    meta = [np.asarray(x, dtype=np.int32)
            for x in ((0, 3, 4), (0, 16, 33, 73), (16, 33, 73, 103))]
    tok, g = _tokens(103, heads, d, dtype, 52)
    s0 = torch.randn(2, heads, d, d, generator=g) * 0.1
    dy = torch.randn(tok["r"].shape, generator=g).to(dtype)
    ds = torch.randn(s0.shape, generator=g) * 0.05
    ({**tok, "dy": dy})[where][token, 1, 3] = value
    leaves = [tok[x].to(DEV).requires_grad_() for x in NAMES]
    state = s0.to(DEV).requires_grad_()
    y, final, boundary, sda = flashrwkv_amd.statetune_recurrent_fp32io16(
        state, *(torch.from_numpy(x).to(DEV) for x in meta), *leaves, scale=0.7)
    grads = torch.autograd.grad((y, final), [*leaves, state], (dy.to(DEV), ds.to(DEV)))
    torch.cuda.synchronize()
    with np.errstate(all="ignore"):
        x64 = _reference(tok)
        kw = dict(seg_offsets=meta[0], seg_starts=meta[1], seg_ends=meta[2],
                  state_slots=np.arange(2, dtype=np.int32), scale=0.7)
        args = [x64[x] for x in NAMES] + [s0.double().numpy()]
        y_ref, final_ref, boundary_ref, sda_ref = oracle.forward(
            *args, **kw, want_boundary=True, want_state_dot_a=True)
        ref = oracle.backward(*args, dy=dy.double().numpy(), dstate_final=ds.double().numpy(),
                              **kw)
        logits = tok["w"].double().numpy()
        ref["dw"] = ref["dw"] * x64["w"] * oracle.retention_log_derivative(logits)
    for name, got, want, tol in (("y", y, y_ref, 4e-3), ("final", final, final_ref, 1e-5),
                                 ("boundary", boundary, boundary_ref, 1e-5),
                                 ("state_dot_a", sda, sda_ref, 1e-5)):
        _check(name, got, want, tol)
    for name, got in zip(NAMES, grads):
        _check("d" + name, got, ref["d" + name], 4e-3)
    _check("dS0", grads[-1], ref["dstate0"], 1e-5)


# Pretraining: the same backward in the dense layout.
@pytest.mark.parametrize("where,value", [("v", NAN), ("a", INF), ("dy", NAN)])
def test_pretraining_wide_head(where, value):
    batch, tokens, heads, d, dtype = 2, 48, 2, 256, torch.bfloat16
    tok, g = _tokens(batch * tokens, heads, d, dtype, 53)
    dy = torch.randn(tok["r"].shape, generator=g).to(dtype)
    ({**tok, "dy": dy})[where][tokens + 21, 1, 3] = value
    dense = (batch, tokens, heads * d)
    leaves = [tok[x].view(dense).to(DEV).requires_grad_() for x in NAMES]
    y = flashrwkv_amd.pretrain_recurrent_bf16(*leaves, head_size=d)
    grads = torch.autograd.grad(y, leaves, dy.view(dense).to(DEV))
    torch.cuda.synchronize()
    starts = np.arange(0, batch * tokens, 16, dtype=np.int32)
    with np.errstate(all="ignore"):
        x64 = _reference(tok)
        kw = dict(seg_offsets=np.asarray((0, 3, 6), dtype=np.int32), seg_starts=starts,
                  seg_ends=starts + 16, state_slots=np.arange(2, dtype=np.int32), scale=1.0)
        args = [x64[x] for x in NAMES] + [np.zeros((batch, heads, d, d))]
        y_ref = oracle.forward(*args, **kw, want_boundary=True, want_state_dot_a=True)[0]
        ref = oracle.backward(*args, dy=dy.double().numpy(),
                              dstate_final=np.zeros((batch, heads, d, d)), **kw)
        logits = tok["w"].double().numpy()
        ref["dw"] = ref["dw"] * x64["w"] * oracle.retention_log_derivative(logits)
    _check("y", y.view(-1, heads, d), y_ref, 4e-3)
    for name, got in zip(NAMES, grads):
        _check("d" + name, got.view(-1, heads, d), ref["d" + name], 4e-3)
