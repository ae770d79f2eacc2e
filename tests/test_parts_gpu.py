"""Split calls of the chunked kernels (few, long sequences): every sequence is
cut into parts whose start states are composed from transfer states.

Split results are compared with the fp64 oracle at the chunk kernel's own
bounds (normwise 2e-2 for bf16 operands, as in tests/test_chunk_gpu.py) and
with the same call unsplit (no scratch), from which they differ only by the
rounding of the states: at most 1e-2 normwise, half the bound both meet.
"""

from __future__ import annotations

import ctypes

import numpy as np
import pytest
import torch

import flashrwkv_amd
from flashrwkv_amd import capi, workloads
from oracle import oracle
from tests import parity

pytestmark = pytest.mark.gpu

DEV = torch.device("cuda")
TOL, SAME = 2e-2, 1e-2
NAMES = ("r", "w", "k", "v", "a", "b")
CHUNK, RECURRENT, CALLER_CHUNKS = 0, 1, 2


@pytest.fixture(scope="module", autouse=True)
def _require_native():
    if flashrwkv_amd._C is None:
        pytest.fail("flashrwkv_amd native library is not built (no fallback exists)")


def _scratch(kernel, sequences, heads, total, longest):
    size = capi.library().frwkv_split_scratch_bytes(kernel, sequences, heads, 64, total, longest)
    assert size > 0, "the case is meant to split"
    # Filled with NaN: nothing of it may be read before it is written.
    return torch.full((max(size // 4, 1),), float("nan"), device=DEV), size


def _case(lengths, dtype, u_low=-5.0, heads=3):
    case = workloads.make_case(lengths=lengths, heads=heads, head_size=64, dtype=dtype, seed=31,
                               state_std=0.1, u_low=u_low, pool_slots=len(lengths) + 1,
                               slots=list(range(len(lengths)))[::-1])
    return case, {k: v.to(DEV) if isinstance(v, torch.Tensor) else v for k, v in case.items()}


# Chunk counts around the part boundaries (part lengths 1 and up, ragged last
# chunks and parts, sequences shorter than a part), every dtype and pool, and a
# decay that sends chunks through the sub-chunk path.
@pytest.mark.parametrize("lengths,dtype,pool_dtype,u_low", [
    ((257,), torch.bfloat16, torch.float32, -5.0),
    ((64 * 9,), torch.float16, torch.float32, -5.0),
    ((64 * 9 + 1, 1, 64, 300), torch.bfloat16, torch.bfloat16, -5.0),
    ((2111, 65), torch.bfloat16, torch.float32, -5.0),
    ((4100,), torch.float16, torch.bfloat16, -5.0),
    ((640, 70), torch.bfloat16, torch.float32, 3.0),
])
@pytest.mark.parametrize("kernel", (CHUNK, RECURRENT))
def test_split_packed_forward(kernel, lengths, dtype, pool_dtype, u_low):
    if kernel == RECURRENT and (dtype != torch.bfloat16 or pool_dtype != torch.float32):
        pytest.skip("the split-precision variant takes bf16 tokens and an fp32 pool")
    case, d = _case(lengths, dtype, u_low)
    n, h, _ = d["r"].shape
    if u_low > 0:  # strong decay: retentions down to 2^-20
        case["w"] = case["w"].float().clamp_min(2.0 ** -20).to(dtype)
        d["w"] = case["w"].to(DEV)
    lib = capi.library()
    status, cu, idx = capi.metadata_validate(d["cu_seqlens"], d["state_indices"], n,
                                             len(lengths) + 1)
    scratch, size = _scratch(kernel, len(lengths), h, n, max(lengths))
    out = []
    for split in (True, False):
        pool = d["state_pool"].to(pool_dtype, copy=True)
        y = torch.empty_like(d["v"])
        ptrs = [capi._p(x) for x in (cu, idx, status, pool, d["r"], d["w"], None, d["k"], d["v"],
                                     d["a"], d["b"], y)]
        tail = [0.75]
        area = [capi._p(scratch) if split else None, size if split else 0, capi._stream()]
        if kernel == CHUNK:
            rc = lib.frwkv_chunk_forward_split(
                capi.DTYPE[dtype], 1, capi.DTYPE[pool_dtype], len(lengths), h, 64, n,
                len(lengths) + 1, *ptrs, *tail, max(lengths), *area)
        else:
            rc = lib.frwkv_recurrent_forward_split(
                capi.DTYPE[dtype], 1, len(lengths), h, 64, n, max(lengths), len(lengths) + 1,
                *ptrs, *tail, *area)
        capi._check(rc)
        torch.cuda.synchronize()
        out.append((y, pool))
    pool0 = case["state_pool"].to(pool_dtype).double().numpy()
    y_ref, pool_ref = oracle.forward_varlen(
        *(case[x].double().numpy() for x in NAMES), pool0, case["cu_seqlens"].numpy(),
        case["state_indices"].numpy(), scale=0.75)
    (y, pool), (y1, pool1) = out
    parity.check("y", y, y_ref, TOL)
    parity.check("state", pool, pool_ref, TOL)
    parity.check("y against unsplit", y, y1.double().cpu(), SAME)
    parity.check("state against unsplit", pool, pool1.double().cpu(), SAME)
    assert torch.equal(pool[-1], d["state_pool"].to(pool_dtype)[-1])  # the slot of no sequence
