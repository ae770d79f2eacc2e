"""Split calls of the chunked kernels (few, long sequences): every sequence is
cut into parts whose start states are composed from transfer states.

Split results are compared with the fp64 oracle at the chunk kernel's own
bounds (normwise 2e-2 for bf16 operands, as in tests/test_chunk_gpu.py) and
with the same call unsplit (no scratch), from which they differ only by the
rounding of the states: at most 1e-2 normwise, half the bound both meet. The
split-precision route's state has that route's own bound, 2e-3
(tests/test_recurrent_gpu.py), and half of it against unsplit.
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
TOL_STATE = 2e-3
NAMES = ("r", "w", "k", "v", "a", "b")
CHUNK, RECURRENT, CALLER_CHUNKS = 0, 1, 2


@pytest.fixture(scope="module", autouse=True)
def _require_native():
    if flashrwkv_amd._C is None:
        pytest.fail("flashrwkv_amd native library is not built (no fallback exists)")


def _scratch(kernel, io, sequences, heads, total, longest):
    size = capi.library().frwkv_split_scratch_bytes(kernel, io, 1, sequences, heads, 64, total,
                                                    longest)
    assert size > 0, "the case is meant to split"
    # Filled with NaN: nothing of it may be read before it is written.
    return torch.full((max(size // 4, 1),), float("nan"), device=DEV), size


MIXED = 9.0  # in place of u_low: _mixed_decay


def _mixed_decay(w):
    """Retention 1e-3 on 30% of the entries, about 190 log2 units per 64 tokens
    (such chunks run as sub-chunks) with the others as given, so that states
    still reach over sub-chunks."""
    weak = torch.rand(w.shape, generator=torch.Generator().manual_seed(19)) >= 0.3
    return torch.where(weak, w, torch.full_like(w, 1e-3))


def _case(lengths, dtype, u_low=-5.0, heads=3):
    case = workloads.make_case(lengths=lengths, heads=heads, head_size=64, dtype=dtype, seed=31,
                               state_std=0.1, u_low=-5.0 if u_low == MIXED else u_low,
                               pool_slots=len(lengths) + 1,
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
    ((640, 70), torch.bfloat16, torch.float32, MIXED),
    ((640, 70), torch.float16, torch.float32, MIXED),
    # Short sequences before, between and after long ones, more than one round
    # of the search for a part's sequence.
    ((1,) * 70 + (700,) + (2,) * 5 + (1400, 63), torch.bfloat16, torch.float32, -5.0),
    ((1900, 65) + (1,) * 140, torch.bfloat16, torch.bfloat16, -5.0),
])
@pytest.mark.parametrize("kernel", (CHUNK, RECURRENT))
def test_split_packed_forward(kernel, lengths, dtype, pool_dtype, u_low):
    if kernel == RECURRENT and (dtype != torch.bfloat16 or pool_dtype != torch.float32):
        pytest.skip("the split-precision variant takes bf16 tokens and an fp32 pool")
    case, d = _case(lengths, dtype, u_low)
    n, h, _ = d["r"].shape
    if u_low == MIXED:
        case["w"] = _mixed_decay(case["w"])
        d["w"] = case["w"].to(DEV)
    elif u_low > 0:  # strong decay: retentions down to 2^-20
        case["w"] = case["w"].float().clamp_min(2.0 ** -20).to(dtype)
        d["w"] = case["w"].to(DEV)
    lib = capi.library()
    status, cu, idx = capi.metadata_validate(d["cu_seqlens"], d["state_indices"], n,
                                             len(lengths) + 1)
    scratch, size = _scratch(kernel, capi.DTYPE[dtype], len(lengths), h, n, max(lengths))
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
    parity.check("state", pool, pool_ref, TOL_STATE if kernel == RECURRENT else TOL)
    parity.check("y against unsplit", y, y1.double().cpu(), SAME)
    parity.check("state against unsplit", pool, pool1.double().cpu(),
                 TOL_STATE / 2 if kernel == RECURRENT else SAME)
    assert torch.equal(pool[-1], d["state_pool"].to(pool_dtype)[-1])  # the slot of no sequence


# Tokens that leave the state alone (a, b, k and v zero, retention 1): every chunk
# maps S to S, so an fp32 state comes out of the parts bit for bit, as it does of
# the unsplit kernels, and so does the adjoint at the end in the backward.
@pytest.mark.parametrize("tokens", (640, 2304))
@pytest.mark.parametrize("kernel", (CHUNK, RECURRENT, "backward"))
def test_split_carries_the_state_in_fp32(kernel, tokens):
    heads, lib, io = 3, capi.library(), capi.DTYPE[torch.bfloat16]
    zero = torch.zeros((tokens, heads, 64), dtype=torch.bfloat16, device=DEV)
    one, y = torch.ones_like(zero), torch.empty_like(zero)
    state = torch.randn((1, heads, 64, 64), generator=torch.Generator().manual_seed(3)).to(DEV)
    cu, idx = (torch.tensor(x, dtype=torch.int32, device=DEV) for x in ([0, tokens], [0]))
    if kernel == "backward":
        chunks = tokens // 64
        ends = torch.arange(64, tokens + 1, 64, dtype=torch.int32, device=DEV)
        lists = torch.tensor([0, chunks], dtype=torch.int32, device=DEV)
        scratch, size = _scratch(4, io, 1, heads, chunks, tokens)
        boundary = torch.zeros((chunks, heads, 64, 64), device=DEV)
        work = capi.workspace(capi.statetune_backward_workspace_bytes(64, heads, tokens, False),
                              DEV)
        grads, got = [torch.empty_like(zero) for _ in range(6)], torch.empty_like(state)
        rc = lib.frwkv_statetune_backward_split(
            io, 1, 1, heads, 64, tokens, chunks,
            *(capi._p(x) for x in (lists, ends - 64, ends, boundary, None, zero, one, None, zero,
                                   zero, zero, zero, None, state, *grads, got, work)),
            work.numel(), 1.0, None, capi._p(scratch), size, capi._stream())
    else:
        status, cu, idx = capi.metadata_validate(cu, idx, tokens, 1)
        scratch, size = _scratch(kernel, io, 1, heads, tokens, tokens)
        got = state.clone()
        ptrs = [capi._p(x) for x in (cu, idx, status, got, zero, one, None, zero, zero, zero, zero,
                                     y)]
        area = (capi._p(scratch), size, capi._stream())
        if kernel == CHUNK:
            rc = lib.frwkv_chunk_forward_split(io, 1, capi.DTYPE[torch.float32], 1, heads, 64,
                                               tokens, 1, *ptrs, 1.0, tokens, *area)
        else:
            rc = lib.frwkv_recurrent_forward_split(io, 1, 1, heads, 64, tokens, tokens, 1, *ptrs,
                                                   1.0, *area)
    capi._check(rc)
    torch.cuda.synchronize()
    assert torch.equal(got, state)


# Repeated split calls are equal bit for bit: nothing depends on which workgroup
# comes first. Through the public entries, forward and backward.
@pytest.mark.parametrize("entry", ("recurrent", "chunk", "statetune", "pretrain"))
def test_split_calls_repeat_bitwise(entry):
    lengths, heads = (900, 610), 2
    case = workloads.make_case(lengths=lengths, heads=heads, head_size=64, dtype=torch.bfloat16,
                               seed=23, state_std=0.1)
    dev = {k: v.to(DEV) if isinstance(v, torch.Tensor) else v for k, v in case.items()}
    n = sum(lengths)

    def run():
        if entry in ("recurrent", "chunk"):
            pool = dev["state_pool"].to(torch.float32 if entry == "recurrent" else torch.bfloat16,
                                        copy=True)
            call = (flashrwkv_amd.infer_recurrent_fp32io16_forward_varlen if entry == "recurrent"
                    else flashrwkv_amd.infer_chunk_bf16_forward_varlen)
            out = call(*(dev[x] for x in NAMES), state_pool=pool, cu_seqlens=dev["cu_seqlens"],
                       state_indices=dev["state_indices"], max_seqlen=max(lengths))
            return [out[0] if isinstance(out, tuple) else out, pool]
        leaves = [dev[x].clone().requires_grad_() for x in NAMES]
        if entry == "pretrain":
            out = [flashrwkv_amd.pretrain_recurrent_bf16(
                *(x[:1504].reshape(2, 752, heads * 64) for x in leaves))]
        else:
            state = dev["state_pool"][:2].clone().requires_grad_()
            meta = oracle.chunk_metadata(lengths, 64)
            out = list(flashrwkv_amd.statetune_recurrent_fp32io16(
                state, *(torch.from_numpy(x).to(DEV) for x in meta[:3]), *leaves)[:2])
            leaves.append(state)
        return out + list(torch.autograd.grad([x.float().square().sum() for x in out], leaves))

    kernel = {"recurrent": RECURRENT, "chunk": CHUNK, "statetune": 4, "pretrain": 3}[entry]
    total, longest = {"statetune": (25, n), "pretrain": (1504, 752)}.get(entry, (n, max(lengths)))
    assert capi.library().frwkv_split_scratch_bytes(
        kernel, capi.DTYPE[torch.bfloat16], capi.DECAY_LOGITS, 2, heads, 64, total, longest) > 0
    first, second = run(), run()
    torch.cuda.synchronize()
    for x, y in zip(first, second, strict=True):
        assert torch.equal(x, y)


# Head sizes and lengths around the 16-token pieces of the fp32 matrix form,
# which the public entries take with fp16 tokens or wide heads (decay logits):
# one piece and a token, ragged, a sequence in the middle shorter than a piece.
# Expected against the oracle: the fp32 state as the per-token kernels (the
# sums' order alone differs, about 1e-6 normwise over these lengths), outputs
# at the io type's rounding (2^-9 bf16, 2^-11 fp16, of the largest entry).
@pytest.mark.parametrize("dtype,d,lengths", [
    (torch.float16, 64, (33,)),
    (torch.float16, 64, (1, 48, 7, 65, 16)),
    (torch.float16, 64, (40,) * 70 + (33, 1, 17)),  # two rounds of the slot search
    (torch.float16, 128, (40, 3)),
    (torch.bfloat16, 128, (32, 95)),
    (torch.float16, 256, (17, 50)),
    (torch.bfloat16, 256, (64,)),
])
def test_fp32_matrix_recurrence(dtype, d, lengths):
    heads = 2
    assert capi.library().frwkv_split_scratch_bytes(
        RECURRENT, capi.DTYPE[dtype], capi.DECAY_LOGITS, len(lengths), heads, d, sum(lengths),
        max(lengths)) > 0, "the case is meant to take the matrix form"
    case = workloads.make_case(lengths=lengths, heads=heads, head_size=d, dtype=dtype, seed=5,
                               state_std=0.1, pool_slots=len(lengths) + 1,
                               slots=list(range(len(lengths)))[::-1])
    gen = torch.Generator().manual_seed(6)
    logits = (torch.randn(case["r"].shape, generator=gen) * 3.0).to(dtype)
    bias = torch.randn((heads, d), generator=gen).to(dtype)
    dev = {k: v.to(DEV) if isinstance(v, torch.Tensor) else v for k, v in case.items()}
    y = flashrwkv_amd.infer_recurrent_fp32io16_forward_varlen(
        dev["r"], logits.to(DEV), dev["k"], dev["v"], dev["a"], dev["b"],
        state_pool=dev["state_pool"], cu_seqlens=dev["cu_seqlens"],
        state_indices=dev["state_indices"], scale=0.5, decay_bias=bias.to(DEV))
    torch.cuda.synchronize()
    w = oracle.retention_from_logits(logits.double().numpy(), bias.double().numpy())
    y_ref, pool_ref = oracle.forward_varlen(
        case["r"].double().numpy(), w, *(case[x].double().numpy() for x in "kvab"),
        case["state_pool"].double().numpy(), case["cu_seqlens"].numpy(),
        case["state_indices"].numpy(), scale=0.5)
    parity.check("y", y, y_ref, 4e-3 if dtype == torch.bfloat16 else 1e-3)
    parity.check("state", dev["state_pool"], pool_ref, 1e-5)


# Without room for the scratch a call runs as one without scratch does.
def test_no_room_for_scratch():
    n, heads = 4096, 32
    case = workloads.make_case(lengths=(n,), heads=heads, head_size=64, dtype=torch.float16,
                               seed=7, state_std=0.1)
    dev = {k: v.to(DEV) if isinstance(v, torch.Tensor) else v for k, v in case.items()}

    def run():
        pool = dev["state_pool"].clone()
        y = flashrwkv_amd.infer_recurrent_fp32io16_forward_varlen(
            *(dev[x] for x in NAMES), state_pool=pool, cu_seqlens=dev["cu_seqlens"],
            state_indices=dev["state_indices"])
        torch.cuda.synchronize()
        return y, pool

    before = flashrwkv_amd.tmix.wkv7.set_recurrent_long_route("per_token")
    try:
        want = run()
    finally:
        flashrwkv_amd.tmix.wkv7.set_recurrent_long_route(before)
    size = capi.library().frwkv_split_scratch_bytes(RECURRENT, capi.DTYPE[torch.float16],
                                                    capi.DECAY_LOGITS, 1, heads, 64, n, n)
    assert size > 128 << 20
    torch.cuda.empty_cache()
    total = torch.cuda.get_device_properties(DEV).total_memory
    torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved() + size // 2) / total)
    try:
        got = run()
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)
    for x, y in zip(got, want):
        assert torch.equal(x, y)


# Head size 256 training: caller chunks of one piece, of a piece and a token,
# longer ones and an empty one, and no upstream gradient of y or of the state.
@pytest.mark.parametrize("dtype", (torch.bfloat16, torch.float16))
@pytest.mark.parametrize("chunks,with_dy,with_ds", [
    ([[16, 17, 40], [1]], True, True),
    ([[33], [0, 64, 15]], True, False),
    ([[70]], False, True),
])
def test_fp32_matrix_training(dtype, chunks, with_dy, with_ds):
    heads, d = 2, 256
    ends = np.cumsum([c for seq in chunks for c in seq])
    starts = np.concatenate([[0], ends[:-1]])
    offsets = np.concatenate([[0], np.cumsum([len(seq) for seq in chunks])])
    meta = [np.asarray(x, dtype=np.int32) for x in (offsets, starts, ends)]
    n = int(ends[-1])
    case = workloads.make_case(lengths=(n,), heads=heads, head_size=d, dtype=dtype, seed=9,
                               state_std=0.1)
    gen = torch.Generator().manual_seed(10)
    tok = {x: case[x] for x in "rkvab"}
    tok["w"] = (torch.randn(case["r"].shape, generator=gen) * 3.0).to(dtype)
    s0 = torch.randn((len(chunks), heads, d, d), generator=gen) * 0.1
    dy = torch.randn(case["r"].shape, generator=gen).to(dtype)
    ds = torch.randn(s0.shape, generator=gen) * 0.05
    leaves = [tok[x].to(DEV).requires_grad_() for x in NAMES]
    state = s0.to(DEV).requires_grad_()
    y, final, boundary, sda = flashrwkv_amd.statetune_recurrent_fp32io16(
        state, *(torch.from_numpy(x).to(DEV) for x in meta), *leaves, scale=0.7)
    grads = torch.autograd.grad([t for t, on in ((y, with_dy), (final, with_ds)) if on],
                                [*leaves, state],
                                [t.to(DEV) for t, on in ((dy, with_dy), (ds, with_ds)) if on])
    torch.cuda.synchronize()
    x64 = {x: tok[x].double().numpy() for x in NAMES}
    logits = x64["w"]
    x64["w"] = oracle.retention_from_logits(logits)
    kw = dict(seg_offsets=meta[0], seg_starts=meta[1], seg_ends=meta[2],
              state_slots=np.arange(len(chunks), dtype=np.int32), scale=0.7)
    args = [x64[x] for x in NAMES] + [s0.double().numpy()]
    y_ref, final_ref, boundary_ref, sda_ref = oracle.forward(
        *args, **kw, want_boundary=True, want_state_dot_a=True)
    ref = oracle.backward(*args, dy=dy.double().numpy() * with_dy,
                          dstate_final=ds.double().numpy() * with_ds, **kw)
    ref["dw"] = ref["dw"] * x64["w"] * oracle.retention_log_derivative(logits)
    tol = 4e-3 if dtype == torch.bfloat16 else 1e-3
    parity.check("y", y, y_ref, tol)
    parity.check("final", final, final_ref, 1e-5)
    parity.check("boundary", boundary, boundary_ref, 1e-5)
    parity.check("state_dot_a", sda, sda_ref, 1e-5)
    for name, got in zip(NAMES, grads):
        parity.check("d" + name, got, ref["d" + name], tol)
    parity.check("dS0", grads[-1], ref["dstate0"], 1e-5)


# Chunks that overlap have more 16-token pieces than the matrix form has slots
# for: the final states, the boundaries, y of the last visit of a token and dS0
# (which depends on no state) are still those of the recurrence. Both sequences
# visit the same tokens, each four times, so y is checked with one sequence.
@pytest.mark.parametrize("sequences", (1, 2))
def test_fp32_matrix_training_overlapping_chunks(sequences):
    heads, d, n, visits = 2, 256, 64, 4
    case = workloads.make_case(lengths=(n,), heads=heads, head_size=d, dtype=torch.bfloat16,
                               seed=11, state_std=0.1)
    gen = torch.Generator().manual_seed(12)
    tok = {x: case[x] for x in NAMES}
    tok["w"] = torch.randn(case["r"].shape, generator=gen).to(torch.bfloat16)
    s0 = torch.randn((sequences, heads, d, d), generator=gen) * 0.1
    dy = torch.randn(case["r"].shape, generator=gen).to(torch.bfloat16)
    ds = torch.randn(s0.shape, generator=gen) * 0.05
    chunks = sequences * visits
    meta = [np.asarray(x, dtype=np.int32)
            for x in (range(0, chunks + 1, visits), [0] * chunks, [n] * chunks)]
    leaves = [tok[x].to(DEV).requires_grad_() for x in NAMES]
    state = s0.to(DEV).requires_grad_()
    y, final, boundary, _ = flashrwkv_amd.statetune_recurrent_fp32io16(
        state, *(torch.from_numpy(x).to(DEV) for x in meta), *leaves)
    grad = torch.autograd.grad((y, final), state, (dy.to(DEV), ds.to(DEV)))[0]
    torch.cuda.synchronize()
    x64 = {x: tok[x].double().numpy() for x in NAMES}
    x64["w"] = oracle.retention_from_logits(x64["w"])
    kw = dict(seg_offsets=meta[0], seg_starts=meta[1], seg_ends=meta[2],
              state_slots=np.arange(sequences, dtype=np.int32))
    args = [x64[x] for x in NAMES] + [s0.double().numpy()]
    y_ref, final_ref, boundary_ref, _ = oracle.forward(
        *args, **kw, want_boundary=True, want_state_dot_a=True)
    ref = oracle.backward(*args, dy=dy.double().numpy(), dstate_final=ds.double().numpy(), **kw)
    parity.check("final", final, final_ref, 1e-5)
    parity.check("boundary", boundary, boundary_ref, 1e-5)
    parity.check("dS0", grad, ref["dstate0"], 1e-5)
    if sequences == 1:
        parity.check("y", y, y_ref, 4e-3)


# Training at head size 64: caller chunks of whole, partial, several and no
# pieces, sequences shorter than the split and without chunks, a decay that
# sends pieces through the sub-piece path, no upstream gradient of y or of the
# state, and the dense pretraining layout (chunks None) with a ragged last piece.
@pytest.mark.parametrize("dtype", (torch.bfloat16, torch.float16))
@pytest.mark.parametrize("chunks,tokens,strong,with_dy,with_ds", [
    ([[64] * 12], 0, False, True, True),
    ([[64] * 9 + [17], [1], [], [33, 0, 64, 130, 15]], 0, False, True, False),
    ([[4] * 24 + [0, 0]], 0, False, False, True),
    ([[64] * 6 + [50]], 0, True, True, True),
    (None, 1040, False, True, False),
    (None, 192, False, True, False),
    (None, 400, True, True, False),
])
def test_split_training_backward(dtype, chunks, tokens, strong, with_dy, with_ds):
    heads, scale = 2, 0.75 if chunks else 1.0
    lens = [sum(seq) for seq in chunks] if chunks else [tokens] * 2
    n = sum(lens)
    case = workloads.make_case(lengths=[n], heads=heads, head_size=64, dtype=dtype, seed=17,
                               state_std=0.1, u_low=-5.0)
    tok = {x: case[x] for x in NAMES}
    if strong:
        tok["w"] = _mixed_decay(tok["w"])
    pieces = chunks or [[16] * (tokens // 16)] * 2
    ends = np.cumsum([c for seq in pieces for c in seq])
    starts = np.concatenate([[0], ends[:-1]])
    offsets = np.concatenate([[0], np.cumsum([len(seq) for seq in pieces])])
    meta = [np.asarray(x, dtype=np.int32) for x in (offsets, starts, ends)]
    gen = torch.Generator().manual_seed(18)
    s0 = torch.randn((len(lens), heads, 64, 64), generator=gen) * (0.1 if chunks else 0.0)
    dy = torch.randn(tok["r"].shape, generator=gen).to(dtype)
    ds = torch.randn(s0.shape, generator=gen) * 0.05
    kw = dict(seg_offsets=meta[0], seg_starts=meta[1], seg_ends=meta[2],
              state_slots=np.arange(len(lens), dtype=np.int32), scale=scale)
    args = [tok[x].double().numpy() for x in NAMES] + [s0.double().numpy()]
    _, _, boundary, _ = oracle.forward(*args, **kw, want_boundary=True, want_state_dot_a=True)
    ref = oracle.backward(*args, dy=dy.double().numpy() * with_dy,
                          dstate_final=ds.double().numpy() * with_ds, **kw)
    boundary = torch.from_numpy(boundary).float().to(DEV)
    if not chunks:  # [B, H, T / 16, D, D]
        boundary = boundary.view(2, tokens // 16, heads, 64, 64).transpose(1, 2).contiguous()

    lib, io = capi.library(), capi.DTYPE[dtype]
    dev = [tok[x].to(DEV) for x in NAMES]
    dev_meta = [torch.from_numpy(x).to(DEV) for x in meta]
    upstream = [dy.to(DEV) if with_dy else None, ds.to(DEV) if with_ds else None]
    scratch, size = _scratch(4 if chunks else 3, io, len(lens), heads,
                             meta[1].size if chunks else n, n if chunks else tokens)
    work = capi.workspace(capi.statetune_backward_workspace_bytes(64, heads, n, False), DEV)
    results = []
    for split in (True, False):
        grads = [torch.empty_like(x) for x in dev]
        ds0 = torch.empty_like(s0, device=DEV)
        area = [None, capi._p(scratch) if split else None, size if split else 0, capi._stream()]
        grad_ptrs = [capi._p(g) for g in grads]
        if chunks:
            rc = lib.frwkv_statetune_backward_split(
                io, 1, len(lens), heads, 64, n, meta[1].size, *(capi._p(x) for x in dev_meta),
                capi._p(boundary), None, *(capi._p(x) for x in (*dev[:2], None, *dev[2:])),
                *(capi._p(x) for x in upstream), *grad_ptrs, capi._p(ds0), capi._p(work),
                work.numel(), scale, *area)
        else:
            rc = lib.frwkv_pretrain_backward_split(
                io, 1, 2, tokens, heads, 64, *(capi._p(x) for x in dev), capi._p(upstream[0]),
                capi._p(boundary), *grad_ptrs, None, 0, *area)
        capi._check(rc)
        torch.cuda.synchronize()
        results.append(grads + ([ds0] if chunks else []))
    names = ["d" + x for x in NAMES] + ["dstate0"]
    for name, got, unsplit in zip(names, *results):
        parity.check(name, got, ref[name], TOL)
        # dw = dlg / w: at a retention of 1e-3 the roundings of dlg, which
        # differ between the two, are a thousand times larger. Each is within
        # TOL of the oracle, so they are within 2 TOL of each other.
        same = 2 * TOL if strong and name == "dw" else SAME
        parity.check(name + " against unsplit", got, unsplit.double().cpu(), same)
        parity.check(name + " unsplit", unsplit, ref[name], TOL)
