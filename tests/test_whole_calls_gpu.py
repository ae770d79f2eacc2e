"""The native whole calls of the decode chain and of pretraining against the
contract tables: every form of a call has the same outcome on both, the same
result or an error of the same type and text."""

import sys
import threading
import time

import pytest
import torch
from torch.overrides import TorchFunctionMode
from torch.utils._python_dispatch import TorchDispatchMode

from flashrwkv_amd.tmix import wkv7
from flashrwkv_amd.tmix.wkv7 import pretrain

pytestmark = pytest.mark.gpu
DEV = "cuda"


class Wrapped(torch.Tensor):
    """A subclass, which the whole calls leave to the tables."""


def _tokens(dtype, tokens=5, heads=2, d=64):
    g = torch.Generator().manual_seed(3)
    return [(torch.randn(tokens, heads, d, generator=g) * 0.2).to(DEV, dtype) for _ in range(6)]


def _metadata():
    cu = torch.tensor([0, 1, 5], dtype=torch.int32, device=DEV)
    slots = torch.tensor([2, 0], dtype=torch.int32, device=DEV)
    return cu, slots, wkv7.prepare_recurrent_metadata(
        cu, slots, total_tokens=5, state_pool_size=3)


def _strided(x):
    return torch.cat([x, x], -1)[..., :x.shape[-1]]


FORMS = {
    "as given": lambda c: c,
    "no ticket": lambda c: {**c, "validated_metadata": None},
    "a ticket of another type": lambda c: {**c, "validated_metadata": object()},
    "longest 4": lambda c: {**c, "max_seqlen": 4},
    "longest 0": lambda c: {**c, "max_seqlen": 0},
    "longest -3": lambda c: {**c, "max_seqlen": -3},
    "longest 5": lambda c: {**c, "max_seqlen": 5},
    "longest True": lambda c: {**c, "max_seqlen": True},
    "longest 4.0": lambda c: {**c, "max_seqlen": 4.0},
    "longest 2^80": lambda c: {**c, "max_seqlen": 1 << 80},
    "scale 2": lambda c: {**c, "scale": 2},
    "scale as text": lambda c: {**c, "scale": "2"},
    "scale as a tensor": lambda c: {**c, "scale": torch.tensor(0.5)},
    "bias": lambda c: {**c, "decay_bias": c["r"][0].clone()},
    "bias of another size": lambda c: {**c, "decay_bias": c["r"][0, :, :7].clone()},
    "bias no tensor": lambda c: {**c, "decay_bias": 1.0},
    "r no tensor": lambda c: {**c, "r": [1.0]},
    "r of two dimensions": lambda c: {**c, "r": c["r"][0]},
    "k strided": lambda c: {**c, "k": _strided(c["k"])},
    "v of another size": lambda c: {**c, "v": c["v"][:4]},
    "v empty": lambda c: {**c, "v": c["v"][:0]},
    "a double": lambda c: {**c, "a": c["a"].double()},
    "b on the host": lambda c: {**c, "b": c["b"].cpu()},
    "b a subclass": lambda c: {**c, "b": c["b"].as_subclass(Wrapped)},
    "k a parameter": lambda c: {**c, "k": torch.nn.Parameter(c["k"])},
    "pool strided": lambda c: {**c, "state_pool": _strided(c["state_pool"])},
    "pool of another type": lambda c: {**c, "state_pool": c["state_pool"].bfloat16()},
    "pool on the host": lambda c: {**c, "state_pool": c["state_pool"].cpu()},
    "pool of no dimension": lambda c: {**c, "state_pool": c["state_pool"].sum()},
    "offsets of 64 bits": lambda c: {**c, "cu_seqlens": c["cu_seqlens"].long()},
    "offsets of two dimensions": lambda c: {**c, "cu_seqlens": c["cu_seqlens"][None]},
    "offsets of one sequence": lambda c: {**c, "cu_seqlens": c["cu_seqlens"][:2]},
    "slots no tensor": lambda c: {**c, "state_indices": [2, 0]},
    "slots of 64 bits": lambda c: {**c, "state_indices": c["state_indices"].long()},
    "phases of 64 bits": lambda c: {**c, "elapsed_state_pool": c["elapsed_state_pool"].long()},
    "phases on the host": lambda c: {**c, "elapsed_state_pool": c["elapsed_state_pool"].cpu()},
    "phases too few": lambda c: {**c, "elapsed_state_pool": c["elapsed_state_pool"][:2]},
    "total 4": lambda c: {**c, "total_tokens": 4},
    "total True": lambda c: {**c, "total_tokens": True},
    "total 0": lambda c: {**c, "total_tokens": 0},
    "8 tokens": lambda c: {**{n: c[n][:, :8] for n in "rwkvab"}, "head_size": c["head_size"]},
    "head size 128": lambda c: {**c, "head_size": 128},
    "head size 32": lambda c: {**c, "head_size": 32},
    "head size 64.0": lambda c: {**c, "head_size": 64.0},
}


def _call(which):
    cu, slots, ticket = _metadata()
    pool = torch.arange(3 * 2 * 64 * 64, device=DEV).view(3, 2, 64, 64).remainder(13).div(50)
    if which == "fp32":
        r, w, k, v, a, b = _tokens(torch.bfloat16)
        return wkv7.infer_recurrent_fp32io16_forward_varlen, dict(
            r=r, decay_logits=w, k=k, v=v, a=a, b=b, state_pool=pool, cu_seqlens=cu,
            state_indices=slots, validated_metadata=ticket)
    if which == "fp16":
        r, w, k, v, a, b = _tokens(torch.float16)
        return wkv7.infer_recurrent_fp16_forward_varlen, dict(
            r=r, decay_logits=w, k=k, v=v, a=a, b=b, state_pool=pool.half(),
            elapsed_state_pool=torch.zeros(3, dtype=torch.int32, device=DEV), cu_seqlens=cu,
            state_indices=slots, validated_metadata=ticket)
    if which == "advance":
        return wkv7.infer_recurrent_fp16_advance_i32_varlen, dict(
            elapsed_state_pool=torch.zeros(3, dtype=torch.int32, device=DEV), cu_seqlens=cu,
            state_indices=slots, total_tokens=5, validated_metadata=ticket)
    r, w, k, v, a, b = (x.view(1, 16, 128).requires_grad_()
                        for x in _tokens(torch.bfloat16, tokens=16))
    return pretrain.pretrain_recurrent_bf16, dict(r=r, w=w, k=k, v=v, a=a, b=b, head_size=64)


def _outcome(entry, call):
    try:
        out = entry(**call) if "w" in call else entry(
            *(call[n] for n in wkv7.C.PACKED_TOKENS if n in call),
            **{n: x for n, x in call.items() if n not in wkv7.C.PACKED_TOKENS}) \
            if "r" in call else entry(call["elapsed_state_pool"], call["cu_seqlens"],
                                      call["state_indices"],
                                      total_tokens=call["total_tokens"],
                                      validated_metadata=call["validated_metadata"])
    except Exception as error:  # noqa: BLE001 - the outcome itself is compared
        return type(error), str(error)
    if out is not None and out.requires_grad:
        return [out.detach(), *torch.autograd.grad((out.float() * 0.25).sum(),
                                                   [call[n] for n in "rwkvab"])]
    return [x for x in (out, call.get("state_pool"), call.get("elapsed_state_pool"))
            if x is not None]


@pytest.mark.parametrize("which", ["fp32", "fp16", "advance", "pretrain"])
def test_whole_call_and_tables_agree(which, monkeypatch):
    for form, change in FORMS.items():
        outcomes = []
        for direct in (True, False):
            entry, call = _call(which)
            try:
                changed = change(call)
            except KeyError:  # an argument that this entry has not
                break
            if set(changed) != set(call):
                break
            with monkeypatch.context() as patch:
                if not direct:
                    patch.setattr(wkv7, "_whole_call", lambda name: None)
                    patch.setattr(torch.compiler, "is_compiling", lambda: True)
                outcomes.append(_outcome(entry, changed))
            torch.cuda.synchronize()
        if not outcomes:
            continue
        here, tables = outcomes
        if isinstance(tables, tuple):
            assert here == tables, form
            continue
        assert isinstance(here, list), (form, here)
        for x, y in zip(here, tables, strict=True):
            assert x.dtype == y.dtype and torch.equal(x, y), form


class _Seen(TorchDispatchMode):
    """A dispatch mode that lists the operators it sees."""

    def __init__(self):
        super().__init__()
        self.names = []

    def __torch_dispatch__(self, func, types, args=(), kwargs=None):
        self.names.append(str(func))
        return func(*args, **(kwargs or {}))


class _SeenFunctions(TorchFunctionMode):
    def __init__(self):
        super().__init__()
        self.names = []

    def __torch_function__(self, func, types, args=(), kwargs=None):
        self.names.append(getattr(func, "__name__", str(func)))
        return func(*args, **(kwargs or {}))


def _gradients(entry, call, dy=None):
    out = entry(**call)
    dy = torch.full_like(out, 0.25) if dy is None else dy
    return [out.detach(), *torch.autograd.grad(out, [call[n] for n in "rwkvab"], dy)]


# Modes see the operators of a call, as through the tables.
@pytest.mark.parametrize("which", ["fp32", "fp16", "advance", "pretrain"])
@pytest.mark.parametrize("mode", [_Seen, _SeenFunctions])
def test_modes_see_the_operators(which, mode, monkeypatch):
    outcomes, names = [], []
    for tables in (False, True):
        entry, call = _call(which)
        with monkeypatch.context() as patch, mode() as seen:
            if tables:
                patch.setattr(wkv7, "_whole_call", lambda name: None)
                patch.setattr(pretrain.C.native().direct, "clampw_accepts", lambda *x: False)
            outcomes.append(_outcome(entry, call))
        names.append(seen.names)
    torch.cuda.synchronize()
    assert names[0] == names[1] and (names[0] or which == "advance")
    for x, y in zip(*outcomes, strict=True):
        assert torch.equal(x, y)


def _under_vmap(entry, call):
    names = [n for n in "rwkvab" if n in call]
    fixed = {n: x for n, x in call.items() if n not in names}
    return torch.vmap(lambda *t: entry(**fixed, **dict(zip(names, t))))(
        *(torch.stack([call[n], call[n]]) for n in names))


def _under_jvp(entry, call):
    with torch.autograd.forward_ad.dual_level():
        r = torch.autograd.forward_ad.make_dual(call["r"].detach(), torch.ones_like(call["r"]))
        return entry(**{**call, "r": r})


# Transforms have the same outcome on both, an error here: no derivative or
# batching rule is passed by.
@pytest.mark.parametrize("transform", [_under_vmap, _under_jvp])
def test_transforms_have_the_same_outcome(transform, monkeypatch):
    outcomes = []
    for direct in (True, False):
        entry, call = _call("pretrain")
        with monkeypatch.context() as patch:
            if not direct:
                patch.setattr(torch.compiler, "is_compiling", lambda: True)
            try:
                outcomes.append(transform(entry, call))
            except Exception as error:  # noqa: BLE001 - the outcome itself is compared
                outcomes.append(type(error))
        torch.cuda.synchronize()
    assert outcomes[0] is outcomes[1] and issubclass(outcomes[0], Exception)


# Saved tensors go through the hooks of the forward, and a gradient comes in any
# layout.
@pytest.mark.parametrize("form", ["hooks", "expanded", "strided", "wrapped"])
def test_pretraining_backward_takes_every_form(form):
    entry, call = _call("pretrain")
    packed, dy = [], torch.full_like(call["r"], 0.25)
    want = _gradients(entry, call, dy)
    if form == "hooks":
        with torch.autograd.graph.saved_tensors_hooks(
                lambda x: packed.append(x.shape) or x.cpu(), lambda x: x.to(DEV)):
            got = _gradients(entry, call, dy)
        assert len(packed) == 8
    else:
        given = {"expanded": dy[:, :1, :1].expand(dy.shape), "strided": _strided(dy),
                 "wrapped": dy.as_subclass(Wrapped)}[form]
        got = _gradients(entry, call, given)
    torch.cuda.synchronize()
    for x, y in zip(got, want, strict=True):
        assert torch.equal(x, y)


# On another stream than the default one the launches are that stream's, and so is
# the backward's (autograd runs it on the forward's).
@pytest.mark.parametrize("which", ["fp32", "fp16", "advance", "pretrain"])
def test_whole_calls_on_another_stream(which):
    entry, call = _call(which)
    want = _outcome(entry, call)
    torch.cuda.synchronize()
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        entry, call = _call(which)
        torch.cuda._sleep(20_000_000)
        if which != "pretrain":  # the inputs are final only after the wait
            for x in call.values():
                if isinstance(x, torch.Tensor) and x.is_floating_point():
                    x.add_(0)
        got = _outcome(entry, call)
        side.synchronize()
    for x, y in zip(got, want, strict=True):
        assert torch.equal(x, y)


# With a switch interval of minutes a thread that waits for the interpreter runs
# only where the calling thread lets go of it.
@pytest.mark.parametrize("direction", ["forward", "backward"])
def test_pretraining_calls_release_the_interpreter(direction):
    native = pretrain.C.native().direct
    tokens = [x.view(1, 16, 128) for x in _tokens(torch.bfloat16, tokens=16)]
    y, ckpt, sda = native.clampw_forward_call(*tokens, 64)
    calls = {"forward": lambda: native.clampw_forward_call(*tokens, 64),
             "backward": lambda: native.clampw_backward_call(y, [*tokens, ckpt, sda], 64)}
    ran, kept, stop = [], [], threading.Event()

    def other():
        while not stop.is_set():
            ran.append(1)
            time.sleep(0)

    call, interval = calls[direction], sys.getswitchinterval()
    thread = threading.Thread(target=other)
    sys.setswitchinterval(600.0)
    try:
        thread.start()
        before = len(ran)
        for _ in range(2000):
            kept.append(call())  # freeing a tensor lets go of it too
            if len(ran) > before:
                break
        released = len(ran) > before
    finally:
        sys.setswitchinterval(interval)
        stop.set()
        thread.join()
    torch.cuda.synchronize()
    assert released
