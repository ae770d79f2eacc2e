"""Pretraining recurrence (clampw v3), importable as ``flashrwkv2.tmix.wkv7.pretrain``.

``pretrain_recurrent_bf16`` keeps the reference's signature, error contract
and autograd behaviour (reference ``flashrwkv2/tmix/wkv7/pretrain.py:14-129``):
dense bf16 ``[B,T,C]`` tokens with decay logits ``w`` (retention
``exp(-e^{-1/2} sigmoid(w))``), zero initial state, output ``[B,T,C]``.

Both directions run through ``torch.ops.rwkv7_clampw_v3``: head size 64 on
the chunked bf16-MFMA kernels, 128 on the bf16-MFMA kernels over 16-token
pieces, 256 on the fp32 matrix kernels over 16-token pieces. The forward saves
the state every 16 tokens; the backward recomputes from those states and never
divides by the decay.
"""

from __future__ import annotations

import sys

import torch

from ... import _contract as C
from ..._contract import check, is_tensor

CHUNK_LEN = 16
_DECAY_AND_FRIENDS = ("w", "k", "v", "a", "b")


def _bf16(x, ns) -> bool:
    return x.dtype == torch.bfloat16


def _cuda_contig(x, ns) -> bool:
    return x.is_cuda and x.is_contiguous()


# Reference ``pretrain.py:14-48``.
PRETRAIN = (
    check("head_size", C.one_of({64, 128, 256}), ValueError,
          "head_size must be one of 64, 128, or 256"),
    check(None, lambda _, ns: len(ns["tensors"]) == 6, ValueError,
          "clampw requires r, w, k, v, a, and b"),
    is_tensor("r"),
    check("r", lambda x, ns: x.ndim == 3 and min(x.shape) > 0, ValueError,
          "r must have shape [B,T,C] with nonzero dimensions"),
    check("r", _bf16, TypeError, "r must be bfloat16"),
    check("r", _cuda_contig, ValueError, "r must be contiguous CUDA"),
    C.Each(_DECAY_AND_FRIENDS, (
        is_tensor(),
        check(None, _bf16, TypeError, "{name} must be bfloat16"),
        check(None, _cuda_contig, ValueError, "{name} must be contiguous CUDA"),
        check(None, C.same_shape_as("r"), ValueError, "{name} must match r shape"),
        check(None, C.same_device_as("r"), ValueError, "{name} must share the r device"),
    )),
    check("r", lambda x, ns: x.shape[2] % ns["head_size"] == 0, ValueError,
          "C must be divisible by head_size"),
    check("r", lambda x, ns: x.shape[1] % CHUNK_LEN == 0, ValueError,
          "T must be divisible by the canonical chunk length 16"),
)


def _check(tensors: tuple, head_size: int) -> None:
    ns = {"tensors": tensors, "head_size": head_size, "r": tensors[0] if tensors else None}
    ns.update(zip(_DECAY_AND_FRIENDS, tensors[1:]))
    C.enforce(PRETRAIN, ns)


class _ClampwV3(torch.autograd.Function):
    """Autograd node over the two ``rwkv7_clampw_v3`` ops (forward saves the
    state before every 16th token, [B,H,T/16,D,D], and a^T S, [B,T,H,D];
    backward recomputes from them). ``direct``: plain tensors outside of modes,
    tracing and compiling take the native calls that allocate the buffers too;
    others go through the registered ops."""

    @staticmethod
    def forward(ctx, direct: bool, head_size: int, *tensors):
        ctx.direct, ctx.head_size = direct, head_size
        if direct:
            y, ckpt, sda = C.native().direct.clampw_forward_call(*tensors, head_size)
        else:
            batch, tokens, channels = tensors[0].shape
            heads = channels // head_size
            split = [t.view(batch, tokens, heads, head_size) for t in tensors]
            like = {"device": tensors[0].device, "dtype": torch.float32}
            y = torch.empty_like(split[3])
            ckpt = torch.empty((batch, heads, tokens // CHUNK_LEN, head_size, head_size), **like)
            sda = torch.empty((batch, tokens, heads, head_size), **like)
            torch.ops.rwkv7_clampw_v3.forward(*split, y, ckpt, sda, head_size)
            y = y.view(batch, tokens, channels)
        ctx.save_for_backward(*tensors, ckpt, sda)
        return y

    @staticmethod
    def backward(ctx, dy):
        saved, d = ctx.saved_tensors, ctx.head_size
        if ctx.direct:
            grads = C.native().direct.clampw_backward_call(dy, saved, d)
            if grads is not None:
                return (None, None, *grads)
        *tensors, ckpt, sda = saved
        split = [t.view(*t.shape[:2], -1, d) for t in tensors]
        grads = [torch.empty_like(t) for t in split]
        torch.ops.rwkv7_clampw_v3.backward(*split, dy.contiguous().view(split[0].shape), ckpt, sda,
                                           *grads, d)
        return (None, None, *(g.view(tensors[0].shape) for g in grads))


def pretrain_recurrent_bf16(r: torch.Tensor, w: torch.Tensor, k: torch.Tensor,
                            v: torch.Tensor, a: torch.Tensor, b: torch.Tensor, *,
                            head_size: int = 64) -> torch.Tensor:
    """clampw v3 pretraining recurrence with autograd (reference ``pretrain.py:109-126``)."""
    facade = getattr(sys.modules[__name__.split(".")[0]], "_C", None)
    direct = (facade is not None and not torch.compiler.is_compiling()
              and facade.direct.clampw_accepts(r, w, k, v, a, b, head_size))
    if not direct:
        _check((r, w, k, v, a, b), head_size)
    C.native()
    if torch.cuda.is_current_stream_capturing():
        raise RuntimeError("pretrain_recurrent_bf16 does not run under HIP graph capture: "
                           "its chunked kernels are not validated inside a captured graph")
    return _ClampwV3.apply(direct, int(head_size), r, w, k, v, a, b)


__all__ = ["pretrain_recurrent_bf16"]
