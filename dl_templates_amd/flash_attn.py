"""Flash attention with separate qk / vo head dims (drop-in for src/flash_attn.py).

``attention(q, k, v, causal, sm_scale)`` = ``_attention.apply`` as in the reference
(src/flash_attn.py:452-541), an ``autograd.Function``; backward returns ``(dq, dk, dv, None, None)``.  Unlike the
reference (one N_CTX, :479) the key length may differ from the query length when
``causal`` is False, and there is no ``N_CTX % 128`` requirement (:512).  ``apply`` runs plain eager calls as one compiled
node (csrc/torch_binding.cpp); under a trace, a ``torch.func`` transform or a dispatch mode, and with forward-mode tangents,
the class itself runs.
"""
from __future__ import annotations

import torch

from . import _lib


def _pad_plan(q, v):
    """Head dims (dk, dv) that ``attention`` pads q / k and v to before the launch, or None."""
    return _lib.native.pad_plan(q.shape[-1], v.shape[-1], q, -1)


def _forward(q, k, v, causal, sm_scale):
    """(o, M): the output and the saved log2-domain log-sum-exp [B, H, Lq] (src/flash_attn.py:463-483), no graph."""
    return _lib.native.flash_forward(q, k, v, causal, sm_scale)


def _pad_last(x, d):
    return x if x.shape[-1] == d else torch.nn.functional.pad(x, (0, d - x.shape[-1]))


def _cut_last(x, d):
    return x if x.shape[-1] == d else x[..., :d].contiguous()


class _attention(torch.autograd.Function):

    @classmethod
    def apply(cls, *args):
        o = _lib.native.flash(*args) if cls is _attention else NotImplemented
        return super().apply(*args) if o is NotImplemented else o

    @staticmethod
    def forward(ctx, q, k, v, causal, sm_scale):
        ctx.dims, plan = (q.shape[-1], v.shape[-1]), _pad_plan(q, v)
        if plan is not None:
            q, k, v = _pad_last(q, plan[0]), _pad_last(k, plan[0]), _pad_last(v, plan[1])
        ctx.scalars = (causal, sm_scale)
        o, M = _forward(q, k, v, causal, sm_scale)
        ctx.save_for_backward(q, k, v, o, M)
        return _cut_last(o, ctx.dims[1])

    @staticmethod
    def backward(ctx, do):
        q, k, v, o, M = ctx.saved_tensors
        dq, dk, dv = _lib.native.flash_backward(q, k, v, o, M, _pad_last(do, v.shape[-1]), *ctx.scalars)
        return _cut_last(dq, ctx.dims[0]), _cut_last(dk, ctx.dims[0]), _cut_last(dv, ctx.dims[1]), None, None


attention = _attention.apply
