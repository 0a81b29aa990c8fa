"""Flash attention with separate qk / vo head dims (drop-in for src/flash_attn.py).

``attention(q, k, v, causal, sm_scale)`` = ``_attention.apply`` as in the reference
(src/flash_attn.py:452-541); gradients for q, k and v.  Unlike the
reference (one N_CTX, :479) the key length may differ from the query length when
``causal`` is False, and there is no ``N_CTX % 128`` requirement (:512).  The graph node and the argument checks are
compiled (csrc/torch_binding.cpp).
"""
from __future__ import annotations

from . import _lib


def _pad_plan(q, v):
    """Head dims (dk, dv) that ``attention`` pads q / k and v to before the launch, or None."""
    return _lib.native.pad_plan(q.shape[-1], v.shape[-1], q, -1)


def _forward(q, k, v, causal, sm_scale):
    """(o, M): the output and the saved log2-domain log-sum-exp [B, H, Lq] (src/flash_attn.py:463-483), no graph."""
    return _lib.native.flash_forward(q, k, v, causal, sm_scale)


class _attention:

    @staticmethod
    def apply(*args):
        return _lib.native.flash(*args)


attention = _attention.apply
