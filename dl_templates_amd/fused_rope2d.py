"""Fused in-place 2D rotary position encoding (drop-in for src/fused_rope2d.py).

Same names and call signatures as the reference: ``RotaryPE2D`` (autograd.Function,
src/fused_rope2d.py:124-168), ``FusedInplaceRotaryPositionEncoding2D`` (:171-201).  The
Triton kernels are replaced by the gfx950 HIP kernel behind ``dlt_rope2d``.
"""
from __future__ import annotations

import torch

from . import _lib
from .rope2d import FusedRotaryPositionEncodingContext


def _launch(x: torch.Tensor, idx, row_cs, col_cs, inverse: bool) -> None:
    _lib.native.rope_inplace(x, idx, row_cs, col_cs, inverse)


class RotaryPE2D(torch.autograd.Function):
    """``apply(x[B', N, C], idx, row_cs_buffer, col_cs_buffer)``: x is rotated IN PLACE and returned
    (src/fused_rope2d.py:126-145); the backward pass rotates the gradient back (:148-168).  Plain eager calls run as one compiled
    node (csrc/torch_binding.cpp), any other (trace, transform, dispatch mode, forward-mode tangent) through this class."""

    @classmethod
    def apply(cls, *args):
        y = _lib.native.rope_apply(*args) if cls is RotaryPE2D else NotImplemented
        return super().apply(*args) if y is NotImplemented else y

    @staticmethod
    def forward(ctx, x, idx, row_cs_buffer, col_cs_buffer):
        assert row_cs_buffer.shape[1] == col_cs_buffer.shape[1], "row and column table must have one R"
        assert idx.shape[0] == x.shape[1], "idx must have one entry per token"
        _launch(x, idx, row_cs_buffer, col_cs_buffer, False)
        ctx.mark_dirty(x)
        ctx.save_for_backward(idx, row_cs_buffer, col_cs_buffer)
        return x

    @staticmethod
    @torch.autograd.function.once_differentiable
    def backward(ctx, do):
        dx = do.clone()
        _launch(dx, *ctx.saved_tensors, True)
        return dx, None, None, None


def rope2d_qk_(q: torch.Tensor, k: torch.Tensor, idx: torch.Tensor, row_cs_buffer: torch.Tensor,
               col_cs_buffer: torch.Tensor, inverse: bool = False):
    """Rotate q[B, H, N, C] and k[B, H, N, C] in place with ONE launch (no autograd).

    Equivalent to two ``RotaryPE2D`` forward calls; halves the launch count and shares the
    idx / table reads (the composition of README.md:11)."""
    return _lib.native.rope_pair(q, k, idx, row_cs_buffer, col_cs_buffer, inverse)


def rope_pe_mask(idx: torch.Tensor) -> torch.Tensor:
    """uint8[N]: bit0 = row axis rotated, bit1 = column axis rotated, decoded on the device by
    the code the rotation kernels use (src/fused_rope2d.py:40-45)."""
    _lib.require_cuda(idx)
    out = torch.empty(idx.shape[0], dtype=torch.uint8, device=idx.device)
    with torch.cuda.device(idx.device):
        _lib.check(_lib.load().dlt_rope_pe_mask(_lib.ptr(idx), idx.shape[0], _lib.ptr(out), _lib.stream_of(idx)))
    return out


class FusedInplaceRotaryPositionEncoding2D(torch.nn.Module):
    @staticmethod
    def encode_idx(height: int, width: int) -> torch.Tensor:
        r"""Token indices for image-like 2D data: ``(row << 16) | col``, row-major, int32
        (src/fused_rope2d.py:173-183)."""
        rows = torch.arange(0, height)
        cols = torch.arange(0, width)
        return torch.bitwise_or(rows[:, None] << 16, cols).flatten().to(torch.int32)

    def __init__(self, n_components: int, max_h: int, max_w: int):
        super().__init__()
        self.max_h = max_h
        self.max_w = max_w
        self.row_components = n_components // 2
        self.col_components = n_components // 2
        self.row_buffer = FusedRotaryPositionEncodingContext(self.row_components, max_h)
        self.col_buffer = FusedRotaryPositionEncodingContext(self.col_components, max_w)

    def forward(self, x: torch.Tensor, idx: torch.Tensor) -> torch.Tensor:
        # x: [B, Head, N, C] idx: [N, ]
        rope = (idx, self.row_buffer.cs_components, self.col_buffer.cs_components)
        y = _lib.native.rope_heads(x, *rope)
        if y is NotImplemented:
            B, H, N, C = x.shape
            y = RotaryPE2D.apply(x.reshape((-1, N, C)), *rope).reshape(x.shape)
        return y
