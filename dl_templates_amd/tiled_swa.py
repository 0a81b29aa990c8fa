"""Tiled 2D sliding-window flash attention (drop-in for src/tiled_swa.py).

``TiledSwa`` keeps the reference's autograd contract (src/tiled_swa.py:602-689): an ``autograd.Function`` with positional
arguments ``(q, k, v, b_size, t_height, t_width, row_size, col_size, sm_scale)`` and a backward that returns
``(dq, dk, dv, None * 6)``.  ``apply`` runs plain eager calls as one compiled node (csrc/torch_binding.cpp); under a trace, a
``torch.func`` transform or a dispatch mode, and with forward-mode tangents, the class itself runs.  ``tiled_swa_fwd``
(:564-600) is the no-grad forward.  Deliberate differences from the reference, all documented in the C header:
outputs have the dtype and device of ``q`` (the reference hard-codes fp16 and the default
device, :608-609), the saved log-sum-exp is fp32, and tiles smaller than 16 tokens have a
backward (the reference raises, :660-661).

``TiledSwaRope`` is the fused RoPE-2D + attention op: it equals ``RotaryPE2D`` applied to
q and k followed by ``TiledSwa`` (the composition of README.md:11) with the caller's q and k
left untouched; its backward returns gradients for the un-rotated q and k.

``TiledSwaImage`` takes q, k, v as images ``[B, IH, IW, heads, D]`` (the layout the reference's
demo converts from with reshape / permute / reshape, src/tiled_swa.py:753-755) and returns o in
the same layout; the kernels address pixels themselves, so no permuted copy is made on either side.
"""
from __future__ import annotations

import torch

from . import _lib


def _shape(q, k, v, b_size, t_height, t_width, row_size, col_size, sm_scale) -> _lib.SwaShape:
    B, H, N, KEY_DIM = q.shape
    HEAD_DIM = v.shape[-1]
    assert N == t_height * t_width * b_size, "seqlen should match image size"
    assert k.shape == (B, H, N, KEY_DIM) and v.shape[:3] == (B, H, N)
    assert q.dtype == k.dtype == v.dtype
    return _lib.SwaShape(B, H, b_size, t_height, t_width, row_size, col_size, KEY_DIM, HEAD_DIM, float(sm_scale),
                         _lib.dtype_code(q))


def _image_shape(q, k, v, bh, bw, row_size, col_size, sm_scale):
    """(SwaShape, SwaTile) of a call on image-layout tensors, for callers of the C ABI."""
    B, IH, IW, H, KEY_DIM = q.shape
    assert IH % bh == 0 and IW % bw == 0, "image size should be a multiple of the tile size"
    assert k.shape == q.shape and v.shape[:4] == q.shape[:4]
    assert q.dtype == k.dtype == v.dtype
    shape = _lib.SwaShape(B, H, bh * bw, IH // bh, IW // bw, row_size, col_size, KEY_DIM, v.shape[-1], float(sm_scale),
                          _lib.dtype_code(q))
    return shape, _lib.SwaTile(bh, bw)


def _pad_plan(q, v, b_size):
    """Head dims (dk, dv) that the operators pad q / k and v to before the launch, or None."""
    return _lib.native.pad_plan(q.shape[-1], v.shape[-1], q, b_size)


def _numbers(s: _lib.SwaShape):
    return tuple(getattr(s, name) for name, _ in s._fields_)


def _forward(q, k, v, shape, rope):
    """(o, lse2) of one forward pass without a graph; ``rope``: (idx, row table, column table) or None."""
    return _lib.native.swa_forward(q, k, v, rope, False, *_numbers(shape))


def _backward(q, k, v, o, lse, do, shape, rope):
    return _lib.native.swa_backward(q, k, v, o, lse, do, rope, False, *_numbers(shape))


def _forward_rot(q, k, v, shape, rope):
    """Forward of the fused op that also returns the rotated q and k (kept for the backward pass)."""
    return _lib.native.swa_forward(q, k, v, rope, True, *_numbers(shape))


def _backward_rot(q_rot, k_rot, v, o, lse, do, shape, rope):
    return _lib.native.swa_backward(q_rot, k_rot, v, o, lse, do, rope, True, *_numbers(shape))


def tiled_swa_fwd(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, b_size: int, t_height: int, t_width: int,
                  row_size: int, col_size: int, sm_scale: float = 1.0):
    return _lib.native.tiled_swa_fwd(q, k, v, b_size, t_height, t_width, row_size, col_size, sm_scale)


def _pad_last(x, d):
    return x if x.shape[-1] == d else torch.nn.functional.pad(x, (0, d - x.shape[-1]))


def _cut_last(x, d):
    return x if x.shape[-1] == d else x[..., :d].contiguous()


class TiledSwa(torch.autograd.Function):
    """``apply(q, k, v, b_size, t_height, t_width, row_size, col_size, sm_scale)`` -> o; gradients for q, k, v."""

    @classmethod
    def apply(cls, *args):
        o = _lib.native.tiled_swa(*args) if cls is TiledSwa else NotImplemented
        return super().apply(*args) if o is NotImplemented else o

    @staticmethod
    def forward(ctx, q, k, v, b_size, t_height, t_width, row_size, col_size, sm_scale):
        ctx.dims, plan = (q.shape[-1], v.shape[-1]), _pad_plan(q, v, b_size)
        if plan is not None:
            q, k, v = _pad_last(q, plan[0]), _pad_last(k, plan[0]), _pad_last(v, plan[1])
        ctx.shape = _shape(q, k, v, b_size, t_height, t_width, row_size, col_size, sm_scale)
        o, m = _forward(q, k, v, ctx.shape, None)
        ctx.save_for_backward(q, k, v, m, o)
        return _cut_last(o, ctx.dims[1])

    @staticmethod
    def backward(ctx, do):
        q, k, v, m, o = ctx.saved_tensors
        dq, dk, dv = _backward(q, k, v, o, m, _pad_last(do, v.shape[-1]), ctx.shape, None)
        return (_cut_last(dq, ctx.dims[0]), _cut_last(dk, ctx.dims[0]), _cut_last(dv, ctx.dims[1])) + (None,) * 6


class TiledSwaRope(torch.autograd.Function):
    """o = TiledSwa(rope(q), rope(k), v) with the rotation fused into the q / k tile loads.

    ``apply(q, k, v, idx, row_cs_buffer, col_cs_buffer, b_size, t_height, t_width, row_size, col_size, sm_scale,
    save_rotated=None)``.  ``save_rotated`` (default True): the forward pass also stores the
    rotated q and k (what ``RotaryPE2D`` leaves in place in the reference's composition) and the backward pass
    reads those, rotating only dq and dk back as they are stored.  False keeps nothing but the caller's q and k
    and rotates every staged tile again in the backward kernels: two tensors less memory, slower.  It is a
    per-call argument, kept in the call's own graph node: nothing is shared between calls or threads.
    """

    @classmethod
    def apply(cls, *args):
        o = _lib.native.tiled_swa_rope(*args) if cls is TiledSwaRope else NotImplemented
        return super().apply(*args) if o is NotImplemented else o

    @staticmethod
    def forward(ctx, q, k, v, idx, row_cs_buffer, col_cs_buffer, b_size, t_height, t_width, row_size, col_size,
                sm_scale, save_rotated=None):
        ctx.n_inputs = 12 if save_rotated is None else 13   # backward returns one entry per argument of apply
        ctx.dims, plan = (q.shape[-1], v.shape[-1]), _pad_plan(q, v, b_size)
        if plan is not None:   # zero columns behind the rotated ones
            q, k, v = _pad_last(q, plan[0]), _pad_last(k, plan[0]), _pad_last(v, plan[1])
        ctx.shape = _shape(q, k, v, b_size, t_height, t_width, row_size, col_size, sm_scale)
        assert row_cs_buffer.shape[1] == col_cs_buffer.shape[1], "row and column table must have one R"
        assert idx.shape[0] == q.shape[2], "idx must have one entry per token"
        rope = (idx, row_cs_buffer, col_cs_buffer)
        ctx.rotated = True if save_rotated is None else bool(save_rotated)
        if ctx.rotated:
            o, m, q, k = _forward_rot(q, k, v, ctx.shape, rope)
        else:
            o, m = _forward(q, k, v, ctx.shape, rope)
        ctx.save_for_backward(q, k, v, m, o, *rope)
        return _cut_last(o, ctx.dims[1])

    @staticmethod
    def backward(ctx, do):
        q, k, v, m, o, *rope = ctx.saved_tensors
        run = _backward_rot if ctx.rotated else _backward
        dq, dk, dv = run(q, k, v, o, m, _pad_last(do, v.shape[-1]), ctx.shape, tuple(rope))
        return (_cut_last(dq, ctx.dims[0]), _cut_last(dk, ctx.dims[0]), _cut_last(dv, ctx.dims[1])) + (None,) * (ctx.n_inputs - 3)


class TiledSwaImage(torch.autograd.Function):
    """``TiledSwa`` on image-layout tensors: q, k ``[B, IH, IW, heads, dk]``, v and o ``[B, IH, IW, heads, dv]``.

    ``apply(q, k, v, bh, bw, row_size, col_size, sm_scale)``.  A tile is a block of ``bh x bw`` pixels
    (``b_size = bh * bw``); the window is ``row_size`` / ``col_size`` tiles to each side as in ``TiledSwa``.  Equals the
    reference's conversion to ``[B, heads, N, D]`` (src/tiled_swa.py:753-755, inverted), ``TiledSwa`` and the
    conversion back, without the copies.
    """

    @classmethod
    def apply(cls, *args):
        o = _lib.native.tiled_swa_image(*args) if cls is TiledSwaImage else NotImplemented
        return super().apply(*args) if o is NotImplemented else o

    @staticmethod
    def forward(ctx, q, k, v, bh, bw, row_size, col_size, sm_scale):
        ctx.scalars = (bh, bw, row_size, col_size, sm_scale)
        o, lse = _lib.native.image_forward(q, k, v, *ctx.scalars)
        ctx.save_for_backward(q, k, v, o, lse)
        return o

    @staticmethod
    def backward(ctx, do):
        return _lib.native.image_backward(*ctx.saved_tensors, do, *ctx.scalars) + (None,) * 5


def swa_image_offsets(t_height: int, t_width: int, bh: int, bw: int, stride_y: int, stride_x: int,
                      device="cuda") -> torch.Tensor:
    """int64 [N]: element offset of every token's pixel, computed by the kernels' own token -> pixel routine."""
    out = torch.empty((t_height * t_width * bh * bw,), dtype=torch.int64, device=device)
    with torch.cuda.device(out.device):
        _lib.check(_lib.load().dlt_swa_image_offsets(t_height, t_width, bh, bw, stride_y, stride_x, _lib.ptr(out),
                                                     _lib.stream_of(out)))
    return out


def swa_neighbors(t_height: int, t_width: int, row_size: int, col_size: int, device="cuda") -> torch.Tensor:
    """bool [T, T] neighbour mask computed on the device by the kernels' own window routine."""
    T = t_height * t_width
    out = torch.empty((T, T), dtype=torch.uint8, device=device)
    with torch.cuda.device(out.device):
        _lib.check(_lib.load().dlt_swa_neighbors(t_height, t_width, row_size, col_size, _lib.ptr(out),
                                                 _lib.stream_of(out)))
    return out.bool()
