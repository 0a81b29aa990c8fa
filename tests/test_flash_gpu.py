"""GPU parity of flash attention (dlt_flash_fwd / dlt_flash_bwd) against SDPA on the CPU.

Follows the reference's own check (src/flash_attn.py:616-659: q, k L2-normalised, loss =
o.sum(), allclose(1e-2, 1e-2) on o, dq, dk, dv, Z=4, H in {4,8}, N in {512,2048},
dv in {16,32}, dk in {16,64}) with seeded inputs, plus Lq != Lk, odd lengths, bf16 and the
stated tolerances (forward max-abs <= 2e-2, gradients relative <= 5e-2).
"""
import itertools
import math

import pytest
import torch

from oracle import attn_oracle as orc

pytestmark = pytest.mark.gpu


def _fa():
    from dl_templates_amd import flash_attn
    return flash_attn


def _l2(x):
    return x / torch.linalg.norm(x, dim=-1, keepdims=True)


def _rel(got, want):
    return ((got.float().cpu() - want).abs().max() / want.abs().max().clamp_min(1e-3)).item()


SWEEP = list(itertools.product([False, True], [4, 8], [512, 2048], [16, 32], [16, 64]))


@pytest.mark.parametrize("causal,head,n_ctx,h_dim,k_dim", SWEEP[::3] + [SWEEP[-1]])
def test_reference_correctness_sweep(causal, head, n_ctx, h_dim, k_dim):
    Z = 2 if n_ctx == 2048 else 4
    g = torch.Generator().manual_seed(n_ctx + head + h_dim + k_dim)
    q = _l2(torch.randn((Z, head, n_ctx, k_dim), generator=g)).half()
    k = _l2(torch.randn((Z, head, n_ctx, k_dim), generator=g)).half()
    v = torch.randn((Z, head, n_ctx, h_dim), generator=g).half()
    do = torch.ones((Z, head, n_ctx, h_dim))
    o_std, dq, dk, dv = orc.flash_grads(q.float(), k.float(), v.float(), do, causal, 1.0)
    q2, k2, v2 = (t.cuda().requires_grad_(True) for t in (q, k, v))
    o = _fa().attention(q2, k2, v2, causal, 1.0)
    o.flatten().sum().backward()
    assert torch.allclose(o.float().cpu(), o_std, atol=1e-2, rtol=1e-2)
    assert torch.allclose(q2.grad.float().cpu(), dq, atol=1e-2, rtol=1e-2)
    assert torch.allclose(k2.grad.float().cpu(), dk, atol=1e-2, rtol=1e-2)
    assert torch.allclose(v2.grad.float().cpu(), dv, atol=1e-2, rtol=1e-2)


@pytest.mark.parametrize("Lq,Lk,dk,dv,dtype", [
    (256, 512, 64, 128, torch.bfloat16), (100, 333, 64, 128, torch.bfloat16), (1, 1, 16, 16, torch.bfloat16),
    (129, 31, 32, 64, torch.float16), (64, 1000, 128, 128, torch.bfloat16), (300, 300, 64, 64, torch.float32),
    (17, 257, 48, 80, torch.bfloat16)])
def test_cross_attention_distinct_dims_and_lengths(Lq, Lk, dk, dv, dtype):
    q, k, v, do = orc.make_qkv(Lq * 7 + Lk, 2, 3, Lq, Lk, dk, dv, dtype)
    scale = 1 / math.sqrt(dk)
    o_w, dq_w, dk_w, dv_w = orc.flash_grads(q.float(), k.float(), v.float(), do.float(), False, scale)
    qg, kg, vg = (t.cuda().requires_grad_(True) for t in (q, k, v))
    o = _fa().attention(qg, kg, vg, False, scale)
    o.backward(do.cuda())
    assert o.shape == (2, 3, Lq, dv) and o.dtype == dtype
    assert (o.float().cpu() - o_w).abs().max().item() <= 2e-2
    errs = (_rel(qg.grad, dq_w), _rel(kg.grad, dk_w), _rel(vg.grad, dv_w))
    assert max(errs) <= 5e-2, errs


@pytest.mark.parametrize("causal,Lq,Lk,dk,dv,dtype", [
    (False, 256, 512, 64, 128, torch.bfloat16), (False, 100, 333, 64, 64, torch.float16), (True, 300, 300, 128, 128, torch.bfloat16),
    (True, 129, 129, 32, 32, torch.float16), (False, 77, 190, 48, 80, torch.float32), (False, 1, 1, 16, 16, torch.bfloat16)])
def test_saved_log_sum_exp(causal, Lq, Lk, dk, dv, dtype):
    """M = m + log2(l), the vector the forward pass saves for the backward pass (src/flash_attn.py:168-171),
    directly against the oracle; 2e-2 in log2 units."""
    q, k, v, _ = orc.make_qkv(Lq + 3 * Lk, 2, 2, Lq, Lk, dk, dv, dtype)
    scale = 1 / math.sqrt(dk)
    o, M = _fa()._forward(q.cuda(), k.cuda(), v.cuda(), causal, scale)
    assert M.dtype == torch.float32 and M.shape == (2, 2, Lq)
    want = orc.flash_lse2(q, k, scale, causal)
    assert (M.cpu() - want).abs().max().item() <= 2e-2
    assert (o.float().cpu() - orc.flash_ref(q.float(), k.float(), v.float(), causal, scale)).abs().max().item() <= 2e-2


def test_negative_scale_matches_sdpa():
    q, k, v, do = orc.make_qkv(91, 1, 2, 200, 320, 64, 64, torch.bfloat16)
    o_w, dq_w, dk_w, dv_w = orc.flash_grads(q.float(), k.float(), v.float(), do.float(), False, -0.125)
    qg, kg, vg = (t.cuda().requires_grad_(True) for t in (q, k, v))
    o = _fa().attention(qg, kg, vg, False, -0.125)
    o.backward(do.cuda())
    assert (o.float().cpu() - o_w).abs().max().item() <= 2e-2
    assert max(_rel(qg.grad, dq_w), _rel(kg.grad, dk_w), _rel(vg.grad, dv_w)) <= 5e-2


@pytest.mark.parametrize("causal,Lq,Lk,dk,dv,dtype", [
    (False, 256, 384, 256, 256, torch.bfloat16), (True, 200, 200, 256, 256, torch.float16), (False, 65, 130, 256, 64, torch.bfloat16),
    (False, 100, 100, 64, 256, torch.float16), (True, 129, 129, 192, 160, torch.bfloat16), (False, 40, 70, 256, 256, torch.float32)])
def test_head_dim_256(causal, Lq, Lk, dk, dv, dtype):
    """The reference admits head dims up to 256 (src/flash_attn.py:460-462); forward, saved log-sum-exp and
    gradients against SDPA."""
    q, k, v, do = orc.make_qkv(Lq + dk, 1, 2, Lq, Lk, dk, dv, dtype)
    scale = 1 / math.sqrt(dk)
    o_w, dq_w, dk_w, dv_w = orc.flash_grads(q.float(), k.float(), v.float(), do.float(), causal, scale)
    qg, kg, vg = (t.cuda().requires_grad_(True) for t in (q, k, v))
    o = _fa().attention(qg, kg, vg, causal, scale)
    o.backward(do.cuda())
    assert o.shape == (1, 2, Lq, dv) and o.dtype == dtype
    assert (o.float().cpu() - o_w).abs().max().item() <= 2e-2
    errs = (_rel(qg.grad, dq_w), _rel(kg.grad, dk_w), _rel(vg.grad, dv_w))
    assert max(errs) <= 5e-2, errs
    _, M = _fa()._forward(q.cuda(), k.cuda(), v.cuda(), causal, scale)
    assert (M.cpu() - orc.flash_lse2(q, k, scale, causal)).abs().max().item() <= 2e-2


def test_c5_shape_reduced_batch():
    # benchmark config 5 shape with B=1, H=2 (CPU oracle time): Lq=4096, Lk=8192, 64/128
    q, k, v, do = orc.make_qkv(55, 1, 2, 4096, 8192, 64, 128, torch.bfloat16)
    o_w, dq_w, dk_w, dv_w = orc.flash_grads(q.float(), k.float(), v.float(), do.float(), False, 0.125)
    qg, kg, vg = (t.cuda().requires_grad_(True) for t in (q, k, v))
    o = _fa().attention(qg, kg, vg, False, 0.125)
    o.backward(do.cuda())
    assert (o.float().cpu() - o_w).abs().max().item() <= 2e-2
    errs = (_rel(qg.grad, dq_w), _rel(kg.grad, dk_w), _rel(vg.grad, dv_w))
    print("c5 rel errs", errs)
    assert max(errs) <= 5e-2, errs


def test_causal_matches_sdpa_bf16():
    q, k, v, do = orc.make_qkv(56, 1, 2, 777, 777, 64, 64, torch.bfloat16)
    o_w, dq_w, dk_w, dv_w = orc.flash_grads(q.float(), k.float(), v.float(), do.float(), True, 0.125)
    qg, kg, vg = (t.cuda().requires_grad_(True) for t in (q, k, v))
    o = _fa().attention(qg, kg, vg, True, 0.125)
    o.backward(do.cuda())
    assert (o.float().cpu() - o_w).abs().max().item() <= 2e-2
    assert max(_rel(qg.grad, dq_w), _rel(kg.grad, dk_w), _rel(vg.grad, dv_w)) <= 5e-2


@pytest.mark.parametrize("N,dk,dv,dtype", [
    (1, 64, 64, torch.bfloat16), (63, 64, 128, torch.bfloat16), (64, 128, 128, torch.bfloat16),
    (65, 64, 64, torch.float16), (129, 64, 128, torch.bfloat16), (1000, 128, 128, torch.bfloat16),
    (384, 32, 32, torch.float16)])
def test_causal_lengths_and_dims(N, dk, dv, dtype):
    """Causal fast path: lengths around the 64-key chunk and the 128-query block, all head-dim classes."""
    q, k, v, do = orc.make_qkv(N + dk, 2, 2, N, N, dk, dv, dtype)
    scale = 1 / math.sqrt(dk)
    o_w, dq_w, dk_w, dv_w = orc.flash_grads(q.float(), k.float(), v.float(), do.float(), True, scale)
    qg, kg, vg = (t.cuda().requires_grad_(True) for t in (q, k, v))
    o = _fa().attention(qg, kg, vg, True, scale)
    o.backward(do.cuda())
    assert (o.float().cpu() - o_w).abs().max().item() <= 2e-2
    errs = (_rel(qg.grad, dq_w), _rel(kg.grad, dk_w), _rel(vg.grad, dv_w))
    assert max(errs) <= 5e-2, errs


@pytest.mark.parametrize("B,H,N,dk,dv", [(1, 7, 4096, 128, 128), (3, 3, 2048, 64, 64), (1, 5, 1536, 64, 128)])
def test_causal_block_order_over_heads(B, H, N, dk, dv):
    """Under a causal mask the workgroups of several (batch, head) slabs are interleaved, heaviest blocks first, in groups
    sized by their K / V footprint (groups of 2, 8 and 7 heads here, the last one partial).  The order must not change any
    result: every slab run on its own (one head per call) gives the same bits, and slab 0 matches the oracle."""
    q, k, v, do = orc.make_qkv(N + H, B, H, N, N, dk, dv, torch.bfloat16)
    scale = 1 / math.sqrt(dk)
    qg, kg, vg = (t.cuda().requires_grad_(True) for t in (q, k, v))
    o = _fa().attention(qg, kg, vg, True, scale)
    o.backward(do.cuda())
    for b in range(B):
        for h in range(H):
            q1, k1, v1 = (t[b:b + 1, h:h + 1].contiguous().cuda().requires_grad_(True) for t in (q, k, v))
            o1 = _fa().attention(q1, k1, v1, True, scale)
            o1.backward(do[b:b + 1, h:h + 1].contiguous().cuda())
            assert torch.equal(o1[0, 0], o[b, h]), (b, h)
            assert torch.equal(q1.grad[0, 0], qg.grad[b, h]) and torch.equal(k1.grad[0, 0], kg.grad[b, h]) \
                and torch.equal(v1.grad[0, 0], vg.grad[b, h]), (b, h)
    sl = (slice(0, 1), slice(0, 1))
    o_w, dq_w, dk_w, dv_w = orc.flash_grads(q[sl].float(), k[sl].float(), v[sl].float(), do[sl].float(), True, scale)
    assert (o[sl].float().cpu() - o_w).abs().max().item() <= 2e-2
    assert max(_rel(qg.grad[sl], dq_w), _rel(kg.grad[sl], dk_w), _rel(vg.grad[sl], dv_w)) <= 5e-2


@pytest.mark.parametrize("causal,dk,dv,dtype", [
    (False, 64, 128, torch.bfloat16), (False, 64, 64, torch.float16), (False, 128, 128, torch.bfloat16),
    (True, 64, 128, torch.float16), (True, 128, 128, torch.bfloat16), (True, 64, 64, torch.bfloat16)])
def test_chunk_boundaries_of_the_async_staged_kernels(causal, dk, dv, dtype):
    """Head dims of exactly 64 / 128 run on the kernels that copy chunks HBM -> LDS asynchronously into two or three
    buffers: lengths of one, two, three and four chunks (64 keys in the backward kernels, 128 in the forward kernel),
    one token more and one less, and query counts around the 128- and 256-query workgroups."""
    pairs = [(1, 1), (63, 64), (200, 65), (128, 127), (129, 128), (256, 129), (257, 191), (130, 192), (70, 193), (255, 256),
             (33, 257), (300, 320)]
    scale = 1 / math.sqrt(dk)
    for Lq, Lk in pairs:
        if causal:
            Lq = Lk
        q, k, v, do = orc.make_qkv(Lq * 5 + Lk + dk, 1, 2, Lq, Lk, dk, dv, dtype)
        o_w, dq_w, dk_w, dv_w = orc.flash_grads(q.float(), k.float(), v.float(), do.float(), causal, scale)
        qg, kg, vg = (t.cuda().requires_grad_(True) for t in (q, k, v))
        o = _fa().attention(qg, kg, vg, causal, scale)
        o.backward(do.cuda())
        assert (o.float().cpu() - o_w).abs().max().item() <= 2e-2, (Lq, Lk)
        errs = (_rel(qg.grad, dq_w), _rel(kg.grad, dk_w), _rel(vg.grad, dv_w))
        assert max(errs) <= 5e-2, (Lq, Lk, errs)


@pytest.mark.parametrize("causal,dk,dv,dtype", [
    (False, 40, 40, torch.bfloat16), (True, 48, 80, torch.float16), (False, 80, 80, torch.bfloat16), (True, 96, 96, torch.bfloat16),
    (False, 72, 120, torch.float16), (False, 56, 128, torch.bfloat16), (True, 128, 104, torch.bfloat16), (False, 64, 8, torch.float16)])
def test_async_staged_kernels_with_head_dims_below_the_padded_class(causal, dk, dv, dtype):
    """Head dims that are multiples of 8 below their class (64 or 128) also run on the asynchronously staged kernels: the
    lanes of the missing 16-byte pieces copy nothing and their LDS slots are zeroed once.  Lengths of one to several
    chunks, one token more and less."""
    scale = 1 / math.sqrt(dk)
    for Lq, Lk in [(1, 1), (65, 64), (130, 191), (257, 320), (300, 129), (512, 513)]:
        if causal:
            Lq = Lk
        q, k, v, do = orc.make_qkv(Lq + 3 * Lk + dk + dv, 2, 2, Lq, Lk, dk, dv, dtype)
        o_w, dq_w, dk_w, dv_w = orc.flash_grads(q.float(), k.float(), v.float(), do.float(), causal, scale)
        qg, kg, vg = (t.cuda().requires_grad_(True) for t in (q, k, v))
        o = _fa().attention(qg, kg, vg, causal, scale)
        o.backward(do.cuda())
        assert (o.float().cpu() - o_w).abs().max().item() <= 2e-2, (Lq, Lk)
        errs = (_rel(qg.grad, dq_w), _rel(kg.grad, dk_w), _rel(vg.grad, dv_w))
        assert max(errs) <= 5e-2, (Lq, Lk, errs)


@pytest.mark.parametrize("causal,dk,dv,dtype", [(False, 100, 100, torch.bfloat16), (True, 50, 36, torch.float16), (False, 20, 127, torch.bfloat16),
                                                 (True, 1, 3, torch.float16), (False, 65, 9, torch.bfloat16)])
def test_head_dims_that_are_not_multiples_of_eight(causal, dk, dv, dtype):
    """The public entry pads such head dims with zero columns to the next multiple of 8 (the kernels read 16-byte row
    pieces) and slices the results: shapes, contiguity and values against the oracle."""
    scale = 1 / math.sqrt(dk)
    for Lq, Lk in [(1, 1), (130, 191), (300, 129)]:
        if causal:
            Lq = Lk
        q, k, v, do = orc.make_qkv(Lq + Lk + dk + dv, 1, 3, Lq, Lk, dk, dv, dtype)
        o_w, dq_w, dk_w, dv_w = orc.flash_grads(q.float(), k.float(), v.float(), do.float(), causal, scale)
        qg, kg, vg = (t.cuda().requires_grad_(True) for t in (q, k, v))
        o = _fa().attention(qg, kg, vg, causal, scale)
        o.backward(do.cuda())
        assert o.shape == o_w.shape and o.is_contiguous()
        assert qg.grad.shape == q.shape and kg.grad.shape == k.shape and vg.grad.shape == v.shape
        assert (o.float().cpu() - o_w).abs().max().item() <= 2e-2, (Lq, Lk)
        errs = (_rel(qg.grad, dq_w), _rel(kg.grad, dk_w), _rel(vg.grad, dv_w))
        assert max(errs) <= 5e-2, (Lq, Lk, errs)


@pytest.mark.parametrize("causal,dk,dv", [(False, 64, 128), (False, 128, 128), (True, 128, 128), (True, 64, 64)])
def test_async_staged_kernels_repeat_bit_for_bit(causal, dk, dv):
    """The kernels are deterministic, so a chunk read before its asynchronous copy has landed (or overwritten while it is
    still being read) shows as a difference between repeats: 25 forward + backward passes over many chunks (two chunk
    buffers at 64/128 forward and at 128/128, three elsewhere) must all equal the first, bit for bit."""
    B, H, L = 2, 8, 4096
    q, k, v, do = (t.cuda() for t in orc.make_qkv(77, B, H, L, L, dk, dv, torch.bfloat16))
    scale = 1 / math.sqrt(dk)
    first = None
    for _ in range(25):
        qg, kg, vg = (t.detach().requires_grad_(True) for t in (q, k, v))
        o, M = _fa()._forward(qg.detach(), kg.detach(), vg.detach(), causal, scale)
        o2 = _fa().attention(qg, kg, vg, causal, scale)
        o2.backward(do)
        got = (o, M, o2.detach(), qg.grad, kg.grad, vg.grad)
        if first is None:
            first = got
        else:
            for a, b in zip(first, got):
                assert torch.equal(a, b)


@pytest.mark.parametrize("causal", [False, True])
def test_views_of_a_packed_projection(causal):
    """q, k, v as strided views of one packed [B, L, H, dk + dk + dv] projection output (token stride H (2 dk + dv), head
    stride 2 dk + dv) and a transposed upstream gradient: the asynchronously staged kernels address tokens by stride."""
    B, H, L, dk, dv = 2, 3, 200, 64, 128
    g = torch.Generator().manual_seed(11)
    packed = torch.randn(B, L, H, 2 * dk + dv, generator=g).to(torch.bfloat16)
    do = torch.randn(B, L, H, dv, generator=g).to(torch.bfloat16)
    scale = 1 / math.sqrt(dk)
    views = lambda t: (t[..., :dk].permute(0, 2, 1, 3), t[..., dk:2 * dk].permute(0, 2, 1, 3), t[..., 2 * dk:].permute(0, 2, 1, 3))
    q, k, v = views(packed)
    o_w, dq_w, dk_w, dv_w = orc.flash_grads(q.float().contiguous(), k.float().contiguous(), v.float().contiguous(),
                                            do.permute(0, 2, 1, 3).float().contiguous(), causal, scale)
    pg = packed.cuda().requires_grad_(True)
    qg, kg, vg = views(pg)
    assert not qg.is_contiguous()
    o = _fa().attention(qg, kg, vg, causal, scale)
    o.backward(do.cuda().permute(0, 2, 1, 3))
    assert (o.float().cpu() - o_w).abs().max().item() <= 2e-2
    got = views(pg.grad)
    errs = (_rel(got[0], dq_w), _rel(got[1], dk_w), _rel(got[2], dv_w))
    assert max(errs) <= 5e-2, errs


def test_bad_arguments_raise():
    from dl_templates_amd._lib import DltError
    q = torch.randn(1, 1, 64, 64, dtype=torch.bfloat16).cuda()
    k = torch.randn(1, 1, 128, 64, dtype=torch.bfloat16).cuda()
    with pytest.raises(DltError):
        _fa().attention(q, k, k, True, 1.0)  # causal needs Lq == Lk
    with pytest.raises(AssertionError):
        _fa().attention(q, k[..., :32], k, False, 1.0)


def test_gradients_that_cancel_stay_zero_with_fp32_inputs():
    """A query that sees a single key has p = 1 and dS = dP - delta = 0, so dq = dk = 0.  fp32 operands of the second
    products are rounded to bf16 on load: delta is formed from the same rounded dO as dP, or the difference of the two
    roundings (about 1e-1 at head dim 256) would show up as a gradient; and the backward kernels recompute the scores from
    the same hi + lo pairs as the forward kernel, so p is 1 and not exp of a rounding difference."""
    fa = _fa()
    q, k, v, do = orc.make_qkv(31, 2, 2, 200, 1, 120, 256, torch.float32)
    qg, kg, vg = (t.cuda().requires_grad_(True) for t in (q, k, v))
    o = fa.attention(qg, kg, vg, False, 0.3)
    o.backward(do.cuda())
    assert qg.grad.abs().max().item() <= 1e-4 and kg.grad.abs().max().item() <= 1e-3
    want = do.bfloat16().float().sum(dim=2, keepdim=True)        # dv = sum over the queries of the rounded dO
    assert (vg.grad.cpu() - want).abs().max().item() <= 1e-3 * want.abs().max().item()


# calls whose own blocks do not fill the chip run on the kernels that split the streamed side over the waves of a workgroup:
# fewer blocks than waves, remainders of 16 and of 32 tokens, one and two own blocks, every head-dim class, dims below a class
@pytest.mark.parametrize("causal,Lq,Lk,dk,dv,B,H", [
    (False, 1, 900, 64, 64, 1, 2), (False, 77, 1500, 64, 64, 1, 3), (False, 33, 255, 64, 128, 2, 2), (False, 16, 257, 128, 128, 1, 2), (False, 40, 31, 32, 32, 1, 2),
    (False, 900, 17, 64, 64, 1, 2), (False, 1100, 40, 128, 128, 1, 2), (False, 130, 600, 80, 80, 1, 3), (False, 600, 100, 24, 16, 2, 2), (False, 1000, 1000, 64, 64, 1, 8),
    (True, 1, 1, 64, 64, 1, 2), (True, 221, 221, 64, 64, 1, 4), (True, 255, 255, 128, 128, 1, 2), (True, 513, 513, 64, 128, 1, 2), (True, 97, 97, 40, 32, 1, 2),
    (True, 1030, 1030, 32, 32, 1, 8),
    # 8 waves of one own block (slim) and, with slabs that fill the chip, two own blocks per wave: chunk and block remainders
    (False, 300, 193, 64, 128, 2, 40), (True, 270, 270, 128, 128, 2, 40), (True, 257, 257, 64, 128, 2, 50), (False, 129, 65, 64, 128, 4, 70),
    (False, 257, 63, 128, 128, 3, 90), (True, 130, 130, 64, 64, 5, 110), (False, 40, 127, 80, 80, 4, 70), (True, 150, 150, 128, 128, 6, 90)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_streamed_side_split_over_waves(causal, Lq, Lk, dk, dv, B, H, dtype):
    q, k, v, do = orc.make_qkv(Lq + 2 * Lk + dk, B, H, Lq, Lk, dk, dv, dtype)
    scale = 1 / math.sqrt(dk)
    o_w, dq_w, dk_w, dv_w = orc.flash_grads(q.float(), k.float(), v.float(), do.float(), causal, scale)
    outs = []
    for _ in range(2):
        qg, kg, vg = (t.cuda().requires_grad_(True) for t in (q, k, v))
        o = _fa().attention(qg, kg, vg, causal, scale)
        o.backward(do.cuda())
        outs.append((o.detach(), qg.grad, kg.grad, vg.grad))
    assert all(torch.equal(a, b) for a, b in zip(*outs))
    assert (outs[0][0].float().cpu() - o_w).abs().max().item() <= 2e-2
    errs = [_rel(g, w) for g, w in zip(outs[0][1:], (dq_w, dk_w, dv_w))]
    assert max(errs) <= 5e-2, errs
    _, M = _fa()._forward(q.cuda(), k.cuda(), v.cuda(), causal, scale)
    assert (M.cpu() - orc.flash_lse2(q, k, scale, causal)).abs().max().item() <= 2e-2


# one rule picks the order of summation from the shape of a slab: shapes on both sides of it in every head-dim class, the slab counts on both
# sides of the choices that are left (one or two own blocks per split workgroup, slim or chunked workgroups)
@pytest.mark.parametrize("causal,Lq,Lk,dk,dv,counts", [
    (False, 77, 1500, 64, 64, (1, 16, 130)), (False, 40, 700, 128, 128, (1, 100)), (False, 500, 60, 64, 128, (1, 40)), (False, 33, 300, 32, 32, (1, 300)),
    (False, 1000, 1000, 64, 64, (1, 8, 70)), (False, 600, 2500, 64, 128, (1, 12, 60)), (False, 700, 700, 80, 80, (1, 50)), (False, 1200, 300, 128, 128, (1, 30)),
    (True, 90, 90, 64, 64, (1, 200)), (True, 255, 255, 128, 128, (1, 70)), (True, 513, 513, 64, 128, (1, 8, 70)), (True, 1030, 1030, 64, 64, (1, 9, 40)),
    (True, 1100, 1100, 128, 128, (1, 16, 40)), (True, 300, 300, 40, 24, (1, 150)), (True, 2000, 2000, 64, 64, (1, 40)), (True, 1800, 1800, 64, 128, (1, 20, 40))])
def test_a_slab_has_the_same_bits_in_any_call(causal, Lq, Lk, dk, dv, counts):
    scale = 1 / math.sqrt(dk)
    gen = torch.Generator(device="cuda").manual_seed(Lq + Lk)
    full = [torch.randn(1, max(counts), n, d, generator=gen, device="cuda").to(torch.bfloat16) for n, d in ((Lq, dk), (Lk, dk), (Lk, dv), (Lq, dv))]
    runs = []
    for n in counts:
        q, k, v = (t[:, -n:].contiguous().requires_grad_(True) for t in full[:3])
        o = _fa().attention(q, k, v, causal, scale)
        _, M = _fa()._forward(q.detach(), k.detach(), v.detach(), causal, scale)
        runs.append((o.detach(), M) + torch.autograd.grad(o, (q, k, v), full[3][:, -n:].contiguous()))
    for run in runs[1:]:
        m = min(counts)
        assert [torch.equal(a[:, -m:], b[:, -m:]) for a, b in zip(runs[0], run)] == [True] * 5
    for a, b in zip(runs[-2], runs[-1]):
        n = counts[-2]
        assert torch.equal(a[:, -n:], b[:, -n:])


# backward passes with one own block per wave: 4 waves while their workgroups of 64 fit the chip, without a mask dQ on 8 waves while its workgroups
# of 128 do, two blocks per wave beyond: a token past a workgroup's end, chunk remainders, every class and dims below it, counts on every side of the lines
@pytest.mark.parametrize("causal,Lq,Lk,dk,dv,counts", [
    (False, 1025, 1090, 64, 64, (1, 20, 40)), (False, 1090, 1025, 64, 128, (1, 20, 40)), (False, 1100, 1153, 128, 128, (1, 20, 40)),
    (False, 1030, 1100, 80, 72, (1, 20, 40)), (True, 1090, 1090, 64, 64, (1, 35)), (True, 1090, 1090, 64, 128, (1, 40)),
    (True, 1121, 1121, 128, 128, (1, 35)), (True, 3100, 3100, 64, 128, (1, 12))])
def test_one_own_block_per_wave_backward(causal, Lq, Lk, dk, dv, counts):
    scale = 1 / math.sqrt(dk)
    q, k, v, do = orc.make_qkv(Lq + Lk + dk, 1, 1, Lq, Lk, dk, dv, torch.bfloat16)
    want = orc.flash_grads(q.float(), k.float(), v.float(), do.float(), causal, scale)[1:]
    qg, kg, vg = (t.cuda().requires_grad_(True) for t in (q, k, v))
    got = torch.autograd.grad(_fa().attention(qg, kg, vg, causal, scale), (qg, kg, vg), do.cuda())
    assert max(_rel(g, w) for g, w in zip(got, want)) <= 5e-2
    test_a_slab_has_the_same_bits_in_any_call(causal, Lq, Lk, dk, dv, counts)


# head dims of up to 96 and of up to 80 in the classes of 128 run without the dims beyond: on both sides of those lines, in each tensor, with one and with
# several workgroups per CU, a token past a workgroup's and a chunk's end
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("dk,dv", [(96, 96), (72, 96), (96, 40), (104, 96), (96, 104), (64, 96), (40, 72), (64, 104), (80, 80), (80, 40), (88, 80), (80, 88), (64, 80),
                                   (64, 88)])
def test_head_dims_of_up_to_96(dk, dv, causal):
    L, scale = 1025, 1 / math.sqrt(dk)
    q, k, v, do = orc.make_qkv(dk + dv, 1, 1, L, L, dk, dv, torch.float16)
    want = orc.flash_grads(q.float(), k.float(), v.float(), do.float(), causal, scale)
    for slabs in (1, 20, 40):
        leaves = [t.cuda().repeat(1, slabs, 1, 1).requires_grad_(True) for t in (q, k, v)]
        o = _fa().attention(*leaves, causal, scale)
        got = (o,) + torch.autograd.grad(o, leaves, do.cuda().repeat(1, slabs, 1, 1))
        for g, w in zip(got, want):
            assert torch.equal(g, g[:, :1].expand_as(g))
            assert _rel(g[:, :1], w) <= 1e-2


# other sides cut into shares over several workgroups: a token past a share's end and one before it, a last share of a few tokens, own sides that
# end inside a workgroup, every class, 2 ... 8 shares, one own block per wave and two
@pytest.mark.parametrize("Lq,Lk,dk,dv,counts", [
    (33, 3073, 64, 64, (1, 20)), (129, 3201, 64, 128, (1, 40)), (128, 1281, 128, 128, (1, 90)), (300, 2500, 80, 72, (1, 60)), (700, 4097, 64, 64, (1, 30)),
    (2600, 90, 64, 64, (1, 40)), (1700, 65, 64, 128, (1, 90)), (1281, 130, 128, 128, (1, 40)), (2100, 200, 96, 40, (1, 60)), (64, 2000, 104, 128, (1, 16))])
def test_other_side_in_shares(Lq, Lk, dk, dv, counts):
    scale = 1 / math.sqrt(dk)
    q, k, v, do = orc.make_qkv(Lq + Lk + dk, 1, 1, Lq, Lk, dk, dv, torch.float16)
    want = orc.flash_grads(q.float(), k.float(), v.float(), do.float(), False, scale)
    leaves = [t.cuda().requires_grad_(True) for t in (q, k, v)]
    o = _fa().attention(*leaves, False, scale)
    # fp16 probabilities and results: 1e-2 of the largest value, as for the other kernels
    for g, w in zip((o,) + torch.autograd.grad(o, leaves, do.cuda()), want):
        assert _rel(g, w) <= 1e-2
    _, M = _fa()._forward(q.cuda(), k.cuda(), v.cuda(), False, scale)
    assert (M.cpu() - orc.flash_lse2(q, k, scale, False)).abs().max().item() <= 2e-2
    test_a_slab_has_the_same_bits_in_any_call(False, Lq, Lk, dk, dv, counts)


# a share whose scores are all -inf or hold NaN / inf, and an infinite key in one share: what the whole row gives
def test_shares_with_infinite_and_nan_scores():
    Lq, Lk, d = 40, 3001, 64
    q, k, v, _ = (t.cuda() for t in orc.make_qkv(3, 1, 4, Lq, Lk, d, d, torch.float16))
    q[:, :, :, 0] = 1.0
    k[:, 1, :1500, 0] = -float("inf")     # the first shares of head 1 score -inf
    k[:, 2, 7, 0] = float("nan")
    v[:, 3, 2990, 5] = float("inf")
    o, M = _fa()._forward(q, k, v, False, 0.125)
    kf, vf = k[:, 1, 1500:].float(), v[:, 1, 1500:].float()
    want = torch.softmax(torch.matmul(q[:, 1].float(), kf.transpose(-1, -2).contiguous()) * 0.125, -1) @ vf
    assert torch.isfinite(M[:, :2]).all() and _rel(o[:, 1], want.cpu()) <= 1e-2
    assert torch.isnan(o[:, 2]).all() and torch.isinf(o[:, 3, :, 5]).all() and torch.isfinite(o[:, 3, :, :5]).all() and torch.isfinite(o[:, 0]).all()


# forward passes with one own block per wave, 4 waves or 8, 64-key chunks and (from 3072 queries on, 64/128 and 128/128) 128-key ones: counts on every side
# of the lines, chunk remainders, a token past a workgroup's end, every class and dims below it
@pytest.mark.parametrize("causal,Lq,Lk,dk,dv,counts", [
    (False, 1030, 705, 64, 64, (1, 15, 16)), (False, 705, 1090, 128, 128, (1, 21, 22)), (False, 3100, 193, 64, 128, (1, 6, 12)), (False, 3073, 260, 96, 104, (1, 6, 12)),
    (False, 3137, 129, 80, 80, (1, 5, 12)), (True, 1030, 1030, 64, 64, (1, 30, 31)), (True, 800, 800, 48, 128, (1, 39, 40)), (True, 3100, 3100, 64, 128, (1, 6, 21)),
    (True, 3073, 3073, 128, 128, (1, 6, 21)), (True, 3201, 3201, 80, 72, (1, 5, 21))])
def test_one_own_block_per_wave_forward(causal, Lq, Lk, dk, dv, counts):
    scale = 1 / math.sqrt(dk)
    q, k, v, _ = (t.cuda() for t in orc.make_qkv(Lq + Lk + dk, 1, max(counts), Lq, Lk, dk, dv, torch.float16))
    o, M = _fa()._forward(q, k, v, causal, scale)
    s = torch.matmul(q[:, -1].float(), k[:, -1].float().transpose(-1, -2).contiguous()) * scale
    if causal:
        s = s.masked_fill(torch.ones(Lq, Lk, dtype=torch.bool, device="cuda").triu(1), -math.inf)
    assert _rel(o[:, -1], (torch.softmax(s, -1) @ v[:, -1].float()).cpu()) <= 1e-2
    assert (M[:, -1] - torch.logsumexp(s, -1) / math.log(2)).abs().max().item() <= 2e-2
    for n in counts[:-1]:
        got = _fa()._forward(q[:, -n:].contiguous(), k[:, -n:].contiguous(), v[:, -n:].contiguous(), causal, scale)
        assert torch.equal(got[0], o[:, -n:]) and torch.equal(got[1], M[:, -n:])


# dense split forward passes whose workgroups take a half or a quarter of the output dims: counts on both sides of the lines (256 CUs; 5 blocks of 16
# queries to a slab), dims that fill the last part or not, a last part of one vector, the remainders of 32-key blocks
@pytest.mark.parametrize("Lk", [1500, 2017])
@pytest.mark.parametrize("dk,dv,counts", [(64, 64, (1, 25, 26)), (40, 40, (1, 25, 26)), (64, 128, (1, 12, 13, 25, 26)), (64, 72, (1, 17, 18, 25, 26)),
                                          (128, 128, (1, 12, 13, 25, 26)), (80, 80, (1, 17, 18, 25, 26)), (128, 104, (1, 12, 25, 26)), (128, 24, (1, 26))])
def test_output_dims_over_workgroups(dk, dv, counts, Lk):
    Lq, scale = 77, 1 / math.sqrt(dk)
    q, k, v, _ = (t.cuda() for t in orc.make_qkv(Lk + dk + dv, 1, max(counts), Lq, Lk, dk, dv, torch.bfloat16))
    o, M = _fa()._forward(q, k, v, False, scale)
    s = torch.matmul(q.float(), k.float().transpose(-1, -2).contiguous()) * scale
    assert _rel(o, (torch.softmax(s, -1) @ v.float()).cpu()) <= 2e-2
    assert (M - torch.logsumexp(s, -1) / math.log(2)).abs().max().item() <= 4e-2
    for n in counts[:-1]:
        got = _fa()._forward(q[:, :n].contiguous(), k[:, :n].contiguous(), v[:, :n].contiguous(), False, scale)
        assert torch.equal(got[0], o[:, :n]) and torch.equal(got[1], M[:, :n])


# dense passes in shares: split over workgroups on few slabs, walked by one workgroup once the chip is full (192 workgroups of up to 64 own tokens, 384 of more), with the
# same bits as a slab alone; forward, dQ and dK/dV in shares, every class and dims below it, own tokens of one wave and past a workgroup's end, last shares of one token and of one
# chunk, one full and one short; an infinite score, an infinite value and NaN in one slab
@pytest.mark.parametrize("Lq,Lk,dk,dv,counts", [
    (64, 3073, 64, 64, (2, 191, 192)), (19, 3300, 64, 128, (2, 191, 192)), (37, 2600, 80, 80, (2, 200)), (64, 1281, 128, 128, (2, 200)), (130, 3200, 64, 64, (2, 127, 128)),
    (70, 3585, 48, 40, (2, 200)), (100, 3137, 64, 128, (2, 191, 192)), (129, 2700, 96, 88, (2, 130)), (90, 1300, 128, 104, (2, 200)), (1700, 70, 64, 64, (2, 191, 192)),
    (2600, 19, 64, 64, (2, 200)), (1665, 40, 64, 128, (2, 200)), (2100, 90, 80, 72, (2, 200)), (1300, 33, 128, 128, (2, 200)), (2561, 200, 48, 64, (2, 100))])
def test_shares_walked_by_one_workgroup(Lq, Lk, dk, dv, counts):
    scale = 1 / math.sqrt(dk)
    q, k, v, do = (t.cuda() for t in orc.make_qkv(Lq + Lk + dk, 1, 3, Lq, Lk, dk, dv, torch.bfloat16))
    want = orc.flash_grads(*(t[:, :1].float().cpu() for t in (q, k, v, do)), False, scale)
    k[:, 2, Lk // 2, 0], v[:, 2, Lk - 1, 3], q[:, 2, 0, 1] = float("inf"), float("inf"), float("nan")

    def run(slabs):   # the first, as often as asked, and the two others
        args = [torch.cat([t[:, :1].expand(-1, slabs - 2, -1, -1), t[:, 1:]], 1) if slabs > 2 else t[:, :2] for t in (q, k, v, do)]
        leaves = [t.detach().contiguous().requires_grad_(True) for t in args[:3]]
        o = _fa().attention(*leaves, False, scale)
        _, M = _fa()._forward(*(t.detach() for t in leaves), False, scale)
        return (o.detach(), M) + torch.autograd.grad(o, leaves, args[3].contiguous())

    few, runs = run(3), [run(n) for n in counts]
    assert (few[0][:, :1].float().cpu() - want[0]).abs().max().item() <= 2e-2 and max(_rel(g[:, :1], w) for g, w in zip(few[2:], want[1:])) <= 5e-2
    for n, got in zip(counts, runs):
        for a, b in zip(got, few):
            assert torch.equal(a[:, :1], b[:, :1])
            if n > 2:
                assert torch.equal(a[:, :-2], b[:, :1].expand_as(a[:, :-2])) and torch.equal(a[:, -2], b[:, 1]) and torch.equal(a[:, -1].isfinite(), b[:, 2].isfinite())
                assert torch.equal(a[:, -1].nan_to_num(), b[:, 2].nan_to_num())
