"""GPU parity of the sliding-window attention over tiles of 16 k tokens (b_size a multiple of 16:
the regime of the reference's large kernels and of its demo, src/tiled_swa.py:142-244, :736-750),
which runs on the flash kernels in tile mode: forward and backward through TiledSwa against the
CPU oracle, at the stated tolerances (forward max-abs <= 2e-2, gradients relative <= 5e-2).
"""
import math

import pytest
import torch

from oracle import attn_oracle as orc

pytestmark = pytest.mark.gpu

FWD_TOL, GRAD_TOL = 2e-2, 5e-2


def _swa():
    from dl_templates_amd import tiled_swa
    return tiled_swa


def _rel(got, want):
    return ((got.float().cpu() - want).abs().max() / want.abs().max().clamp_min(1e-3)).item()


CASES = [
    # B, H, th, tw, S, WR, WC, dk, dv, dtype
    (1, 2, 16, 16, 16, 1, 1, 32, 32, torch.float16),    # the reference demo shape, reduced batch
    (1, 2, 5, 7, 16, 1, 2, 64, 64, torch.bfloat16),     # row of 112 tokens: shorter than one 128-token block
    (1, 1, 3, 9, 32, 2, 1, 64, 128, torch.bfloat16),    # distinct head dims, 288 tokens per row
    (2, 1, 4, 4, 48, 1, 1, 128, 128, torch.bfloat16),   # tiles of 48: multiple of 16 but not of 32
    (1, 2, 6, 6, 64, 1, 1, 32, 32, torch.float16),      # one tile = one wave's worth of two blocks
    (1, 1, 2, 3, 16, 5, 5, 64, 64, torch.bfloat16),     # window larger than the grid: dense
    (1, 1, 1, 1, 16, 0, 0, 64, 64, torch.bfloat16),     # a single tile
    (1, 2, 4, 20, 16, 0, 3, 64, 64, torch.bfloat16),    # window of one row, 320 tokens per row (2.5 blocks)
    (1, 1, 7, 5, 80, 3, 0, 16, 16, torch.float16),      # window of one column, head dim below 32
]


@pytest.mark.parametrize("B,H,th,tw,S,WR,WC,dk,dv,dtype", CASES)
def test_tile_windows_forward_backward(B, H, th, tw, S, WR, WC, dk, dv, dtype):
    sw = _swa()
    N = th * tw * S
    q, k, v, do = orc.make_qkv(N + dk + S, B, H, N, N, dk, dv, dtype)
    scale = 1 / math.sqrt(dk)
    o_w, dq_w, dk_w, dv_w = orc.tiled_swa_grads(q.float(), k.float(), v.float(), do.float(), S, th, tw, WR, WC, scale)
    qg, kg, vg = (t.cuda().requires_grad_(True) for t in (q, k, v))
    o = sw.TiledSwa.apply(qg, kg, vg, S, th, tw, WR, WC, scale)
    o.backward(do.cuda())
    assert o.shape == (B, H, N, dv) and o.dtype == dtype
    assert (o.float().cpu() - o_w).abs().max().item() <= FWD_TOL
    errs = (_rel(qg.grad, dq_w), _rel(kg.grad, dk_w), _rel(vg.grad, dv_w))
    assert max(errs) <= GRAD_TOL, errs


def test_tile_mode_matches_generic_kernels_bitwise_close():
    """Two independent GPU implementations: fp32 inputs take the generic kernels (bf16 arithmetic),
    the same values as bf16 take the flash kernels in tile mode."""
    sw = _swa()
    B, H, th, tw, S, W, d = 1, 2, 8, 8, 16, 1, 64
    N = th * tw * S
    q, k, v, do = orc.make_qkv(99, B, H, N, N, d, d, torch.bfloat16)
    outs = []
    for dt in (torch.bfloat16, torch.float32):
        qg, kg, vg = (t.to(dt).cuda().requires_grad_(True) for t in (q, k, v))
        o = sw.TiledSwa.apply(qg, kg, vg, S, th, tw, W, W, 0.125)
        o.backward(do.to(dt).cuda())
        outs.append((o.float(), qg.grad.float(), kg.grad.float(), vg.grad.float()))
    for a, b in zip(*outs):
        assert (a - b).abs().max().item() <= 2e-2 * max(1.0, b.abs().max().item())


# tiles of fewer than 16 tokens (the reference's small-tile regime, src/tiled_swa.py:611: b_size < 16): the streaming
# token-grid kernels on the grid of token slots, a token's window given by its tile
SMALL = [
    # B, H, th, tw, S, WR, WC, d, dtype
    (1, 2, 9, 11, 4, 1, 1, 64, torch.bfloat16),      # 2 x 2-pixel tiles, 3 x 3 tile window
    (1, 2, 7, 5, 9, 1, 1, 128, torch.bfloat16),      # 3 x 3-pixel tiles
    (2, 1, 12, 6, 2, 3, 2, 64, torch.float16),
    (1, 1, 5, 9, 3, 0, 2, 128, torch.float16),       # window of one row
    (1, 2, 6, 4, 8, 2, 1, 64, torch.bfloat16),
    (1, 1, 4, 3, 15, 1, 1, 64, torch.bfloat16),      # 45-slot windows: two column passes
    (1, 1, 3, 2, 12, 4, 4, 128, torch.bfloat16),     # window larger than the grid
    (1, 2, 20, 1, 5, 2, 0, 64, torch.bfloat16),      # one tile per row
]


@pytest.mark.parametrize("B,H,th,tw,S,WR,WC,d,dtype", SMALL)
def test_small_tiles_forward_backward(B, H, th, tw, S, WR, WC, d, dtype):
    from dl_templates_amd import _lib
    sw = _swa()
    N = th * tw * S
    q, k, v, do = orc.make_qkv(N + d + S, B, H, N, N, d, d, dtype)
    scale = 1 / math.sqrt(d)
    o_w, dq_w, dk_w, dv_w = orc.tiled_swa_grads(q.float(), k.float(), v.float(), do.float(), S, th, tw, WR, WC, scale)
    qg, kg, vg = (t.cuda().requires_grad_(True) for t in (q, k, v))
    o = sw.TiledSwa.apply(qg, kg, vg, S, th, tw, WR, WC, scale)
    assert _lib.KERNEL_FAMILIES[_lib.load().dlt_last_kernel_family()] == "streaming"
    o.backward(do.cuda())
    assert _lib.KERNEL_FAMILIES[_lib.load().dlt_last_kernel_family()] == "streaming"
    assert (o.float().cpu() - o_w).abs().max().item() <= FWD_TOL
    errs = (_rel(qg.grad, dq_w), _rel(kg.grad, dk_w), _rel(vg.grad, dv_w))
    assert max(errs) <= GRAD_TOL, errs


# the marching tile-window kernels (tiles of 16 or 32 tokens, head dim 32 / 64): every instantiated window, single rows and
# columns, strips of 8 blocks with a remainder, grids smaller than the window, bands of one and of many rows
MARCH = [(1, 1, 1, 16, 1, 1, 32), (1, 1, 9, 16, 1, 1, 64), (9, 1, 1, 16, 1, 1, 32), (7, 8, 1, 16, 1, 1, 64), (5, 9, 2, 16, 1, 2, 32), (6, 17, 1, 16, 1, 2, 64),
         (7, 10, 1, 16, 2, 1, 32), (9, 11, 1, 16, 2, 2, 32), (2, 2, 2, 16, 2, 2, 32), (5, 5, 1, 32, 1, 1, 32), (4, 9, 2, 32, 1, 1, 64), (11, 3, 40, 16, 1, 1, 32)]


@pytest.mark.parametrize("th,tw,B,S,WR,WC,d", MARCH)
@pytest.mark.parametrize("image", [False, True])
def test_marching_tile_windows(th, tw, B, S, WR, WC, d, image):
    sw = _swa()
    H, N, dt = 3, th * tw * S, torch.bfloat16 if tw % 2 else torch.float16
    q, k, v, do = orc.make_qkv(N + S + d, B, H, N, N, d, d, dt)
    o_w, dq_w, dk_w, dv_w = orc.tiled_swa_grads(q.float(), k.float(), v.float(), do.float(), S, th, tw, WR, WC, 0.2)
    lay = (lambda t: orc.tokens_to_image(t, th, tw, 4, S // 4).contiguous()) if image else (lambda t: t)
    qg, kg, vg = (lay(t).cuda().requires_grad_(True) for t in (q, k, v))
    o = sw.TiledSwaImage.apply(qg, kg, vg, 4, S // 4, WR, WC, 0.2) if image else sw.TiledSwa.apply(qg, kg, vg, S, th, tw, WR, WC, 0.2)
    o.backward(lay(do).cuda())
    assert (o.float().cpu() - lay(o_w)).abs().max().item() <= FWD_TOL
    errs = (_rel(qg.grad, lay(dq_w)), _rel(kg.grad, lay(dk_w)), _rel(vg.grad, lay(dv_w)))
    assert max(errs) <= GRAD_TOL, errs


# the one-launch backward pass (16-token tiles, 3 x 3 window) stages K, V, Q and dO side by side and o behind them: strips of 128
# (d = 32) and 64 (d = 64) tokens with one block left over, every tensor with strides of its own, same bits as contiguous tensors
@pytest.mark.parametrize("th,tw,d", [(3, 9, 32), (2, 5, 64), (21, 8, 32)])
def test_one_launch_backward_takes_each_tensors_own_strides(th, tw, d):
    sw = _swa()
    B, H, S = 2, 3, 16
    N = th * tw * S
    q, k, v, do = (t.cuda() for t in orc.make_qkv(N + d, B, H, N, N, d, d, torch.bfloat16))
    as_bnhd = lambda t: t.transpose(1, 2).contiguous().transpose(1, 2)
    padded = lambda t: torch.cat([t, t[..., :8]], dim=-1)[..., :d]
    spaced = lambda t: torch.stack([t, t], dim=2)[:, :, 0]

    def grads(q, k, v, do):
        leaves = [t.detach().requires_grad_(True) for t in (q, k, v)]
        return torch.autograd.grad(sw.TiledSwa.apply(*leaves, S, th, tw, 1, 1, 0.2), leaves, do)

    want = grads(q, k, v, do)
    got = grads(as_bnhd(q), padded(k), spaced(v), as_bnhd(padded(do)))
    assert all(torch.equal(a, b) for a, b in zip(got, want))


# narrow grids at d = 32: two backward launches from 12 rows per CU on (256 CUs), one below and from 6 tile columns on (images: 3); the same bits
@pytest.mark.parametrize("image", [False, True])
@pytest.mark.parametrize("tw", [1, 2, 3, 5, 6])
def test_narrow_grids_backward(tw, image):
    sw = _swa()
    th, H, S, d = 13, 4, 16, 32
    N = th * tw * S
    q, k, v, do = orc.make_qkv(tw, 1, H, N, N, d, d, torch.float16)
    want = orc.tiled_swa_grads(q.float(), k.float(), v.float(), do.float(), S, th, tw, 1, 1, 0.2)[1:]

    def grads(B):
        lay = (lambda t: orc.tokens_to_image(t, th, tw, 4, 4)) if image else (lambda t: t)
        q_, k_, v_, do_ = (lay(t.cuda().repeat(B, 1, 1, 1)).contiguous() for t in (q, k, v, do))
        leaves = [t.requires_grad_(True) for t in (q_, k_, v_)]
        o = sw.TiledSwaImage.apply(*leaves, 4, 4, 1, 1, 0.2) if image else sw.TiledSwa.apply(*leaves, S, th, tw, 1, 1, 0.2)
        got = torch.autograd.grad(o, leaves, do_)
        assert all(torch.equal(g, g[:1].expand_as(g)) for g in got)
        return [g[:1].clone() for g in got]

    few, many = grads(2), grads(61)
    assert all(torch.equal(a, b) for a, b in zip(few, many))
    lay = (lambda t: orc.tokens_to_image(t, th, tw, 4, 4)) if image else (lambda t: t)
    assert max(_rel(g, lay(w)) for g, w in zip(many, want)) <= GRAD_TOL


# the one-launch backward pass over bands longer than its ring of 3 rows (tests/test_geom_cpu.py checks the plan of these shapes at 256 CUs): several
# strips, the last one ragged.  th, tw, slabs, d
LONG_BANDS = [(11, 9, 100, 64), (11, 9, 130, 32), (23, 17, 40, 64), (23, 12, 64, 32)]


@pytest.mark.parametrize("th,tw,slabs,d", LONG_BANDS)
@pytest.mark.parametrize("image", [False, True])
def test_one_launch_backward_over_long_bands(th, tw, slabs, d, image):
    sw = _swa()
    S, H = 16, 2
    gen = torch.Generator(device="cuda").manual_seed(th + tw + d)
    q, k, v, do = (torch.randn((slabs // H, H, th * tw * S, d), generator=gen, device="cuda").bfloat16() for _ in range(4))
    lay = (lambda t: orc.tokens_to_image(t, th, tw, 4, 4).contiguous()) if image else (lambda t: t)
    leaves = [lay(t).requires_grad_(True) for t in (q, k, v)]
    o = sw.TiledSwaImage.apply(*leaves, 4, 4, 1, 1, 0.2) if image else sw.TiledSwa.apply(*leaves, S, th, tw, 1, 1, 0.2)
    got = (o,) + torch.autograd.grad(o, leaves, lay(do))
    for b in (0, slabs // H - 1):
        one = slice(b, b + 1)
        want = orc.tiled_swa_grads(*(t[one, :1].float().cpu() for t in (q, k, v, do)), S, th, tw, 1, 1, 0.2)
        mine = [g[one, ..., :1, :] if image else g[one, :1] for g in got]
        assert (mine[0].float().cpu() - lay(want[0])).abs().max().item() <= FWD_TOL
        errs = [_rel(g, lay(w)) for g, w in zip(mine[1:], want[1:])]
        assert max(errs) <= GRAD_TOL, errs


# infinite and NaN tiles reach the tiles that see them (and, through a query, that query's other keys) and no others, bit for bit: the
# rows and columns outside the grid that the ring stages in their place are tiles of the window
@pytest.mark.parametrize("d,th,tw,B", [(32, 7, 9, 1), (64, 7, 9, 1), (32, 13, 3, 122)])
@pytest.mark.parametrize("which", ["q", "k", "v", "do"])
def test_infinite_and_nan_tiles_stay_in_their_windows(d, th, tw, B, which):
    sw = _swa()
    S, H = 16, 2
    gen = torch.Generator(device="cuda").manual_seed(d)
    base = dict(zip(("q", "k", "v", "do"), (torch.randn((B, H, th * tw * S, d), generator=gen, device="cuda").half() for _ in range(4))))

    def grads(t):
        leaves = [t[n].clone().requires_grad_(True) for n in ("q", "k", "v")]
        return torch.autograd.grad(sw.TiledSwa.apply(*leaves, S, th, tw, 1, 1, 0.2), leaves, t["do"])

    clean = grads(base)
    assert all(torch.isfinite(g).all() for g in clean)
    # how far a tile's values reach in dq, dk and dv (tiles; -1: not at all): dv holds probabilities and dO only
    reach = {"q": (0, 1, 1), "k": (1, 2, 2), "v": (1, 2, -1), "do": (0, 1, 1)}[which]
    for r, c in ((th // 2, tw // 2), (0, 0), (th - 1, tw - 1), (0, tw - 1)):
        for value in (float("inf"), float("-inf"), float("nan")):
            bad = dict(base, **{which: base[which].clone()})
            at = ((r * tw + c) * S + 5, (r * tw + c) * S + 11)
            bad[which][..., at[0], 3] = value
            bad[which][..., at[1], d - 1] = value
            rows, cols = torch.meshgrid(torch.arange(th), torch.arange(tw), indexing="ij")
            far = torch.maximum((rows - r).abs(), (cols - c).abs()).reshape(-1).repeat_interleave(S).cuda()
            for g, w, n in zip(grads(bad), clean, reach):
                assert torch.equal(g[:, :, far > n], w[:, :, far > n]), (r, c, value)


# few tiles of 16 k tokens: 16 own tokens to a workgroup, the window's keys dealt over its waves; one slab, and as many as leave that rule (whose bits are
# others, but at five tile rows or columns where strips of four take the pass).  Odd and even
# numbers of 16-token runs, runs of one, windows of one tile and beyond the grid, every class and dims below it.  The image layout has the same bits.
# A tile of infinities and NaN is not read for the tiles that do not see it
@pytest.mark.parametrize("th,tw,S,WR,WC,dk,dv,many", [
    (7, 5, 16, 2, 2, 64, 64, 40), (4, 10, 16, 2, 1, 64, 64, 60), (5, 9, 16, 0, 0, 64, 64, 90), (3, 7, 16, 1, 1, 128, 128, 40), (1, 9, 16, 4, 3, 64, 128, 60),
    (9, 1, 16, 3, 2, 32, 32, 90), (7, 5, 16, 3, 2, 64, 64, 40), (4, 10, 16, 2, 3, 64, 64, 60), (3, 4, 48, 1, 1, 64, 64, 40), (2, 5, 80, 1, 0, 32, 32, 40), (4, 3, 16, 2, 2, 40, 64, 90), (3, 5, 32, 2, 1, 80, 80, 40)])
def test_few_tiles_over_waves(th, tw, S, WR, WC, dk, dv, many):
    sw = _swa()
    N, scale = th * tw * S, 1 / math.sqrt(dk)
    ops = orc.make_qkv(N + dk + th, 1, 1, N, N, dk, dv, torch.float16)
    want = orc.tiled_swa_grads(*(t.float() for t in ops), S, th, tw, WR, WC, scale)
    def run(q, k, v, do):
        leaves = [t.requires_grad_(True) for t in (q, k, v)]
        o = sw.TiledSwa.apply(*leaves, S, th, tw, WR, WC, scale)
        return (o.detach(),) + torch.autograd.grad(o, leaves, do)
    one = run(*(t.cuda() for t in ops))
    apart = run(*(t.cuda().permute(0, 2, 1, 3).repeat(1, 1, 3, 1)[:, :, 1:2].permute(0, 2, 1, 3) for t in ops))   # token rows of three heads
    all_ = run(*(t.cuda().repeat(many, 1, 1, 1) for t in ops))
    for got in (one, apart, all_):
        assert (got[0][-1:].float().cpu() - want[0]).abs().max().item() <= FWD_TOL
        errs = [_rel(g[-1:], w) for g, w in zip(got[1:], want[1:])]
        assert max(errs) <= 1e-2, errs   # fp16
    assert all(torch.equal(x, y) for x, y in zip(one, apart))
    bh, lay = 4 if S == 16 else 2, lambda t: orc.tokens_to_image(t.cpu(), th, tw, bh, S // bh).contiguous().cuda()
    leaves = [lay(t).requires_grad_(True) for t in ops[:3]]
    o = sw.TiledSwaImage.apply(*leaves, bh, S // bh, WR, WC, scale)
    assert all(torch.equal(x, lay(y)) for x, y in zip((o,) + torch.autograd.grad(o, leaves, lay(ops[3])), one))
    q, k, v, do = (t.cuda() for t in ops)
    cell = torch.arange(N, device="cuda") // S
    far = ((cell // tw - th // 2).abs() > WR) | ((cell % tw - tw // 2).abs() > WC)
    k[:, :, cell == th // 2 * tw + tw // 2] = float("inf")
    v[:, :, cell == th // 2 * tw + tw // 2] = float("nan")
    o, dq, _, _ = run(q, k, v, do)
    assert torch.equal(o[:, :, far], one[0][:, :, far]) and torch.equal(dq[:, :, far], one[1][:, :, far])


# tiles of 64 k tokens on the asynchronously staged kernels: workgroups of 64 own tokens (few, or rows that leave 128 a sixth empty) and of 128, tiles of
# two and three chunks, rows of odd and even tile counts, windows beyond the grid, every class; image tiles of whole pixel rows per chunk and others
@pytest.mark.parametrize("th,tw,tile,WR,WC,dk,dv,many", [
    (3, 6, 64, 1, 1, 32, 32, 60), (2, 9, 64, 1, 2, 64, 64, 60), (4, 1, 128, 1, 1, 64, 64, 110), (2, 4, 192, 2, 0, 32, 32, 50), (3, 5, 64, 0, 1, 128, 128, 60),
    (1, 8, 64, 3, 1, 64, 128, 110), (3, 4, (8, 8), 1, 1, 32, 32, 80), (2, 6, (4, 16), 1, 1, 64, 64, 80), (2, 3, (64, 2), 1, 1, 128, 128, 80),
    (2, 4, (2, 64), 1, 2, 64, 128, 50), (2, 4, (4, 48), 1, 1, 64, 64, 50)])
def test_tiles_of_64_tokens(th, tw, tile, WR, WC, dk, dv, many):
    sw = _swa()
    img = isinstance(tile, tuple)
    S = tile[0] * tile[1] if img else tile
    N, scale = th * tw * S, 1 / math.sqrt(dk)
    ops = orc.make_qkv(N + dk + th, 1, 1, N, N, dk, dv, torch.float16)
    want = orc.tiled_swa_grads(*(t.float() for t in ops), S, th, tw, WR, WC, scale)
    lay = (lambda t: orc.tokens_to_image(t, th, tw, *tile).contiguous()) if img else (lambda t: t)
    runs = []
    for slabs in (1, many):
        q, k, v, do = (lay(t).cuda().repeat(slabs, *[1] * (4 if img else 3)) for t in ops)
        leaves = [t.requires_grad_(True) for t in (q, k, v)]
        o = sw.TiledSwaImage.apply(*leaves, *tile, WR, WC, scale) if img else sw.TiledSwa.apply(*leaves, S, th, tw, WR, WC, scale)
        runs.append((o.detach(),) + torch.autograd.grad(o, leaves, do))
    assert (runs[0][0].float().cpu() - lay(want[0])).abs().max().item() <= FWD_TOL
    errs = [_rel(g, lay(w)) for g, w in zip(runs[0][1:], want[1:])]
    assert max(errs) <= 1e-2, errs   # fp16
    for one, all_ in zip(*runs):
        assert torch.equal(all_, one.expand_as(all_))   # the same bits in both workgroup sizes


# windows of 5 x 3 tiles at d = 64 and, forward, 3 x 3 at d = 128 and 5 x 5 at d = 64, on strips of four tiles: grids below the window, rows below a band's ring, strips whole,
# ragged and with one tile; image layout with the same bits; infinite and NaN tiles stay with the queries that see them
@pytest.mark.parametrize("WR,WC,d", [(2, 1, 64), (1, 1, 128), (2, 2, 64)])
@pytest.mark.parametrize("th,tw,B,dtype", [(1, 4, 80, torch.float16), (2, 5, 20, torch.bfloat16), (4, 8, 8, torch.float16), (11, 9, 2, torch.bfloat16), (7, 13, 9, torch.float16),
                                          (5, 4, 200, torch.bfloat16)])
def test_strips_of_four_tiles(th, tw, B, dtype, WR, WC, d):
    sw = _swa()
    S, H, scale = 16, 2, 0.125
    N = th * tw * S
    ops = orc.make_qkv(N, B, H, N, N, d, d, dtype)
    dev = [t.cuda() for t in ops]

    def run(q, k, v, do):
        leaves = [t.detach().requires_grad_(True) for t in (q, k, v)]
        o = sw.TiledSwa.apply(*leaves, S, th, tw, WR, WC, scale)
        return (o.detach(),) + torch.autograd.grad(o, leaves, do)

    got = run(*dev)
    for b in (0, B - 1):
        want = orc.tiled_swa_grads(*(t[b:b + 1].float() for t in ops), S, th, tw, WR, WC, scale)
        assert (got[0][b:b + 1].float().cpu() - want[0]).abs().max().item() <= FWD_TOL
        assert max(_rel(g[b:b + 1], w) for g, w in zip(got[1:], want[1:])) <= GRAD_TOL
    lay = lambda t: orc.tokens_to_image(t.cpu(), th, tw, 4, 4).contiguous().cuda()
    leaves = [lay(t).requires_grad_(True) for t in ops[:3]]
    o = sw.TiledSwaImage.apply(*leaves, 4, 4, WR, WC, scale)
    assert all(torch.equal(x, lay(y)) for x, y in zip((o,) + torch.autograd.grad(o, leaves, lay(ops[3])), got))
    cell = torch.arange(N, device="cuda") // S
    at = cell == th // 2 * tw + tw // 2
    far = ((cell // tw - th // 2).abs() > WR) | ((cell % tw - tw // 2).abs() > WC)
    q, k, v, do = (t.clone() for t in dev)
    k[:, :, at], v[:, :, at] = float("inf"), float("nan")
    o, dq, _, _ = run(q, k, v, do)
    assert torch.equal(o[:, :, far], got[0][:, :, far])
    if d == 128 or WC == 2:   # the gradients come from the chunked flash kernels, whose masked products of a whole chunk meet NaN
        return
    assert torch.equal(dq[:, :, far], got[1][:, :, far])
    q, k, v, do = (t.clone() for t in dev)
    q[:, :, at], do[:, :, at] = float("nan"), float("inf")
    _, _, dk, dv = run(q, k, v, do)
    assert torch.equal(dk[:, :, far], got[2][:, :, far]) and torch.equal(dv[:, :, far], got[3][:, :, far])


# A value row with infinities: queries that see it get them in those dims and their plain results in the others, also where the window has an odd number of
# 16-token runs (the last pair of runs holds nothing beside the last one) and where it hangs over the grid's edge (strips of eight tiles: rows
# away from it, `edge`); the same for dV under a dO row with them.  Windows' keys over waves (runs of 16, 48 and 80 tokens), strips of four tiles and of eight
@pytest.mark.parametrize("th,tw,S,WR,WC,d,slabs,bwd,edge", [
    (5, 6, 16, 1, 3, 64, 1, True, True), (4, 5, 16, 1, 1, 128, 1, True, True), (3, 5, 48, 1, 1, 64, 1, True, True), (3, 4, 80, 1, 1, 32, 1, True, True),
    (9, 8, 16, 1, 1, 128, 8, False, True), (9, 8, 16, 2, 1, 64, 8, True, True), (6, 9, 16, 2, 2, 64, 16, False, True), (7, 9, 16, 1, 1, 32, 4, True, False)])
def test_infinite_values_reach_the_queries_that_see_them(th, tw, S, WR, WC, d, slabs, bwd, edge):
    sw, N, scale, inf = _swa(), th * tw * S, 1 / math.sqrt(d), float("inf")
    q, k, v, do = (t.cuda() for t in orc.make_qkv(N + d, 1, slabs, N, N, d, d, torch.bfloat16))

    def run(v, do):
        leaves = [t.detach().requires_grad_(True) for t in (q, k, v)]
        o = sw.TiledSwa.apply(*leaves, S, th, tw, WR, WC, scale)
        return (o.detach(),) + torch.autograd.grad(o, leaves, do)

    o, _, dk, dv = run(v, do)
    cell = torch.arange(N, device="cuda") // S
    for r, c in ((th // 2, tw // 2),) + (((0, 0), (th - 1, tw - 1), (0, tw - 1), (th - 1, 0)) if edge else ()):
        at = (r * tw + c) * S + (S - 1 if r else 0)
        sees = ((cell // tw - r).abs() <= WR) & ((cell % tw - c).abs() <= WC)
        bad, want = v.clone(), o.clone()
        for t, rows in ((bad, at), (want, sees)):
            t[:, :, rows, 3], t[:, :, rows, d - 1] = inf, -inf
        assert torch.equal(run(bad, do)[0], want), (r, c)
        if bwd:
            bad, want = do.clone(), dv.clone()
            for t, rows in ((bad, at), (want, sees)):
                t[:, :, rows, 3], t[:, :, rows, d - 1] = inf, -inf
            _, _, dk2, dv2 = run(v, bad)
            assert torch.equal(dv2, want) and torch.equal(dk2[:, :, ~sees], dk[:, :, ~sees]), (r, c)


# ... where a slab has the same bits alone and beside any number of others (backward: not two strips of which the second is mostly empty)
@pytest.mark.parametrize("th,tw,WR,WC,d,bwd", [
    (3, 4, 2, 1, 64, True), (1, 7, 2, 1, 64, True), (14, 9, 2, 1, 64, True), (5, 6, 2, 1, 64, False), (7, 5, 2, 2, 64, False), (2, 4, 2, 2, 64, False), (6, 4, 1, 1, 128, False),
    (5, 7, 1, 1, 128, False), (1, 12, 1, 1, 128, False)])
def test_strips_of_four_tiles_bits_of_a_slab(th, tw, WR, WC, d, bwd):
    sw, S = _swa(), 16
    N = th * tw * S
    ops = [t.cuda() for t in orc.make_qkv(N + d, 1, 1, N, N, d, d, torch.bfloat16)]

    def run(slabs):
        leaves = [t.repeat(slabs, 1, 1, 1).requires_grad_(True) for t in ops[:3]]
        o = sw.TiledSwa.apply(*leaves, S, th, tw, WR, WC, 0.125)
        return (o.detach(),) + (torch.autograd.grad(o, leaves, ops[3].repeat(slabs, 1, 1, 1)) if bwd else ())

    one = run(1)
    for slabs in (2, 7, 40, 300):
        assert all(torch.equal(a, b.expand_as(a)) for a, b in zip(run(slabs), one)), slabs
