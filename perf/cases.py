"""The calls whose speed this package answers for, as a program that uses it makes them.

Four operators and their data types, sizes and directions:

* ``swa``    attention over a window of a 2D token grid, one token per cell (``TiledSwa`` / ``tiled_swa_fwd``; with
             ``"rope"`` the 2D rotation of q and k is part of the operator, ``TiledSwaRope``);
* ``tiles``  the same window over tiles of several tokens (``TiledSwa`` with ``b_size`` > 1);
* ``image``  the same on tensors kept as images (``TiledSwaImage``);
* ``flash``  dense or causal attention, query and key length and qk / vo head dims of their own (``attention``);
* ``rope``   the 2D rotation alone: of q and k in place (``rope2d_qk_``), or of one tensor through the module with its
             backward pass (``FusedInplaceRotaryPositionEncoding2D``).

``"train": True`` is a forward and a backward pass through autograd; otherwise the forward pass alone without gradients.
"""
import math

import torch

from dl_templates_amd.flash_attn import attention
from dl_templates_amd.fused_rope2d import FusedInplaceRotaryPositionEncoding2D, rope2d_qk_
from dl_templates_amd.tiled_swa import TiledSwa, TiledSwaImage, TiledSwaRope, tiled_swa_fwd

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
BYTES = {"bf16": 2, "fp16": 2, "fp32": 4}


def listed():
    return [
        # the smallest call: one little map, 32-bit tensors, inference (latency of a single launch)
        dict(name="swa_fwd_16x16_fp32", op="swa", dtype="fp32", train=False, rope=False, B=1, H=2, th=16, tw=16, wr=3, wc=3, d=32),
        # one feature map of odd size at small batch, half precision: training with few tokens (launches and host work)
        dict(name="swa_train_33x47_fp16", op="swa", dtype="fp16", train=True, rope=False, B=2, H=4, th=33, tw=47, wr=3, wc=4, d=64),
        # the rotation of q and k in front of an attention layer, 32 of 64 dims rotated
        dict(name="rope_qk_64x64", op="rope", dtype="bf16", train=False, inverse=False, B=4, H=8, th=64, tw=64, d=64, n_rot=32),
        # the rotation module inside a training step, whole head rotated, a map of odd height
        dict(name="rope_train_75x100", op="rope", dtype="bf16", train=True, inverse=False, B=2, H=16, th=75, tw=100, d=64, n_rot=64),
        # a layer of a window-attention network at its usual size: rotation and attention, training
        dict(name="swa_rope_train_64x64", op="swa", dtype="bf16", train=True, rope=True, B=2, H=8, th=64, tw=64, wr=6, wc=6, d=64),
        # a large map with a large window and wide heads, training
        dict(name="swa_train_128x128_d128", op="swa", dtype="bf16", train=True, rope=False, B=1, H=16, th=128, tw=128, wr=10, wc=10, d=128),
        # the same layer at inference on a map that no tile divides
        dict(name="swa_fwd_97x161_d128", op="swa", dtype="bf16", train=False, rope=False, B=1, H=16, th=97, tw=161, wr=10, wc=10, d=128),
        # tiles of 16 tokens, half precision: small tiles and small heads
        dict(name="tiles_train_16x16_b16", op="tiles", dtype="fp16", train=True, B=4, H=8, th=16, tw=16, S=16, wr=1, wc=1, d=32),
        # a whole image kept in its own layout, tiles of 4 x 4 pixels
        dict(name="image_train_256x256", op="image", dtype="fp16", train=True, B=4, H=8, th=64, tw=64, bh=4, bw=4, wr=1, wc=1, d=32),
        # a short ragged set of queries (text tokens, latents) attending to a longer memory at inference
        dict(name="flash_cross_fwd_77x1500", op="flash", dtype="bf16", train=False, causal=False, B=2, H=8, Lq=77, Lk=1500, dk=64, dv=64, scale=0.125),
        # causal self-attention of a long sequence, training in half precision
        dict(name="flash_causal_train_4096", op="flash", dtype="fp16", train=True, causal=True, B=4, H=32, Lq=4096, Lk=4096, dk=64, dv=64, scale=0.125),
        # long cross-attention with different qk and vo head dims, training: the largest
        dict(name="flash_cross_train_4096x8192", op="flash", dtype="bf16", train=True, causal=False, B=2, H=16, Lq=4096, Lk=8192, dk=64, dv=128, scale=0.125),
    ]


def _log(rng, lo, hi):
    """A whole number between lo and hi, spread evenly over the logarithm."""
    return min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def _draw(rng):
    op = rng.choice(["swa", "swa", "swa", "flash", "flash", "flash", "rope", "tiles", "image"])
    dtype = rng.choice(["bf16", "bf16", "fp16"])
    train = rng.random() < 0.6
    B, H = rng.choice([1, 1, 2, 4]), rng.choice([2, 4, 8, 16])
    if op == "swa":
        if rng.random() < 0.1:   # 32-bit tensors: small maps at inference
            return dict(op=op, dtype="fp32", train=False, rope=False, B=B, H=H, th=_log(rng, 8, 32), tw=_log(rng, 8, 32),
                        wr=rng.randint(1, 4), wc=rng.randint(1, 4), d=rng.choice([32, 64]))
        d = rng.choice([32, 64, 64, 128, 128])
        rope = train and d >= 64 and rng.random() < 0.4
        wmax = 6 if d <= 64 and rng.random() < 0.5 else 10
        return dict(op=op, dtype=dtype, train=train, rope=rope, B=B, H=H, th=_log(rng, 12, 160), tw=_log(rng, 12, 160),
                    wr=rng.randint(2, wmax), wc=rng.randint(2, wmax), d=d)
    if op == "tiles":
        S = rng.choice([4, 16, 16, 64])
        return dict(op=op, dtype=dtype, train=train, B=B, H=H, th=_log(rng, 4, 40), tw=_log(rng, 4, 40), S=S, wr=rng.randint(1, 2),
                    wc=rng.randint(1, 2), d=rng.choice([32, 64, 64, 128]))
    if op == "image":
        bh, bw = rng.choice([(4, 4), (4, 4), (4, 8), (8, 8)])
        return dict(op=op, dtype=dtype, train=train, B=B, H=rng.choice([2, 4, 8]), th=_log(rng, 4, 48), tw=_log(rng, 4, 48), bh=bh, bw=bw,
                    wr=1, wc=1, d=rng.choice([32, 64]))
    if op == "rope":
        d = rng.choice([64, 64, 128])
        return dict(op=op, dtype=rng.choice(["bf16", "bf16", "fp16", "fp32"]), train=rng.random() < 0.4, inverse=rng.random() < 0.3, B=B, H=H,
                    th=_log(rng, 12, 128), tw=_log(rng, 12, 128), d=d, n_rot=rng.choice([d // 2, d]))
    causal = rng.random() < 0.4
    Lq, Lk = _log(rng, 32, 8192), _log(rng, 64, 8192)
    dk, dv = rng.choice([(64, 64), (64, 64), (64, 128), (128, 128), (128, 128), (80, 80)])
    return dict(op=op, dtype=dtype, train=train, causal=causal, B=B, H=rng.choice([4, 8, 16, 32]), Lq=Lk if causal else Lq, Lk=Lk, dk=dk, dv=dv,
                scale=round(1.0 / math.sqrt(dk), 6))


def draw(rng):
    largest = work(listed()[-1])
    while True:
        case = _draw(rng)
        w = work(case)
        if w["flops"] <= 0.8 * largest["flops"] and w["bytes"] <= 1.0e9:
            return case


def _tokens(c):
    if c["op"] == "flash":
        return c["Lq"], c["Lk"]
    n = c["th"] * c["tw"] * (c["S"] if c["op"] == "tiles" else c["bh"] * c["bw"] if c["op"] == "image" else 1)
    return n, n


def _rotation(c, gen, n_rot):
    """(module with the cos / sin tables, idx): grid positions, one token in twenty without a position."""
    pe = FusedInplaceRotaryPositionEncoding2D(n_rot, c["th"], c["tw"]).cuda()
    idx = FusedInplaceRotaryPositionEncoding2D.encode_idx(c["th"], c["tw"]).cuda()
    idx[torch.rand(idx.shape, generator=gen, device="cuda") < 0.05] = -1
    return pe, idx


def prepare(case, seed):
    c = case
    gen = torch.Generator(device="cuda").manual_seed(seed)
    dt = DTYPES[c["dtype"]]
    nq, nk = _tokens(c)
    dk, dv = (c["dk"], c["dv"]) if c["op"] == "flash" else (c["d"], c["d"])

    def tensor(n, d, leaf=False):
        shape = (c["B"], c["th"] * c["bh"], c["tw"] * c["bw"], c["H"], d) if c["op"] == "image" else (c["B"], c["H"], n, d)
        return torch.randn(shape, generator=gen, device="cuda").to(dt).requires_grad_(leaf)

    s = dict(case=c, train=c["train"])
    if c["op"] == "rope":
        s["pe"], s["idx"] = _rotation(c, gen, c["n_rot"])
        if c["train"]:
            s["x"], s["dy"] = tensor(nq, dk, leaf=True), tensor(nq, dk)
        else:
            s["q"], s["k"] = tensor(nq, dk), tensor(nk, dk)
        return s
    s["q"], s["k"], s["v"] = tensor(nq, dk, c["train"]), tensor(nk, dk, c["train"]), tensor(nk, dv, c["train"])
    if c["train"]:
        s["do"] = tensor(nq, dv)
    if c.get("rope"):
        s["pe"], s["idx"] = _rotation(c, gen, dk // 2)
    s["scale"] = c["scale"] if c["op"] == "flash" else 1.0 / math.sqrt(dk)
    return s


def _attend(s):
    c, q, k, v, scale = s["case"], s["q"], s["k"], s["v"], s["scale"]
    if c["op"] == "flash":
        return attention(q, k, v, c["causal"], scale)
    if c["op"] == "image":
        return TiledSwaImage.apply(q, k, v, c["bh"], c["bw"], c["wr"], c["wc"], scale)
    if c.get("rope"):
        return TiledSwaRope.apply(q, k, v, s["idx"], s["pe"].row_buffer.cs_components, s["pe"].col_buffer.cs_components, 1, c["th"], c["tw"],
                                  c["wr"], c["wc"], scale)
    if s["train"]:
        return TiledSwa.apply(q, k, v, c.get("S", 1), c["th"], c["tw"], c["wr"], c["wc"], scale)
    return tiled_swa_fwd(q, k, v, c.get("S", 1), c["th"], c["tw"], c["wr"], c["wc"], scale)


def run(state):
    s = state
    if s["case"]["op"] == "rope":
        if not s["train"]:
            return rope2d_qk_(s["q"], s["k"], s["idx"], s["pe"].row_buffer.cs_components, s["pe"].col_buffer.cs_components, s["case"]["inverse"])
        y = s["pe"](s["x"].clone(), s["idx"])
        return (y,) + torch.autograd.grad(y, (s["x"],), s["dy"])
    if not s["train"]:
        with torch.no_grad():
            return _attend(s)
    o = _attend(s)
    return (o,) + torch.autograd.grad(o, (s["q"], s["k"], s["v"]), s["do"])


def _pairs(c):
    """(query, key) pairs that see each other."""
    if c["op"] == "flash":
        return c["B"] * c["H"] * (c["Lq"] * (c["Lq"] + 1) // 2 if c["causal"] else c["Lq"] * c["Lk"])
    S = c["S"] if c["op"] == "tiles" else c["bh"] * c["bw"] if c["op"] == "image" else 1

    def along(n, w):
        return sum(min(n, i + w + 1) - max(0, i - w) for i in range(n))

    return c["B"] * c["H"] * S * S * along(c["th"], c["wr"]) * along(c["tw"], c["wc"])


def work(case):
    c = case
    e = BYTES[c["dtype"]]
    nq, nk = _tokens(c)
    rows = c["B"] * c["H"]
    if c["op"] == "rope":
        # each direction reads and writes the rotated dims; a pass of q and k is two tensors, a training step one tensor
        # there and back, with a copy of it made for the operator that works in place
        moved = 2 * e * rows * nq * c["n_rot"]
        if c["train"]:
            moved = 2 * 2 * e * rows * nq * c["d"]
        else:
            moved *= 2
        return {"bytes": moved + 4 * nq, "flops": 2 * 3 * rows * nq * c["n_rot"]}
    dk, dv = (c["dk"], c["dv"]) if c["op"] == "flash" else (c["d"], c["d"])
    q, k, v, o = (e * rows * n for n in (nq * dk, nk * dk, nk * dv, nq * dv))
    pairs = _pairs(c)
    if not c["train"]:
        return {"bytes": q + k + v + o, "flops": 2 * pairs * (dk + dv)}
    # forward and backward: q, k, v, dO in; o, dq, dk, dv out
    return {"bytes": 2 * (q + k + v + o), "flops": 2 * pairs * (dk + dv) + 2 * pairs * (3 * dk + 2 * dv)}


def tolerance(case):
    # rotation: one rounding of the result (32-bit: of two products and their sum); attention: probabilities and score
    # gradients pass through 16 bits before the second products, also where tensors are 32-bit
    if case["op"] == "rope":
        return {"rel": {"bf16": 4e-3, "fp16": 6e-4, "fp32": 2e-6}[case["dtype"]]}
    return {"rel": {"bf16": 1e-2, "fp16": 3e-3, "fp32": 1e-2}[case["dtype"]]}
