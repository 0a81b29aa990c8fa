"""The operators inside autograd as a program uses it: activation checkpointing, saved-tensor hooks, second
derivatives, forward mode, function transforms, tracing and dispatch modes."""
import math

import pytest
import torch
import torch.autograd.forward_ad as fwd_ad
from torch.utils._python_dispatch import TorchDispatchMode
from torch.utils.checkpoint import checkpoint

from oracle import attn_oracle as orc

pytestmark = pytest.mark.gpu

TH, TW, D = 6, 10, 64
SCALE = 1 / math.sqrt(D)


def _rope_args():
    return (orc.make_rope_idx(1, TH, TW, 0.1).cuda(), orc.rope_tables(8, TH).cuda(), orc.rope_tables(8, TW).cuda())


def _ops():
    """name -> (operator on three tensors, shape of the tensors); every operator with an autograd node."""
    from dl_templates_amd.flash_attn import attention
    from dl_templates_amd.fused_rope2d import FusedInplaceRotaryPositionEncoding2D, RotaryPE2D
    from dl_templates_amd.tiled_swa import TiledSwa, TiledSwaImage, TiledSwaRope
    tokens, dims = (1, 2, TH * TW, D), (1, TH, TW, 3, 3, SCALE)
    rope, module = _rope_args(), FusedInplaceRotaryPositionEncoding2D(32, TH, TW).cuda()
    return {
        "flash": (lambda q, k, v: attention(q, k, v, False, SCALE), tokens),
        "flash_padded": (lambda q, k, v: attention(q, k, v, False, SCALE), (1, 2, 50, 36)),
        "swa": (lambda q, k, v: TiledSwa.apply(q, k, v, *dims), tokens),
        "swa_rope": (lambda q, k, v: TiledSwaRope.apply(q, k, v, *rope, *dims), tokens),
        "swa_rope_again": (lambda q, k, v: TiledSwaRope.apply(q, k, v, *rope, *dims, False), tokens),
        "image": (lambda q, k, v: TiledSwaImage.apply(q, k, v, 2, 2, 1, 1, SCALE), (1, TH, TW, 2, D)),
        "rotation": (lambda q, k, v: RotaryPE2D.apply((q * k * v)[0], *rope), tokens),
        "rotation_module": (lambda q, k, v: module(q * k * v, rope[0]), tokens),
    }


OPS = ["flash", "flash_padded", "swa", "swa_rope", "swa_rope_again", "image", "rotation", "rotation_module"]


def _inputs(name, dtype=torch.bfloat16):
    op, shape = _ops()[name]
    gen = torch.Generator().manual_seed(len(name))
    return op, [torch.randn(shape, generator=gen).to(dtype).cuda().requires_grad_(True) for _ in range(3)]


@pytest.mark.parametrize("first", [False, True])
@pytest.mark.parametrize("name", OPS)
def test_checkpointed_region(name, first):
    """Non-reentrant checkpointing runs the region again inside an unpack hook of its nodes.  Bit-equal to the plain step, with the
    operator as the last of the region (its node is the first one unpacked) and as the first."""
    op, x = _inputs(name)
    block = (lambda q, k, v: op(q * 2, k * 2, v * 2) * 3) if first else (lambda q, k, v: op(q * 2, k * 2, v * 2))
    o = block(*x)
    do = torch.randn_like(o)
    want = torch.autograd.grad(o, x, do)
    got_o = checkpoint(block, *x, use_reentrant=False)
    assert torch.equal(got_o, o)
    for g, w in zip(torch.autograd.grad(got_o, x, do), want):
        assert torch.equal(g, w)


@pytest.mark.parametrize("name", OPS)
def test_saved_tensor_hooks_run_with_autograd_on(name):
    op, x = _inputs(name)
    o = op(*x)
    do = torch.randn_like(o)
    want = torch.autograd.grad(o, x, do)
    leaf, seen = torch.ones(1, device="cuda", requires_grad=True), []

    def hook(where):
        def run(t):
            with torch.enable_grad():   # hooks run with gradients off
                seen.append((where, (leaf * 2).requires_grad))
            return t.cpu() if where == "pack" else t.cuda()
        return run

    with torch.autograd.graph.saved_tensors_hooks(hook("pack"), hook("unpack")):
        o2 = op(*x)
    got = torch.autograd.grad(o2, x, do)
    assert {w for w, _ in seen} == {"pack", "unpack"} and all(on for _, on in seen), seen
    assert torch.equal(o2, o) and all(torch.equal(a, b) for a, b in zip(got, want))


@pytest.mark.parametrize("name", ["rotation", "rotation_module"])
def test_rotation_refuses_a_second_derivative(name):
    """A gradient penalty through the rotation raises; ``create_graph`` alone, for first derivatives, is fine."""
    op, x = _inputs(name, torch.float32)
    o = op(*x)
    want = torch.autograd.grad((o ** 2).sum(), x, retain_graph=True)
    got = torch.autograd.grad((o ** 2).sum(), x, create_graph=True)
    for g, w in zip(got, want):
        assert torch.equal(g, w)
    with pytest.raises(RuntimeError, match="differentiate twice"):
        ((o ** 2).sum() + 10 * sum((g ** 2).sum() for g in got)).backward()


@pytest.mark.parametrize("which", [0, 1, 2])
@pytest.mark.parametrize("name", OPS)
def test_forward_mode_is_refused(name, which):
    """There is no derivative in forward mode: a tangent on any input raises instead of being dropped."""
    op, x = _inputs(name, torch.float32)
    x = [t.detach() for t in x]
    with fwd_ad.dual_level():
        x[which] = fwd_ad.make_dual(x[which], torch.ones_like(x[which]))
        with pytest.raises(NotImplementedError):
            op(*x)


@pytest.mark.parametrize("name", OPS)
def test_function_transforms_are_refused(name):
    op, x = _inputs(name, torch.float32)
    x = [t.detach() for t in x]
    with pytest.raises(RuntimeError, match="setup_context"):
        torch.func.grad(lambda q: op(q, *x[1:]).sum())(x[0])
    with pytest.raises(RuntimeError, match="setup_context"):
        torch.func.vmap(lambda q: op(q, *x[1:]))(torch.stack([x[0], x[0]]))


class _Plain(TorchDispatchMode):
    def __torch_dispatch__(self, func, types, args=(), kwargs=None):
        return func(*args, **(kwargs or {}))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("name", OPS)
def test_class_and_compiled_node_agree(name, dtype):
    """Under a dispatch mode the class itself runs: same bits as the compiled node, forward and backward."""
    op, x = _inputs(name, dtype)
    o = op(*x)
    do = torch.randn_like(o)
    with _Plain():
        o2 = op(*x)
    assert torch.equal(o, o2)
    for a, b in zip(torch.autograd.grad(o, x, do), torch.autograd.grad(o2, x, do)):
        assert torch.equal(a, b)


@pytest.mark.parametrize("name", [n for n in OPS if not n.startswith("rotation")])
def test_traced_call_depends_on_its_inputs(name):
    op, x = _inputs(name)
    x = [t.detach() for t in x]
    traced = torch.jit.trace(lambda q, k, v: op(q, k, v), tuple(x), check_trace=False)
    y = [t.flip(0, 1) * 0.5 for t in x]
    assert torch.equal(traced(*y), op(*y))


class _NoGrad(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x):
        return x.clone()

    @staticmethod
    def backward(ctx, g):
        return None


@pytest.mark.parametrize("name", [n for n in OPS if n != "rotation"])   # it rotates a view: the missing gradient ends at the base
def test_missing_gradient_counts_as_zeros(name):
    op, x = _inputs(name)
    for g in torch.autograd.grad(_NoGrad.apply(op(*x)).sum(), x):
        assert not g.any()
