"""Attention's products recorded as one native node each, against the Functions they stand for: the same values, gradients and refusals."""
import pytest
import torch

import bgemm_linear as bl

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


class Scores(bl.bgemm_matmul):
    """The Function itself: a class of its own does not take the node."""


class Context(bl.bgemm_attn_matmul):
    pass


def leaves(kind, B, H, N, M, D, seed=0):
    """Two fp16 leaves and the product's operands made of them: head-split views (B 0: three dimensions)."""
    g = torch.Generator(device=DEV).manual_seed(seed)
    rnd = lambda *s: torch.randn(*s, generator=g, device=DEV).half().requires_grad_(True)
    if B == 0:
        a, b = rnd(H, N, D if kind == "scores" else M), rnd(H, M, D)
        return (a, b), (lambda: (a, b.transpose(-1, -2) if kind == "scores" else b))
    split = lambda t: t.view(t.shape[0], t.shape[1], H, D).permute(0, 2, 1, 3)
    b = rnd(B, M, H * D)
    a = rnd(B, N, H * D) if kind == "scores" else rnd(B, H, N, M)
    return (a, b), (lambda: (split(a), split(b).transpose(-1, -2)) if kind == "scores" else (a, split(b)))


PAIRS = {"scores": (bl.bgemm_matmul, Scores, "BinaryScoresBackward"), "context": (bl.bgemm_attn_matmul, Context, "BinaryContextBackward")}


# sizes the gradients' kernels take, and ones they do not: another head size, rows beyond their limit, one of something
@pytest.mark.parametrize("B,H,N,M,D", [(2, 3, 64, 64, 64), (1, 2, 33, 65, 32), (0, 3, 70, 50, 96), (2, 2, 40, 24, 40), (1, 1, 8, 4104, 32), (1, 1, 2100, 16, 64)])
@pytest.mark.parametrize("kind", ["scores", "context"])
def test_node_gives_what_the_function_gives(kind, B, H, N, M, D):
    node, fn, name = PAIRS[kind]
    for wants in ((0, 1), (0,), (1,)):
        (a, b), args = leaves(kind, B, H, N, M, D, seed=N + M)
        for i, t in enumerate((a, b)):
            t.requires_grad_(i in wants)
        got, want = node.apply(*args()), fn.apply(*args())
        assert got.grad_fn.name() == name and want.grad_fn.name() != name and torch.equal(got, want)
        g = torch.randn_like(got)
        ins = [(a, b)[i] for i in wants]
        for x, y in zip(torch.autograd.grad(got, ins, g, retain_graph=True), torch.autograd.grad(want, ins, g)):
            assert x.dtype == y.dtype and x.stride() == y.stride() and torch.equal(x, y), (kind, wants)
        got.backward(g)                       # the second pass over a graph that was kept; a third is refused
        with pytest.raises(RuntimeError, match="second time"):
            torch.autograd.grad(got, ins, g)


@pytest.mark.parametrize("kind", ["scores", "context"])
def test_what_torch_has_to_see_goes_its_way(kind):
    node, fn, name = PAIRS[kind]
    (a, b), args = leaves(kind, 1, 2, 64, 64, 64)
    seen = []
    with torch.autograd.graph.saved_tensors_hooks(lambda t: (seen.append(t), t)[1], lambda t: t):
        assert node.apply(*args()).grad_fn.name() != name
    assert len(seen) == 2
    with torch.no_grad():
        assert node.apply(*args()).grad_fn is None
    assert node.apply(*(t.float() for t in args())).grad_fn.name() != name       # other types: the Function
    # a gradient that is itself differentiated: by the upstream one
    out, ref = node.apply(*args()), fn.apply(*args())
    g = torch.randn_like(out).requires_grad_(True)
    first, second = torch.autograd.grad(out, (a, b), g, create_graph=True), torch.autograd.grad(ref, (a, b), g, create_graph=True)
    for x, y in zip(first, second):
        assert torch.equal(x, y) and x.requires_grad
        assert torch.equal(*(torch.autograd.grad(t.float().sum(), g, retain_graph=True)[0] for t in (x, y)))
    # a batch of upstream gradients, and forward mode, which the Function has no rule for
    gs = torch.randn(3, *out.shape, device=DEV).half()
    for x, y in zip(torch.autograd.grad(out, (a, b), gs, is_grads_batched=True, retain_graph=True), torch.autograd.grad(ref, (a, b), gs, is_grads_batched=True, retain_graph=True)):
        assert torch.equal(x, y)
    with torch.autograd.forward_ad.dual_level():
        dual = torch.autograd.forward_ad.make_dual(a.detach(), torch.ones_like(a))
        for f in (node, fn):
            with pytest.raises((RuntimeError, NotImplementedError)):
                f.apply(*((dual, b.detach().transpose(-1, -2)) if kind == "scores" and a.dim() == 3 else (dual, args()[1]) if kind == "context" else
                          (dual.view(1, 64, 2, 64).permute(0, 2, 1, 3), args()[1])))
    # an operand changed between the passes is refused
    with torch.no_grad():
        b.add_(1)
    for t in (out, ref):
        with pytest.raises(RuntimeError, match="inplace"):
            torch.autograd.grad(t, (a, b), g.detach())


class Stops(torch.autograd.Function):
    """Gives what it is given, and no gradient for it."""

    @staticmethod
    def forward(ctx, t):
        return t.clone()

    @staticmethod
    def backward(ctx, grad):
        return None


@pytest.mark.parametrize("kind", ["scores", "context"])
def test_no_gradient_from_above_is_zeros(kind):
    node, fn, _ = PAIRS[kind]
    for wants in ((0, 1), (0,), (1,)):
        got = []
        for f in (node, fn):
            (a, b), args = leaves(kind, 1, 2, 40, 56, 32)
            for i, t in enumerate((a, b)):
                t.requires_grad_(i in wants)
            ins, out = [(a, b)[i] for i in wants], Stops.apply(f.apply(*args()))
            got.append(torch.autograd.grad(out, ins, torch.ones_like(out), retain_graph=True))
            out.backward(torch.ones_like(out))
            assert all(torch.equal(t.grad, g) for t, g in zip(ins, got[-1]))
        for x, y, t in zip(*got, ins):
            assert x.dtype == y.dtype == t.dtype and x.stride() == y.stride() and torch.equal(x, y) and torch.equal(x, torch.zeros_like(t))
