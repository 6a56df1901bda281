"""The one-launch gradients of both attention products against float64, and against the torch operations they stand for."""
import pytest
import torch

pytestmark = pytest.mark.gpu

import bgemm_linear as bl
import lowbit_kernel as lk

DEV = "cuda:0"


class Scores(bl.bgemm_matmul):
    """The Function itself: a class of its own does not take the node."""


class Context(bl.bgemm_attn_matmul):
    pass


def head_split(t, H):
    return t.view(t.shape[0], t.shape[1], H, -1).permute(0, 2, 1, 3)


def bound(terms):
    """Products of fp16 numbers and +-1 (1/2) are exact in fp32; `terms` sums of them in any order, rounded to fp16 once: half a last
    place of the result, 2^-24 of the absolute sum for each addition, and the smallest fp16 step."""
    return lambda got, want, total: bool(((got.double() - want).abs() <= want.abs() * 2.0 ** -11 + total * terms * 2.0 ** -23 + 2.0 ** -24).all())


@pytest.mark.parametrize("B, H, N, M, d", [(1, 1, 1, 1, 32), (2, 3, 7, 65, 64), (1, 2, 64, 64, 96), (3, 1, 63, 8, 128), (2, 2, 129, 71, 32),
                                           (1, 5, 130, 200, 64), (4, 12, 512, 512, 64),
                                           # both sides of the dispatch's limits on the rows
                                           (1, 1, 2048, 100, 32), (1, 1, 2049, 100, 32), (1, 1, 90, 2049, 64), (1, 1, 4096, 100, 32),
                                           (1, 1, 4097, 100, 32),
                                           # and of the one on the products, which is for heads of more than 96 columns
                                           (48, 1, 1024, 1024, 128), (47, 1, 1024, 1024, 128), (64, 1, 1024, 1024, 96)])
def test_gradients(B, H, N, M, d, monkeypatch):
    g = torch.Generator(device=DEV).manual_seed(N * 131 + M)
    rnd = lambda *s: torch.randn(*s, generator=g, device=DEV).half()
    q, k, v, p = rnd(B, N, H * d), rnd(B, M, H * d), rnd(B, M, H * d), rnd(B, H, N, M)
    for t in (q, k, v, p):
        t.view(-1)[::3] = 0                                       # sign 0 / weight 1/2
        t.view(-1)[1::7] = -0.0
        t.view(-1)[2::11] = float("nan")
        t.view(-1)[5::13] = float("inf")
    for t in (q, k, v, p):
        t.requires_grad_(True)
    gs, gc = rnd(B, H, N, M), rnd(B, H, N, d)

    def grads(scores_fn, context_fn, **kw):
        scores = scores_fn.apply(head_split(q, H), head_split(k, H).transpose(-1, -2))
        context = context_fn.apply(p, head_split(v, H))
        assert (scores.grad_fn.name() == "BinaryScoresBackward") == (scores_fn is bl.bgemm_matmul)
        assert (context.grad_fn.name() == "BinaryContextBackward") == (context_fn is bl.bgemm_attn_matmul)
        return torch.autograd.grad([scores, context], [q, k, v, p], [gs, gc], **kw)

    # the Functions call the kernels' launches by name; the nodes call the Functions' gradients where they launch nothing themselves
    calls, left = [], []
    for module, names, seen in ((lk, ("scores_backward", "context_backward"), calls), (bl, ("_scores_grads", "_context_grads"), left)):
        for name in names:
            monkeypatch.setattr(module, name, lambda *a, fn=getattr(module, name), name=name, seen=seen: seen.append(name) or fn(*a))
    rows, want_calls = max(N, M), []
    if rows <= bl.CONTEXT_GRAD_ROWS:
        want_calls.append("context_backward")
    if bl._scores_grad_ahead(B * H, N, M, d):
        want_calls.append("scores_backward")
    got = grads(Scores, Context)
    assert sorted(calls) == want_calls
    general = grads(Scores, Context, create_graph=True)           # needs the torch operations
    assert sorted(calls) == want_calls
    left.clear()
    node = grads(bl.bgemm_matmul, bl.bgemm_attn_matmul)
    assert sorted(calls) == want_calls and sorted(n.replace("grads", "backward")[1:] for n in left) == sorted({"context_backward", "scores_backward"} - set(want_calls))
    sign = lambda t: ((t > 0).double() - (t < 0).double())
    sq, sk, sv = (sign(head_split(t.detach(), H)) for t in (q, k, v))
    w = 0.5 + 0.5 * sign(p.detach()).abs()
    gs, gc = gs.double(), gc.double()
    merge = lambda t: t.permute(0, 2, 1, 3).reshape(B, -1, H * d)
    T = lambda t: t.transpose(-1, -2).contiguous()
    want = [merge(gs @ sk), merge(T(gs) @ sq), merge(T(w) @ gc), gc @ T(sv) / 2]
    total = [merge(gs.abs() @ sk.abs()), merge(T(gs.abs()) @ sq.abs()), merge(T(w) @ gc.abs()), gc.abs() @ T(sv.abs()) / 2]
    kernel = ["scores_backward", "scores_backward", "context_backward", "context_backward"]
    for way in (got, node):
        for a, b, x, y, terms, which in zip(way, (t.detach() for t in general), want, total, (M, N, N, d), kernel):
            assert a.shape == b.shape and a.dtype == b.dtype
            assert which not in calls or a.is_contiguous()           # the kernels' gradients lie as their operands do
            assert bound(terms)(a, x, y)
            assert float((a.double() - x).norm()) <= 1.02 * float((b.double() - x).norm()) + 1e-9


# grad_P in strips of 128, 256 and 512 columns: the last strip whole, of one 64 and a rest, and ending before its columns do; rows of 128 and a rest
@pytest.mark.parametrize("chunks, B, H, N, M, d", [(2, 70, 3, 129, 550, 128), (2, 70, 3, 257, 577, 32), (2, 128, 4, 128, 512, 96), (4, 175, 4, 5, 577, 64), (4, 350, 2, 33, 641, 128),
                                                   (8, 103, 10, 3, 577, 32), (8, 1024, 1, 130, 8, 96), (8, 300, 7, 31, 449, 128)])
def test_probabilities_gradient_in_strips(chunks, B, H, N, M, d):
    blocks = lambda c: B * H * -(-N // 128) * -(-M // (64 * c))
    assert chunks == next(c for c in (1, 2, 4, 8) if c == 8 or blocks(2 * c) < 2048)
    g = torch.Generator(device=DEV).manual_seed(N * 131 + M)
    rnd = lambda *s: torch.randn(*s, generator=g, device=DEV).half()
    v, p, gc = rnd(B, M, H * d), rnd(B, H, N, M).requires_grad_(True), rnd(B, H, N, d)
    v.view(-1)[::3] = 0
    v.view(-1)[2::11] = float("nan")
    v.requires_grad_(True)
    gp, gv = torch.autograd.grad(bl.bgemm_attn_matmul.apply(p, head_split(v, H)), [p, v], gc)
    alone, = torch.autograd.grad(bl.bgemm_attn_matmul.apply(p, head_split(v.detach(), H)), [p], gc)
    sv = head_split(v.detach(), H)
    sv = ((sv > 0).double() - (sv < 0).double()).transpose(-1, -2).contiguous()
    assert torch.equal(gp, alone) and bound(d)(gp, gc.double() @ sv / 2, gc.double().abs() @ sv.abs() / 2)
    w, gd = (1 - (p.detach() == 0).double() / 2).transpose(-1, -2).contiguous(), gc.double()      # (randn in fp16 holds a zero now and then)
    merge = lambda t: t.permute(0, 2, 1, 3).reshape(B, -1, H * d)
    assert bound(N)(gv, merge(w @ gd), merge(w @ gd.abs()))


def test_other_forms_take_the_way_they_took(monkeypatch):
    """fp32 operands, one gradient only, gradients and operands in other strides, an infinite gradient, two dimensions."""
    g = torch.Generator(device=DEV).manual_seed(5)
    rnd = lambda *s: torch.randn(*s, generator=g, device=DEV)
    q, k, p = rnd(2, 40, 64), rnd(2, 50, 64), rnd(2, 40, 50)
    gs, gc = rnd(2, 50, 40).transpose(1, 2), rnd(2, 64, 40).transpose(1, 2)
    gs[0, 3, 4] = float("inf")

    def run(fn, a, b, up, which):
        a, b = a.detach().requires_grad_("a" in which), b.detach().requires_grad_("b" in which)
        leaves = [t for t in (a, b) if t.requires_grad]
        out = fn.apply(a, b)
        return torch.autograd.grad(out, leaves, up.to(out.dtype))

    cases = [(bl.bgemm_matmul, q, k.transpose(1, 2), gs), (bl.bgemm_matmul, q.half(), rnd(2, 64, 50).half(), gs),
             (bl.bgemm_matmul, q.transpose(0, 1).contiguous().transpose(0, 1).half(), k.half().transpose(1, 2), gs),
             (bl.bgemm_attn_matmul, p, k, gc), (bl.bgemm_attn_matmul, p.half().transpose(1, 2).contiguous().transpose(1, 2), k.half(), gc),
             (bl.bgemm_matmul, rnd(2, 40, 72).half()[..., 3:67], k.half().transpose(1, 2), gs), (bl.bgemm_matmul, q[0], k[0].T, gs[0])]
    functions = {bl.bgemm_matmul: Scores, bl.bgemm_attn_matmul: Context}
    ways = [[run(f(c[0]), *c[1:], which) for c in cases for which in ("a", "b", "ab")] for f in (lambda fn: fn, functions.get)]
    monkeypatch.setattr(bl, "_one_launch_grads", lambda *a: False)
    operations = [run(functions[c[0]], *c[1:], which) for c in cases for which in ("a", "b", "ab")]
    for have, want in zip(ways[0] + ways[1], operations + operations):
        assert len(have) == len(want)
        for x, y in zip(have, want):
            assert x.dtype == y.dtype and x.shape == y.shape
            # both round exact products' fp32 sums (at most 64 terms) to fp16: a last place apart
            assert torch.allclose(x.double(), y.double(), rtol=2.0 ** -9, atol=2.0 ** -10, equal_nan=True)


def test_tangents_of_the_upstream_gradients(monkeypatch):
    """Forward over reverse: the torch operations carry the tangent."""
    fwAD = torch.autograd.forward_ad
    g = torch.Generator(device=DEV).manual_seed(6)
    rnd = lambda *s: torch.randn(*s, generator=g, device=DEV).half()
    q, k, v, p = (t.requires_grad_(True) for t in (rnd(3, 40, 32), rnd(3, 50, 32), rnd(3, 50, 32), rnd(3, 40, 50)))
    up = [rnd(3, 40, 50), rnd(3, 40, 32)]
    scores, context = bl.bgemm_matmul.apply(q, k.transpose(-1, -2)), bl.bgemm_attn_matmul.apply(p, v)

    def run():
        with fwAD.dual_level():
            duals = [fwAD.make_dual(t, t * 2) for t in up]
            return [t for o in torch.autograd.grad([scores, context], [q, k, v, p], duals, retain_graph=True) for t in fwAD.unpack_dual(o)]

    got = run()
    monkeypatch.setattr(bl, "_one_launch_grads", lambda *a: False)
    for a, b in zip(got, run()):
        assert torch.equal(a, b)


def test_a_mode_sees_the_operations_of_the_gradients():
    from torch.utils._python_dispatch import TorchDispatchMode

    class Operations(TorchDispatchMode):
        names = []

        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            self.names.append(func.overloadpacket._qualified_op_name.split("::")[1])
            return func(*args, **(kwargs or {}))

    rnd = lambda *s: torch.randn(*s, device=DEV).half().requires_grad_(True)
    q, k, v, p = rnd(3, 40, 32), rnd(3, 50, 32), rnd(3, 50, 32), rnd(3, 40, 50)
    scores, context = bl.bgemm_matmul.apply(q, k.transpose(-1, -2)), bl.bgemm_attn_matmul.apply(p, v)
    with Operations() as mode:
        torch.autograd.grad([scores, context], [q, k, v, p], [torch.ones_like(scores), torch.ones_like(context)])
    assert mode.names.count("bmm") == 4
