"""Training the scaled binary Linear as one node against the separate operations it stands for, at the edges of its kernels'
tiles: rows, columns and contractions around multiples of 32, 64 and 256, exact zeros of both signs in both operands, every
subset of gradients.

Tolerances.  The output and g16 are rounded step by step as torch rounds them: equal.  The products' terms are g16 * {-1, 0, 1},
exact; R of them summed in fp32 in any order are within R * 2^-24 * sum|g16| of the true sum, and the separate operations round that
to fp16 (2^-11 relative, 2^-25 below the normal range) once more; Bi-Real's factor (at most 2, itself the same fp16 number on both
sides) and the rounding of its product twice more.  The scales' gradients are fp32 sums of N (N * M) products; in fp16 the
separate operations also round every product (2^-11 each) and both round the sum."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

import bgemm_linear as bl

DEV = "cuda:0"
SHAPES = [(1, 1, 2), (31, 63, 33), (32, 256, 64), (33, 257, 65), (64, 64, 1000), (200, 784, 31), (97, 100, 129), (700, 300, 515), (1030, 33, 66),
          (2100, 520, 130)]


def layer_and_inputs(cls, N, K, M, dtype, bias, seed=0):
    torch.manual_seed(seed)
    lin = cls(K, M, bias=bias).to(DEV).to(dtype)
    x = torch.randn(N, K, device=DEV, dtype=dtype)
    lin(torch.randn(64, K, device=DEV, dtype=dtype))              # sets the scales
    with torch.no_grad():
        # scales of one (the initial ones are so small that fp16 gradients vanish), zero points that some elements equal
        lin.sw.copy_(torch.rand_like(lin.sw) + 0.5)
        lin.sa.fill_(0.75)
        x.view(-1)[::7] = lin.zpa
        lin.weight.view(-1)[::5] = lin.zpw
    g = (torch.randn(N, M, device=DEV) * 0.05).to(dtype)
    return lin, x.requires_grad_(True), g


def grads(lin, x, g, wanted):
    y = lin(x)
    return [y.detach()] + list(torch.autograd.grad(y, wanted, g))


@pytest.mark.parametrize("cls", [bl.BGEMMLinear, bl.BGEMMLinear_bireal])
@pytest.mark.parametrize("dtype", [torch.float32, torch.half])
@pytest.mark.parametrize("N, K, M", SHAPES)
def test_one_node_gives_what_the_separate_operations_give(cls, dtype, N, K, M):
    bias = (N + M) % 2 == 0
    lin, x, g = layer_and_inputs(cls, N, K, M, dtype, bias)
    wanted = [x, lin.weight, lin.sw, lin.sa] + ([lin.bias] if bias else [])
    assert lin(x).grad_fn.name() == "ScaledBinaryLinearBackward"
    got = grads(lin, x, g, wanted)
    lin.fuse_training = False
    want = grads(lin, x, g, wanted)
    assert torch.equal(got[0], want[0])
    d = lambda t: t.detach().double()
    g16 = ((g * lin.sa.detach()) * lin.sw.detach()).half()
    eps, tiny = 2.0 ** -11, 2.0 ** -25
    rounds = (1 if cls is bl.BGEMMLinear else 3) * (1 if dtype == torch.float32 else 2)
    factor = 1.0 if cls is bl.BGEMMLinear else 2.0
    bound_x = rounds * (eps * d(want[1]).abs() + factor * tiny) + factor * M * 2.0 ** -24 * d(g16).abs().sum(1, keepdim=True)
    assert (d(got[1]) - d(want[1])).abs().le(bound_x).all()
    w_rounds = 1 if dtype == torch.float32 else 2
    bound_w = w_rounds * (eps * d(want[2]).abs() + tiny) + N * 2.0 ** -24 * d(g16).abs().sum(0)[:, None]
    assert (d(got[2]) - d(want[2])).abs().le(bound_w).all()
    # the scales' gradients against float64
    pm = lambda t: torch.where(torch.signbit(t), -1.0, 1.0).double()
    acc = pm((x - lin.zpa).half()) @ pm((lin.weight - lin.zpw).half()).T
    acc16, sa, sw = acc.half().double(), d(lin.sa), d(lin.sw)
    gs = d(g * lin.sa.detach())
    rel = 2.0 ** -24 * (N + 8) if dtype == torch.float32 else 2.0 ** -10
    terms_sw, terms_sa = gs * acc16, d(g) * (acc16 * sw)
    assert (d(got[3]) - terms_sw.sum(0)).abs().le(rel * terms_sw.abs().sum(0) + tiny).all()
    rel_sa = 2.0 ** -24 * (N * 2 + M) if dtype == torch.float32 else 2.0 ** -10
    assert float((d(got[4]) - terms_sa.sum()).abs()) <= rel_sa * float(terms_sa.abs().sum()) + tiny
    if bias:
        assert (d(got[5]) - d(g).sum(0)).abs().le(rel * d(g).abs().sum(0) + tiny).all()


@pytest.mark.parametrize("dtype", [torch.float32, torch.half])
def test_any_subset_of_gradients_leading_dimensions_and_strides(dtype):
    lin, x, g = layer_and_inputs(bl.BGEMMLinear, 60, 100, 70, dtype, True)
    full = grads(lin, x, g, [x, lin.weight, lin.sw, lin.sa, lin.bias])
    y = lin(x.detach())                                        # the first layer of a network: no input gradient
    for a, b in zip(torch.autograd.grad(y, [lin.weight, lin.bias], g), (full[2], full[5])):
        assert torch.equal(a, b)
    lin.weight.requires_grad_(False)
    assert torch.equal(torch.autograd.grad(lin(x), [x], g)[0], full[1])
    lin.weight.requires_grad_(True)
    x3 = x.detach().reshape(3, 4, 5, 100).requires_grad_(True)
    g3 = g.reshape(3, 4, 5, 70)
    y3 = lin(x3)
    assert torch.equal(y3.detach().reshape(60, 70), full[0])
    assert torch.equal(torch.autograd.grad(y3, x3, g3)[0].reshape(60, 100), full[1])
    # a row slice with a stride, an expanded upstream gradient
    wide = torch.cat([x.detach(), x.detach()], 1)[:, :100].requires_grad_(True)
    assert torch.equal(torch.autograd.grad(lin(wide), wide, g)[0], full[1])
    one = torch.ones((), device=DEV, dtype=dtype).expand(60, 70)
    assert torch.equal(torch.autograd.grad(lin(x), x, one)[0], torch.autograd.grad(lin(x), x, one.contiguous())[0])


def test_gradients_can_be_differentiated_and_modified_scales_are_refused():
    lin, x, g = layer_and_inputs(bl.BGEMMLinear, 32, 64, 48, torch.float32, True)
    out = {}
    for fused in (True, False):
        lin.fuse_training = fused
        gx, gsw = torch.autograd.grad(lin(x), [x, lin.sw], g, create_graph=True)
        out[fused] = [t.detach() for t in torch.autograd.grad(gx.sum() + (gsw ** 2).sum(), [lin.sa, lin.sw], allow_unused=True) if t is not None]
    assert len(out[True]) == len(out[False]) and all(torch.equal(a, b) for a, b in zip(out[True], out[False]))
    lin.fuse_training = True
    y = lin(x)
    with torch.no_grad():
        lin.sw.mul_(2.0)
    with pytest.raises(RuntimeError):
        torch.autograd.grad(y, x, g)


@pytest.mark.parametrize("N, K, M", SHAPES)
def test_learned_scale_layer_as_one_node(N, K, M):
    """Against the separate operations (torch's own means, fp32 matmul).  The upstream gradient's three bf16 planes hold all of its bits
    and the products' terms are exact, so the two sides differ by the order of fp32 sums of R terms (R * 2^-24 * sum|terms|), the means'
    last bits (an element within 2^-22 of its operand's mean would flip: none does here), and a few roundings of the surrogate (cosh
    within 4 ulp on either side: 2^-20)."""
    torch.manual_seed(N + K)
    lin = bl.BGEMMLinear_elastic_signed(K, M).to(DEV)
    x = torch.randn(N, K, device=DEV) * 1.5 + 0.25
    lin(torch.randn(64, K, device=DEV))
    with torch.no_grad():
        lin.sw.copy_(torch.rand_like(lin.sw) + 0.5)
        lin.sa.fill_(0.75 if M % 2 else -0.75)
    x.requires_grad_(True)
    g = torch.randn(N, M, device=DEV) * torch.logspace(-6, 2, M, device=DEV)
    wanted = [x, lin.weight, lin.sa, lin.sw, lin.bias]
    assert lin(x).grad_fn.name() == "ElasticBinaryLinearBackward"
    got = grads(lin, x, g, wanted)
    lin.fuse_training = False
    want = grads(lin, x, g, wanted)
    assert torch.equal(got[0], want[0])
    d = lambda t: t.detach().double()
    xs, ws = (d(x) - d(x).mean()) / d(lin.sa), d(lin.weight) - d(lin.weight).mean()
    ga = d(g).abs()
    sur = lambda t: 2 / torch.cosh(t.abs().clamp(max=4)) ** 2
    assert ((d(got[1]) - d(want[1])).abs() <= sur(xs) * (M + 8) * 2.0 ** -23 * ga.sum(1, keepdim=True) + 2.0 ** -19 * d(want[1]).abs()).all()
    assert ((d(got[2]) - d(want[2])).abs() <= sur(ws) * (N + 8) * 2.0 ** -23 * ga.sum(0)[:, None] + 2.0 ** -19 * d(want[2]).abs()).all()
    f, h = d(g) @ ws.sign(), d(g).T @ xs.sign()
    inner = (xs > 1).double() - (xs < -1).double() + (xs.abs() <= 1) * (xs.sign() - xs)
    c = lin.grad_scale
    slack = 2.0 ** -20 * (N + M + K)
    assert float((d(got[3]) - (inner * f * c).sum()).abs()) <= slack * float((inner.abs() * ga.sum(1, keepdim=True) * c).sum())
    assert ((d(got[4]) - (ws.sign() * h * c).sum(1)).abs() <= slack * c * K * ga.sum(0)).all()
    assert ((d(got[5]) - d(g).sum(0)).abs() <= N * 2.0 ** -24 * ga.sum(0)).all()
    lin.fuse_training = True
    x3 = x.detach()[: N // 2 * 2].reshape(2, N // 2, K).requires_grad_(True) if N > 1 else x
    if N > 1:                                                # leading dimensions, a subset of gradients
        y3 = lin(x3)
        assert y3.shape == (2, N // 2, M)
        a = torch.autograd.grad(y3, [lin.weight, lin.bias], g[: N // 2 * 2].reshape(2, N // 2, M))
        lin.fuse_training = False
        b = torch.autograd.grad(lin(x3), [lin.weight, lin.bias], g[: N // 2 * 2].reshape(2, N // 2, M))
        for p, q in zip(a, b):
            assert torch.allclose(p, q, rtol=1e-4, atol=1e-4 * float(q.abs().max()))
