"""The native host side of inference and attention against the Python forms behind it: the same results, bit for bit, over the orders,
strides, types and sizes that both take, the same refusals, and updates of parameters seen."""
import pytest
import torch

pytestmark = pytest.mark.gpu

import _lib
import attention_demo
import bgemm_linear as bl
import lowbit_kernel as lk

DEV = "cuda:0"


@pytest.fixture
def both(monkeypatch):
    """both(fn) -> fn() with the native part and fn() without; an exception stands for a result."""
    def run(fn):
        got = []
        for native in (True, False):
            with monkeypatch.context() as m:
                if not native:
                    m.setattr(_lib, "_native", None)
                    m.setattr(_lib, "_native_looked_for", True)
                assert (_lib.native_or_none() is not None) == native
                try:
                    got.append(fn())
                except Exception as e:
                    got.append(e)
        return got
    return run


def same(a, b):
    if isinstance(a, Exception) or isinstance(b, Exception):
        return type(a) is type(b)
    if isinstance(a, (tuple, list)):
        return len(a) == len(b) and all(same(x, y) for x, y in zip(a, b))
    if isinstance(a, lk.PackedBits):
        return (a.rows, a.K, a.batch) == (b.rows, b.K, b.batch) and torch.equal(lk.logical_from_tiled(a), lk.logical_from_tiled(b))
    if a is None or b is None:
        return a is b
    return a.dtype == b.dtype and a.shape == b.shape and torch.equal(a.nan_to_num(), b.nan_to_num())


def rnd(*shape, dt=torch.float32, seed=1):
    return torch.randn(*shape, generator=torch.Generator(device=DEV).manual_seed(seed + sum(shape)), device=DEV).to(dt)


def inputs(K, dt):
    """One to many rows: dense, with leading dimensions, transposed, with gaps, expanded, at odd addresses, empty."""
    base = rnd(70, K + 5, dt=dt)
    return [base[:1, :K].contiguous(), base[:3, 1:K + 1], base[:, 2:K + 2], base[:, :K].contiguous(), rnd(K, 9, dt=dt).T, base[:1, :K].expand(6, K), rnd(2, 5, K, dt=dt),
            rnd(5, 2, K, dt=dt).transpose(0, 1), rnd(K, dt=dt), rnd(0, K, dt=dt)]


@pytest.mark.parametrize("dt", [torch.float32, torch.half])
@pytest.mark.parametrize("K, M", [(40, 33), (300, 64), (1100, 257), (2100, 70)])
def test_linear_layers(both, K, M, dt):
    lin = bl.BGEMMLinear(K, M, bias=K != 300).to(DEV).to(dt)
    with torch.no_grad():
        lin(rnd(64, K, dt=dt))
        for x in inputs(K, dt) + [rnd(5, K, dt=torch.half if dt == torch.float32 else torch.float32), rnd(5, K + 1, dt=dt)]:
            assert same(*both(lambda: lin(x)))
        x = rnd(7, K, dt=dt)
        before = lin(x)
        for change in (lambda: lin.weight.neg_(), lambda: lin.zpw.add_(0.01), lambda: lin.sw.mul_(2), lambda: setattr(lin, "sa", torch.nn.Parameter(lin.sa.detach() * 3)),
                       lambda: lin.zpa.add_(0.5), lambda: lin.train(), lambda: setattr(lin, "fuse_inference", False), lambda: setattr(lin, "zpa", lin.zpa.double())):
            change()
            after = both(lambda: lin(x))
            assert same(*after)
        assert not torch.equal(before, after[0])
    assert lin(x).requires_grad


@pytest.mark.parametrize("dt", [torch.float32, torch.half])
def test_chains(both, dt):
    chain = bl.BGEMMChain(bl.BGEMMLinear(300, 500, bias=True), bl.BGEMMLinear_bireal(500, 256), bl.BGEMMLinear(256, 10, bias=True)).to(DEV).to(dt)
    with torch.no_grad():
        chain(rnd(64, 300, dt=dt))
        for _ in range(2):                                                 # the second time the buffers are there
            for x in inputs(300, dt):
                assert same(*both(lambda: chain(x)))
        x = rnd(40, 300, dt=dt)
        chain[1].weight.neg_()
        a, b = both(lambda: chain(x))
        h = x
        for layer in chain:
            h = layer(h)
        assert same(a, b) and torch.equal(a, h)


@pytest.mark.parametrize("N", [1, 2, 5, 33, 600])
def test_products(both, N):
    K, M = 520, 130
    w, wh = rnd(M, K), rnd(M, K).half()
    wp = lk.pack_sign(w)
    x = rnd(N, K + 3)[:, 1:K + 1]
    x[:, ::4] = 0
    sw, sa, bias = rnd(M).abs(), rnd(1).abs(), rnd(M)
    for dt in (torch.float32, torch.half):
        xd = x.to(dt)
        for mode in (lk.MODE_AND, lk.MODE_XOR, lk.MODE_ATTN, lk.MODE_BWTA, 9):
            for out in (torch.int32, torch.half, torch.float64):
                assert same(*both(lambda: lk.bgemm_packed_weight_forward(wp, xd, mode, out)))
            for sdt in (torch.float32, torch.half):
                scale = (sw.to(sdt), sa.to(sdt), bias.to(sdt))
                for s in (scale, scale[:2] + (None,), (scale[0][1:],) + scale[1:], (scale[0].cpu(),) + scale[1:], (scale[0].double(),) + scale[1:]):
                    assert same(*both(lambda: lk.bgemm_packed_weight_forward(wp, xd, mode, scale=s)))
            assert same(*both(lambda: lk.bgemm_packed_weight_forward(wp, xd, mode, x_zero_point=rnd(1))))
        xp = lk.pack_ternary(xd)
        for mode, p in ((lk.MODE_XOR, lk.pack_sign(xd)), (lk.MODE_BWTA, xp), (lk.MODE_XOR, xp), (lk.MODE_ATTN_X, lk.pack_sign(rnd(3, N, K)))):
            for out in (torch.int32, torch.half, torch.float32):
                assert same(*both(lambda: lk.bgemm_packed_forward(wp, p, mode, out)))
    for instr in (0, 1, 2, 3):
        for split in (1, 3, 0):
            assert same(*both(lambda: lk.bgemm_linear_forward_cuda(x.half(), wh, split, instr)))
    assert same(*both(lambda: lk.bgemm_linear_forward_cuda(rnd(K, N).half().T, wh[:, ::2].repeat_interleave(2, 1), 1, 1)))
    assert same(*both(lambda: lk.bgemm_linear_forward_cuda(x, wh, 1, 1))) and same(*both(lambda: lk.bgemm_linear_forward_cuda(x.half(), wh[:, 1:], 1, 1)))


@pytest.mark.parametrize("dt", [torch.float32, torch.half])
def test_batched_products_and_their_gradients(both, dt):
    B, H, S, d = 2, 3, 37, 64
    split = lambda t: t.view(B, S, H, d).permute(0, 2, 1, 3)
    q, k, v = (rnd(B, S, H * d, dt=dt, seed=i) for i in range(3))
    p = rnd(B, H, S, S, dt=dt)
    pairs = [(bl.bgemm_matmul, split(q), split(k).transpose(-1, -2)), (bl.bgemm_attn_matmul, p, split(v)), (bl.bgemm_matmul, split(q), split(k).transpose(-1, -2).contiguous()),
             (bl.bgemm_matmul, split(q)[0], split(k)[0].transpose(-1, -2)), (bl.bgemm_matmul, split(q).transpose(-1, -2), split(k)), (bl.bgemm_matmul, split(q)[:, :1], split(k).transpose(-1, -2)),
             (bl.bgemm_matmul, split(q).expand(B, H, S, d)[..., :40], split(k).transpose(-1, -2)[..., :40, :]), (bl.bgemm_attn_matmul, p.transpose(-1, -2), split(v)),
             (bl.bgemm_matmul, q[:1].unsqueeze(0).expand(2, 3, S, H * d), k[:1].unsqueeze(0).expand(2, 3, S, H * d).transpose(-1, -2))]
    for fn, a, b in pairs:
        with torch.no_grad():
            assert same(*both(lambda: fn.apply(a, b)))

        def step():
            x, y = a.detach().requires_grad_(), b.detach().requires_grad_()
            out = fn.apply(x, y)
            return [out.detach(), *torch.autograd.grad(out, [x, y], rnd(*out.shape, dt=torch.half))]

        assert same(*both(step))


@pytest.mark.parametrize("dt", [torch.float32, torch.half])
def test_attention_block(both, dt):
    block = attention_demo.BinarySelfAttention(192, 3).to(DEV).to(dt)
    with torch.no_grad():
        block(rnd(2, 50, 192, dt=dt))
        for x in (rnd(2, 50, 192, dt=dt), rnd(50, 2, 192, dt=dt).transpose(0, 1), rnd(2, 50, 200, dt=dt)[..., :192], rnd(1, 1, 192, dt=dt), rnd(2, 5, 190, dt=dt)):
            assert same(*both(lambda: block(x)))
        x = rnd(2, 50, 192, dt=dt)
        for change in (lambda: block.dense.weight.neg_(), lambda: block.query.weight.neg_(), lambda: block.dense.zpa.add_(1.0), lambda: setattr(block.dense, "zpa", block.dense.zpa.double()),
                       lambda: block.dense.register_forward_hook(lambda m, i, o: o * 2), lambda: setattr(block, "dense", torch.nn.Linear(192, 192).to(DEV).to(dt))):
            change()
            assert same(*both(lambda: block(x)))
