"""Both attention products in one launch on fp16 operands against packing and multiplying them: the same integers, bit for bit."""
import pytest
import torch

pytestmark = pytest.mark.gpu

import _lib
import bgemm_linear as bl
import lowbit_kernel as lk

DEV = "cuda:0"


def packed_way(fn, monkeypatch):
    with monkeypatch.context() as m:
        m.setattr(_lib, "_native", None)
        m.setattr(_lib, "_native_looked_for", True)
        return fn()


def operand(g, shape, order):
    """fp16 with zeros of both signs, NaNs and infinities, its batch as `order` says."""
    B, H, N, D = shape
    if order == "dense":
        t = torch.randn(B, H, N, D, generator=g, device=DEV).half()
    elif order == "heads":                                        # a view of [B, N, H * D]
        t = torch.randn(B, N, H, D, generator=g, device=DEV).half().permute(0, 2, 1, 3)
    elif order == "odd":                                          # rows and matrices at odd element offsets
        t = torch.randn(B, H, N + 1, D + 3, generator=g, device=DEV).half()[:, :, 1:, 1:D + 1]
    else:                                                         # one matrix for all heads
        t = torch.randn(B, 1, N, D, generator=g, device=DEV).half().expand(B, H, N, D)
    if order != "shared":
        flat = torch.randint(0, 9, t.shape, generator=g, device=DEV)
        for at, value in enumerate((0.0, -0.0, float("nan"), -float("inf"))):
            t[flat == at] = value
    return t


# edges of the 32-row waves, the 128-row blocks, the 64- and 256-column groups; every D; the context's longest rows at each
SHAPES = [(1, 1, 1, 1, 32), (1, 2, 3, 7, 64), (2, 3, 31, 8, 96), (2, 1, 33, 9, 128), (1, 2, 128, 64, 32), (3, 2, 129, 65, 64), (1, 3, 127, 255, 96), (2, 2, 64, 256, 128),
          (1, 2, 97, 257, 64), (2, 12, 200, 321, 32), (1, 1, 40, 1024, 128), (1, 1, 40, 1025, 128), (1, 1, 33, 2048, 64), (1, 2, 5, 4096, 32), (1, 1, 5, 4097, 32), (4, 12, 512, 512, 64)]


@pytest.mark.parametrize("order", ["dense", "heads", "odd", "shared"])
@pytest.mark.parametrize("B, H, N, M, D", SHAPES)
def test_products(B, H, N, M, D, order, monkeypatch):
    g = torch.Generator(device=DEV).manual_seed(N * 131 + M)
    q, k, v = operand(g, (B, H, N, D), order), operand(g, (B, H, M, D), order), operand(g, (B, H, M, D), order)
    p = operand(g, (B, H, N, M), order)
    for mode in ("xor", "and"):
        fn = lambda: bl.bgemm_matmul.apply(q, k.transpose(-1, -2), mode)
        assert torch.equal(fn(), packed_way(fn, monkeypatch))
    fn = lambda: bl.bgemm_attn_matmul.apply(p, v)
    assert torch.equal(fn(), packed_way(fn, monkeypatch))


def test_three_dimensions_and_other_forms(monkeypatch):
    g = torch.Generator(device=DEV).manual_seed(5)
    q, k, p = (torch.randn(6, n, m, generator=g, device=DEV) for n, m in ((70, 64), (90, 64), (70, 90)))
    right = k.transpose(-1, -2)
    for a, b, c in ((q.half(), right.half(), p.half()), (q, right, p), (q.half(), right, p.half()),
                    (q.half(), right.half().contiguous(), p.half().transpose(-1, -2).contiguous().transpose(-1, -2)),
                    (q[..., :40].half(), right[:, :40].half(), p.half())):
        fn = lambda: bl.bgemm_matmul.apply(a, b)
        assert torch.equal(fn(), packed_way(fn, monkeypatch))
        fn = lambda: bl.bgemm_attn_matmul.apply(c, b.transpose(-1, -2))
        assert torch.equal(fn(), packed_way(fn, monkeypatch))


def test_refusals():
    out = torch.empty(1, 64, 64, dtype=torch.half, device=DEV)
    strides = (_lib.ctypes.c_int64 * 6)(0, 0, 64, 0, 0, 64)
    call = lambda D=64, M=64, mode=lk.MODE_XOR: (
        _lib.lib().bgemm_scores_forward(mode, out.data_ptr(), out.data_ptr(), strides, 1, 1, 64, M, D, out.data_ptr(), None),
        _lib.lib().bgemm_context_forward(out.data_ptr(), out.data_ptr(), strides, 1, 1, 64, M, D, out.data_ptr(), None))
    assert all(call(D=48)) and all(call(M=0)) and call(M=7, mode=lk.MODE_ATTN)[0] and call(M=7, mode=lk.MODE_ATTN)[1] and call(M=1 << 17, mode=9)[1]
