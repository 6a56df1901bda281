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


# edges of the 32-row waves, the 128-row blocks, the 64- and 256-column groups; every D; rows too long for the context's kernel (below: at its limits)
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


def packed_product(a, right, mode):
    """a @ right over both leading dimensions by the packs and the general product."""
    B, H, N, K = a.shape
    w = lk.pack_sign_transposed(right.reshape(B * H, K, -1))
    return lk.bgemm_packed_forward(w, lk.pack_sign(a.reshape(B * H, N, K)), mode, torch.half).view(B, H, N, -1)


def strides_of(*tensors):
    return (_lib.ctypes.c_int64 * 6)(*(n for t in tensors for n in (t.stride(0), t.stride(1), t.stride(2))))


# as long a row as the entry point takes at each D and one beside it; one and two parts a row; more than 512 blocks of long rows
@pytest.mark.parametrize("B, H, N, M, D", [(1, 2, 33, 1024, 128), (2, 1, 33, 1365, 96), (2, 1, 129, 1300, 96), (1, 2, 40, 2048, 64), (1, 3, 33, 2000, 64), (1, 2, 5, 4096, 32),
                                           (1, 1, 130, 4090, 32), (1, 2, 140, 255, 128), (1, 2, 140, 256, 128), (64, 9, 100, 300, 32), (60, 9, 100, 256, 128)])
def test_the_contexts_kernel_at_its_limits(B, H, N, M, D):
    g = torch.Generator(device=DEV).manual_seed(M + D)
    for order in ("dense", "odd"):
        p, v = operand(g, (B, H, N, M), order), operand(g, (B, H, M, D), order)
        p[..., :N // 2, :] = p[..., :N // 2, :].abs()              # rows that count every value: the largest sums
        v[..., ::2] = -v[..., ::2].abs()
        out = torch.empty(B, H, N, D, dtype=torch.half, device=DEV)
        _lib.check(_lib.lib().bgemm_context_forward(p.data_ptr(), v.data_ptr(), strides_of(p, v), B * H, H, N, M, D, out.data_ptr(), None))
        assert torch.equal(out, packed_product(p, v, lk.MODE_ATTN_X))


# blocks of eight waves (256 rows, from 192 of them on) at every D that has them, and of four; whole and ragged column blocks
@pytest.mark.parametrize("D", [32, 64, 96, 128])
@pytest.mark.parametrize("B, H, N, M", [(16, 12, 256, 64), (16, 12, 200, 64), (8, 12, 250, 300), (8, 12, 511, 31), (2, 3, 256, 300),
                                        # a matrix's blocks on one XCD: broken rows (and 499, which are not), many operands, also of D = 32 up to 512 columns
                                        (3, 3, 130, 501), (3, 3, 130, 499), (11, 9, 520, 512), (11, 9, 520, 576)])
def test_the_scores_kernel_in_blocks_of_four_and_eight_waves(B, H, N, M, D):
    g = torch.Generator(device=DEV).manual_seed(N + M + D)
    q, k = operand(g, (B, H, N, D), "heads"), operand(g, (B, H, M, D), "odd")
    for mode in (lk.MODE_XOR, lk.MODE_AND):
        out = torch.empty(B, H, N, M, dtype=torch.half, device=DEV)
        _lib.check(_lib.lib().bgemm_scores_forward(mode, q.data_ptr(), k.data_ptr(), strides_of(q, k), B * H, H, N, M, D, out.data_ptr(), None))
        assert torch.equal(out, packed_product(q, k.transpose(-1, -2), mode))


# both sides of the lines: (batch, heads, rows, columns, D), scores in one launch, context in one launch
@pytest.mark.parametrize("B, H, N, M, D, scores, context", [
    (1, 1, 40, 1024, 32, True, True), (1, 1, 40, 1025, 32, True, False), (2, 1, 40, 2048, 32, True, True), (2, 1, 40, 2049, 32, True, False), (1, 1, 40, 1024, 64, True, False),
    (1, 2, 40, 1024, 64, True, True), (1, 2, 40, 1025, 64, True, False), (2, 1, 40, 341, 96, True, True), (2, 1, 40, 342, 96, True, False), (1, 1, 40, 256, 128, True, True),
    (2, 1, 40, 257, 128, True, False), (2, 1, 40, 64, 40, False, False), (1, 1, 9, 7, 32, True, False), (8, 8, 2048, 1024, 64, False, False), (8, 8, 2047, 1024, 64, True, True)])
def test_products_go_where_they_are_ahead(B, H, N, M, D, scores, context):
    """Seen from what a call allocates: its output alone, or the packed operands beside it."""
    g = torch.Generator(device=DEV).manual_seed(7)
    q, k, v, p = (torch.randn(B, H, n, d, generator=g, device=DEV).half() for n, d in ((N, D), (M, D), (M, D), (N, M)))
    count = lambda: torch.cuda.memory_stats()["allocation.all.allocated"]
    for fn, one in ((lambda: bl.bgemm_matmul.apply(q, k.transpose(-1, -2)), scores), (lambda: bl.bgemm_attn_matmul.apply(p, v), context)):
        before = count()
        out = fn()
        assert count() - before == (1 if one else 2)
        del out
