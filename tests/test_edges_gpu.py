"""Products whose tiles beside the whole 256 x 128 ones go to 32 x 32 blocks of the same launch, against the popcount kernel: the same
integers, and values made of them, and nothing written past the output."""
import pytest
import torch

pytestmark = pytest.mark.gpu

import _lib as B
import lowbit_kernel as lk

DEV = "cuda:0"
# rows and columns beside 256 tiles (edge blocks last) and 512 (first): one, all but one of a tile's, none; K-tiles 24, 25, 33, 12, 17
SHAPES = [(1025, 8193, 6139), (1055, 8192, 6400), (1024, 8223, 8200), (2049, 8193, 3072), (2079, 8192, 4345), (2048, 8319, 4096), (8193, 2050, 4100)]


def operands(N, M, K, seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    return [lk.pack_sign(torch.randn(r, K, generator=g, device=DEV).half()) for r in (M, N)]


@pytest.mark.parametrize("N, M, K", SHAPES)
def test_edge_tiles(N, M, K):
    w, x = operands(N, M, K, N + M)
    g = torch.Generator(device=DEV).manual_seed(1)
    for mode in (lk.MODE_XOR, lk.MODE_AND, lk.MODE_ATTN, lk.MODE_ATTN_X):
        assert lk.packed_kernel_id(w, x, mode) == B.KERNEL_MFMA_256x128
        want = lk.bgemm_packed_forward(w, x, mode, torch.int32, variant=B.VARIANT_VALU)
        assert torch.equal(lk.bgemm_packed_forward(w, x, mode, torch.int32), want)
        assert torch.equal(lk.bgemm_packed_forward(w, x, mode, torch.half), want.half())
    # into the middle of a larger buffer: what lies around the output stays
    whole = torch.full((N * M + 64,), -7, dtype=torch.int32, device=DEV)
    want = lk.bgemm_packed_forward(w, x, lk.MODE_XOR, torch.int32, variant=B.VARIANT_VALU)
    lk.bgemm_packed_forward(w, x, lk.MODE_XOR, torch.int32, out=whole[32:32 + N * M].view(1, N, M))
    assert torch.equal(whole[32:32 + N * M].view(1, N, M), want) and (whole[:32] == -7).all() and (whole[-32:] == -7).all()
    for dt in (torch.float32, torch.half):
        scale = (torch.rand(M, generator=g, device=DEV).to(dt), torch.rand(1, generator=g, device=DEV).to(dt), torch.randn(M, generator=g, device=DEV).to(dt))
        for bias in (scale[2], None):
            got = lk.bgemm_packed_forward(w, x, lk.MODE_XOR, dt, scale=(*scale[:2], bias))
            assert torch.equal(got, lk.bgemm_packed_forward(w, x, lk.MODE_XOR, dt, scale=(*scale[:2], bias), variant=B.force_kernel(B.KERNEL_MFMA_256x128)))
    lk.row_popcounts(w), lk.row_popcounts(x)
    assert torch.equal(lk.bgemm_packed_forward(w, x, lk.MODE_XOR, torch.int32), want)


@pytest.mark.parametrize("N, M, K", [(2000, 3001, 2048), (300, 515, 2300), (4096, 4104, 2048)])
def test_int32_rows_that_share_lines(N, M, K):
    # past the caches and through them, by the output's size
    w, x = operands(N, M, K, 3)
    assert torch.equal(lk.bgemm_packed_forward(w, x, lk.MODE_XOR, torch.int32), lk.bgemm_packed_forward(w, x, lk.MODE_XOR, torch.int32, variant=B.VARIANT_VALU))
