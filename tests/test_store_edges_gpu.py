"""The matrix-core kernels' stores at the edges of a row: rows of any length, outputs that start at any element address, every tile.
Exact against torch (the sums are integers; scaling rounds step by step), and nothing beside the output is written."""
import pytest
import torch

pytestmark = pytest.mark.gpu

import _lib
import lowbit_kernel as lk

DEV = "cuda:0"
TILES = [_lib.KERNEL_MFMA_256x256, _lib.KERNEL_MFMA_256x128, _lib.KERNEL_MFMA_128x128, _lib.KERNEL_MFMA_64x128, _lib.KERNEL_MFMA_32x128,
         _lib.KERNEL_MFMA_32x256, _lib.KERNEL_MFMA_64x64, _lib.KERNEL_MFMA_128x64]


@pytest.mark.parametrize("M, N, K, offset", [(1, 1, 64, 0), (3, 33, 300, 1), (7, 40, 100, 0), (9, 64, 4500, 3), (130, 37, 260, 1), (263, 257, 2100, 0),
                                             (264, 31, 64, 4), (136, 300, 300, 8), (1030, 65, 4345, 0)])
def test_rows_of_any_length_at_any_address(M, N, K, offset):
    g = torch.Generator(device=DEV).manual_seed(M * 1009 + N)
    w, x = (torch.randn(r, K, generator=g, device=DEV).half() for r in (M, N))
    wp, xp = lk.pack_sign(w), lk.pack_sign(x)
    pm = lambda t: torch.where(torch.signbit(t), -1.0, 1.0)
    acc = (pm(x) @ pm(w).T).half()                      # integers up to K < 2^24: exact in fp32
    lib, st = _lib.lib(), torch.cuda.current_stream().cuda_stream
    for kind, dt in ((_lib.OUT_F16, torch.half), (_lib.OUT_F16_SCALED, torch.half), (_lib.OUT_F32_SCALED, torch.float32)):
        sw, sa, bias = (torch.randn(s, generator=g, device=DEV).to(dt) for s in (M, 1, M))
        want = acc if kind == _lib.OUT_F16 else acc * sw * sa + bias
        for tile in TILES:
            buf = torch.full((offset + N * M + 16,), 77.0, device=DEV, dtype=dt)
            at = buf.data_ptr() + offset * buf.element_size()
            variant = _lib.force_kernel(tile, _lib.VARIANT_MFMA_F4)
            args = (_lib.MODE_XOR, wp.data.data_ptr(), xp.data.data_ptr(), None, at, kind, 1, M, N, K, 0, 0, N * M, 1, variant, None, 0, None, 0)
            if kind == _lib.OUT_F16:
                _lib.check(lib.bgemm_packed_forward(*args, st))
            else:
                _lib.check(lib.bgemm_packed_forward_scaled(*args, sw.data_ptr(), sa.data_ptr(), bias.data_ptr(), st))
            got = buf[offset:offset + N * M].reshape(N, M)
            assert torch.equal(got, want), (kind, tile, int((got != want).sum()))
            assert (buf[:offset] == 77).all() and (buf[offset + N * M:] == 77).all(), (kind, tile)
