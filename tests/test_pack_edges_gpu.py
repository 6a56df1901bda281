"""The pack kernel at its edges: rows that start at any element address, last chunks of one to eight elements, short rows,
both sides of the number of tiles at which a wave takes a whole tile.  Bit for bit against the CPU oracle."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

import lowbit_kernel as lk

DEV = "cuda:0"


def values(rng, rows, K, dtype):
    x = rng.standard_normal((rows, K)).astype(dtype)
    z = rng.random((rows, K))
    x[z < 0.1] = 0.0
    x[z < 0.05] = -0.0
    # around half the smallest fp16 number, where rounding an fp32 value to fp16 gives zero or not
    for i, v in enumerate((2.0 ** -25, -(2.0 ** -25), 2.0 ** -25 * (1 + 2.0 ** -20), -1e-30)):
        x.flat[i::97] = v
    return x


@pytest.mark.parametrize("dtype", [np.float16, np.float32])
@pytest.mark.parametrize("rows, K, pad", [(1, 1, 0), (33, 7, 0), (31, 8, 1), (40, 9, 0), (32, 63, 1), (65, 65, 0), (33, 127, 3), (64, 130, 1),
                                          (31, 255, 0), (95, 257, 2), (7, 1021, 0),
                                          # from 640 tiles on a wave packs a tile
                                          (20481, 7, 0), (20500, 61, 1), (20511, 100, 1), (10241, 263, 0), (4099, 1281, 1), (1030, 4345, 0)])
def test_pack_reads_rows_of_any_length_at_any_address(oracle, dtype, rows, K, pad):
    rng = np.random.default_rng(rows * 10007 + K)
    x = values(rng, rows, K, dtype)
    wide = torch.from_numpy(np.concatenate([x, np.ones((rows, pad), dtype)], axis=1)).to(DEV)[:, :K]      # row stride K + pad
    assert wide.stride(0) == K + pad
    zp = np.asarray(0.037, dtype)
    zpt = torch.from_numpy(zp.reshape(1)).to(DEV)
    half = x.astype(np.float16)
    centred = oracle.np_center_to_f16(x, zp)
    logical = lambda p, plane=0: lk.logical_from_tiled(p, plane).cpu().numpy().view(np.uint32)
    assert (logical(lk.pack_sign(wide)) == oracle.c_pack_sign(half)).all()
    assert (logical(lk.pack_sign(wide, zero_point=zpt)) == oracle.c_pack_sign(centred)).all()
    nz, sg = oracle.c_pack_ternary(half)
    t = lk.pack_ternary(wide)
    assert (logical(t) == nz).all() and (logical(t, 1) == sg).all()
    # the padding of the tiles is zero: as many bits set in the tiled operand as in the rows
    assert int(lk.row_popcounts(lk.pack_sign(wide)).counts.sum()) == int(np.unpackbits(oracle.c_pack_sign(half).view(np.uint8)).sum())
    words = lk.pack_sign(wide).data.cpu().numpy().view(np.uint8)
    assert int(np.unpackbits(words).sum()) == int(np.unpackbits(oracle.c_pack_sign(half).view(np.uint8)).sum())
