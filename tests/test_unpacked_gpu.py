"""Prepacked weights x activations as they are (bgemm_unpacked_forward) against the pack and the packed entry point, whole numbers: equal."""
import pytest
import torch

import _lib
import lowbit_kernel as lk

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def tern(g, n, k, dtype, special):
    x = torch.randint(-1, 2, (n, k), generator=g, device=DEV).to(dtype)
    if special:           # what the ternary pack calls zero, negative and nonzero
        v = torch.tensor([0.0, -0.0, float("inf"), -float("inf"), float("nan"), 6e-8, -6e-8, 65504.0], device=DEV).to(dtype)
        at = torch.randint(0, 8, (n, k), generator=g, device=DEV)
        x = torch.where(torch.rand(n, k, generator=g, device=DEV) < 0.3, v[at], x)
    return x


def planes_product(w, x, out, scale):
    return lk.bgemm_packed_forward(w, lk.pack_ternary(x), lk.MODE_BWTA, out, scale=scale)[0]


# (rows, columns, K): the two-plane kernels; the signed tile on planes; the same as codes, from where those are taken on: whole tiles and
# ragged ones, an even and an odd number of K-tiles, the last one of a bit, half and whole
@pytest.mark.parametrize("N,M,K", [(64, 1024, 768), (1024, 4352, 512), (2048, 4096, 4096), (1000, 4321, 7937), (1025, 5000, 8000), (2048, 16000, 2047), (2049, 11008, 2177)])
@pytest.mark.parametrize("dtype", [torch.half, torch.float32])
def test_ternary_rows_as_codes_are_the_two_planes(N, M, K, dtype):
    g = torch.Generator(device=DEV).manual_seed(N * 7 + M + K)
    signed = _lib.lib().bgemm_packed_kernel_id(lk.MODE_BWTA, lk.OUT_I32, 1, M, N, K, 8, lk.VARIANT_AUTO) == 8
    assert signed == (N > 64)
    w = lk.pack_sign(torch.randn(M, K, generator=g, device=DEV).half())
    sw, bias, sa = (torch.randn(M, generator=g, device=DEV).half(), torch.randn(M, generator=g, device=DEV).half(), torch.full((1,), 0.37, device=DEV).half())
    for special in (False, True):
        x = tern(g, N, K, dtype, special)
        for out, scale in ((torch.int32, None), (torch.half, None), (None, (sw, sa, bias)), (None, (sw.float(), sa.float(), None))):
            kw = {"scale": scale} if scale else {}
            got = lk.bgemm_packed_weight_forward(w, x, lk.MODE_BWTA, **({"out_dtype": out} if out else {}), **kw)
            want = planes_product(w, x, out or torch.int32, scale)
            assert got.dtype == want.dtype and torch.equal(got, want), (special, out, scale is not None)
    # every product one sign over all of K, rows at odd addresses
    wide = torch.ones(N, K + 3, dtype=dtype, device=DEV)
    wide[::2] = -1
    ones = lk.pack_sign(-torch.ones(M, K, dtype=torch.half, device=DEV))
    assert torch.equal(lk.bgemm_packed_weight_forward(ones, wide[:, 3:], lk.MODE_BWTA), -K * wide[:, :1].int().expand(N, M))


# Which form the activations take, read from the scratch: codes from 4096 tiles x K-tiles on where the signed tile runs, planes elsewhere
@pytest.mark.parametrize("N,M,K,codes", [(2048, 4096, 4096, True), (2048, 4096, 3840, False), (1025, 5000, 8000, True), (2048, 16000, 1792, True), (2048, 512, 65536, False), (128, 4096, 65536, False),
                                         (64, 131072, 2048, False), (129, 8200, 16384, False), (512, 11008, 8192, True)])
def test_the_form_of_ternary_rows(N, M, K, codes):
    L, g = _lib.lib(), torch.Generator(device=DEV).manual_seed(N + M + K)
    signed = L.bgemm_packed_kernel_id(lk.MODE_BWTA, lk.OUT_I32, 1, M, N, K, 8, lk.VARIANT_AUTO) == lk._b.KERNEL_MFMA_128x256T
    assert codes == (signed and -(-N // 128) * -(-M // 256) * -(-K // 256) >= 4096)
    w, x = lk.pack_sign(torch.randn(M, K, generator=g, device=DEV).half()), tern(g, N, K, torch.half, False)
    out, ws = torch.empty(N, M, dtype=torch.int32, device=DEV), torch.empty(L.bgemm_unpacked_workspace_bytes(lk.MODE_BWTA, x.data_ptr(), lk.SRC_F16, K, M, N, K), dtype=torch.uint8, device=DEV)
    _lib.check(L.bgemm_unpacked_forward(lk.MODE_BWTA, w.data.data_ptr(), x.data_ptr(), lk.SRC_F16, K, None, out.data_ptr(), lk.OUT_I32, M, N, K, None, None, None, ws.data_ptr(), ws.numel(), lk._stream()))
    planes = lk.pack_ternary(x)
    words = planes.data.numel()
    first = ws.view(torch.int32)[:words].view_as(planes.data)
    assert torch.equal(first, planes.data) != codes
    assert torch.equal(out, lk.bgemm_packed_forward(w, planes, lk.MODE_BWTA, torch.int32)[0])


def test_sign_rows_and_refusals():
    g = torch.Generator(device=DEV).manual_seed(3)
    w, x = lk.pack_sign(torch.randn(4100, 700, generator=g, device=DEV).half()), torch.randn(1030, 700, generator=g, device=DEV)
    zp = torch.full((1,), 0.1, device=DEV)
    for mode in (lk.MODE_AND, lk.MODE_XOR, lk.MODE_ATTN):
        assert torch.equal(lk.bgemm_packed_weight_forward(w, x, mode, x_zero_point=zp), lk.bgemm_packed_forward(w, lk.pack_sign(x, zero_point=zp), mode)[0])
    with pytest.raises(ValueError):
        lk.bgemm_packed_weight_forward(w, x, lk.MODE_BWTA, x_zero_point=zp)
    L, out, ws = _lib.lib(), torch.empty(1030, 4100, dtype=torch.int32, device=DEV), torch.empty(1 << 20, dtype=torch.uint8, device=DEV)
    call = lambda **k: L.bgemm_unpacked_forward(*{**dict(mode=3, w=w.data.data_ptr(), x=x.data_ptr(), t=lk.SRC_F32, ld=700, zp=None, out=out.data_ptr(), kind=lk.OUT_I32,
                                                         M=4100, N=1030, K=700, sw=None, sa=None, bias=None, ws=ws.data_ptr(), bytes=ws.numel(), stream=None), **k}.values())
    assert call(bytes=1000) == _lib.EWORKSPACE and call(ld=699) == _lib.EINVAL and call(ws=None) == _lib.ENULL and call(kind=lk.OUT_F16_SCALED) == _lib.ENULL
    assert call(x=x.data_ptr() + 1) == _lib.EALIGN and call(mode=9) == _lib.EINVAL and call(zp=zp.data_ptr()) == _lib.EINVAL and call(t=7) == _lib.EINVAL


# rows that one launch packs and multiplies: both ends of N, one and two row tiles a block with and without a rest, K of one chunk, a word and
# a half, one K-tile to sixteen, rows of a wider matrix; and, beside them, rows that launch does not take
@pytest.mark.parametrize("N,M,K,ld", [(5, 64, 256, 256), (8, 33, 264, 272), (16, 100, 2048, 2048), (7, 1000, 1000, 1008), (16, 11008, 2048, 2048), (5, 11008, 4096, 4096), (16, 16384, 4096, 4096),
                                      (32, 500, 2048, 2056), (25, 8225, 512, 520), (17, 77, 8, 8), (31, 16384, 2000, 2000), (9, 300, 8, 16), (10, 4096, 4104, 4104), (32, 2050, 4096, 4096), (16, 700, 4080, 4088),
                                      (16, 200, 2052, 2056), (8, 100, 256, 257), (33, 64, 512, 512), (4, 64, 512, 512)])
@pytest.mark.parametrize("dtype", [torch.half, torch.float32])
def test_few_rows_in_one_launch(N, M, K, ld, dtype):
    g = torch.Generator(device=DEV).manual_seed(N + M + K)
    w = lk.pack_sign(torch.randn(M, K, generator=g, device=DEV).half())
    sw, sa = torch.randn(M, generator=g, device=DEV).to(dtype), torch.full((1,), 0.3, device=DEV).to(dtype)
    special = torch.tensor([0.0, -0.0, float("inf"), -float("inf"), float("nan"), -float("nan"), 6e-8, -6e-8, 0.05], device=DEV).to(dtype)
    for mode in (lk.MODE_AND, lk.MODE_XOR, lk.MODE_ATTN, lk.MODE_BWTA):
        ternary = mode == lk.MODE_BWTA
        x = (torch.randint(-1, 2, (N, ld), generator=g, device=DEV) if ternary else torch.randn(N, ld, generator=g, device=DEV)).to(dtype)
        x = torch.where(torch.rand(N, ld, generator=g, device=DEV) < 0.3, special[torch.randint(0, 9, (N, ld), generator=g, device=DEV)], x)[:, :K]
        f32 = dtype == torch.float32
        one = (5 <= N <= (16 if ternary else 32) and K <= 4096 and K % 8 == 0 and ld * (4 if f32 else 2) % 16 == 0 and M <= 16384
               and not (f32 and (ternary or N * K > 65536)))
        assert one == (_lib.lib().bgemm_unpacked_workspace_bytes(mode, x.data_ptr(), lk.SRC_F32 if f32 else lk.SRC_F16, ld, M, N, K) == 0)
        for zp in (None,) if ternary else (None, special[8:], special[2:3]):
            xp = lk.pack_ternary(x) if ternary else lk.pack_sign(x, zero_point=zp)
            for out, scale in ((torch.int32, None), (torch.half, None), (None, (sw, sa, sw)), (None, (sw, sa, None))):
                got = lk.bgemm_packed_weight_forward(w, x, mode, x_zero_point=zp, scale=scale, **({"out_dtype": out} if out else {}))
                want = lk.bgemm_packed_forward(w, xp, mode, out or torch.int32, scale=scale)[0]
                assert got.dtype == want.dtype and torch.equal(got, want), (mode, None if zp is None else zp.item(), out, scale is not None)


# fp32 rows whose captured call is two launches, on both sides of that rule: rows, K, rows of eight times K, columns
@pytest.mark.parametrize("N,M,K,two", [(9, 4096, 3592, True), (9, 4096, 3584, False), (8, 4096, 4096, False), (16, 4095, 4096, False), (16, 16384, 4096, True), (17, 4100, 2736, True),
                                       (24, 4100, 2728, False), (32, 5000, 2048, False), (25, 5000, 2056, True)])
def test_rows_captured_are_the_rows_of_a_call(N, M, K, two):
    g = torch.Generator(device=DEV).manual_seed(N * M + K)
    L, w, x = _lib.lib(), lk.pack_sign(torch.randn(M, K, generator=g, device=DEV).half()), torch.randn(N, K, generator=g, device=DEV)
    zp, sw, sa = torch.full((1,), 0.1, device=DEV), torch.randn(M, generator=g, device=DEV), torch.full((1,), 0.3, device=DEV)
    args = (lk.MODE_XOR, x.data_ptr(), lk.SRC_F32, K, M, N, K)
    calls = (lambda: lk.bgemm_packed_weight_forward(w, x, lk.MODE_XOR, x_zero_point=zp, scale=(sw, sa, sw)), lambda: lk.bgemm_packed_weight_forward(w, x, lk.MODE_AND))
    bare = torch.empty(N, M, dtype=torch.int32, device=DEV)
    [f() for f in calls]
    assert L.bgemm_unpacked_workspace_bytes(*args) == 0 and L.bgemm_unpacked_workspace_bytes_on(*args, lk._stream()) == 0
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        bytes_on = L.bgemm_unpacked_workspace_bytes_on(*args, lk._stream())
        got = [f() for f in calls]
        # (no scratch: one launch there too)
        _lib.check(L.bgemm_unpacked_forward(lk.MODE_AND, w.data.data_ptr(), x.data_ptr(), lk.SRC_F32, K, None, bare.data_ptr(), lk.OUT_I32, M, N, K, None, None, None, None, 0, lk._stream()))
    assert bool(bytes_on) == two
    for _ in range(3):
        x.copy_(torch.randn(N, K, generator=g, device=DEV))
        want = [f() for f in calls]
        graph.replay()
        assert all(torch.equal(a, b) for a, b in zip([*got, bare], [*want, want[1]]))
