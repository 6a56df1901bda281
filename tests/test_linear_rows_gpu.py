"""Scaled binary layers on unpacked activations in one launch, against the formula evaluated by torch (integer sums, then every step of
the layer as its own elementwise operation), and attention's context as the next layer's operand."""
import pytest
import torch

pytestmark = pytest.mark.gpu

import _lib
import lowbit_kernel as lk

DEV = "cuda:0"
OUT = {(torch.float32, False): _lib.OUT_F32_SCALED, (torch.half, False): _lib.OUT_F16_SCALED,
       (torch.float32, True): _lib.OUT_BITS_F32, (torch.half, True): _lib.OUT_BITS_F16}


def pm1(t):
    return torch.where(torch.signbit(t), -1.0, 1.0)


def made(N, M, K, layers, dt, bias, seed=0):
    g = torch.Generator(device=DEV).manual_seed(N * 131 + M * 7 + K + seed)
    rnd = lambda *s: torch.randn(*s, generator=g, device=DEV)
    x = rnd(N, K + 3)[:, 2:K + 2].to(dt)                                       # rows at any address
    x[:, ::5] = 0.0
    ls = []
    for _ in range(layers):
        ls.append((rnd(M, K).to(dt), (rnd(1) * 0.3).to(dt), (rnd(M) * 0.01).to(dt), (rnd(1).abs() + 0.1).to(dt), rnd(M).to(dt) if bias else None))
    return x, ls


def formula(x, w, zp, sw, sa, bias):
    """[N, M] in x's type, rounded step by step."""
    acc = pm1(x if zp is None else x - zp) @ pm1(w).T                          # exact: integers below 2^24 in fp32
    y = acc.half().to(x.dtype) * sw * sa
    return y if bias is None else y + bias


def packed(ls):
    return [(lk.pack_sign(w), zp, sw, sa, bias) for w, zp, sw, sa, bias in ls]


# tile edges in rows (32), columns (32) and K (256), every launch shape: one and two column tiles a wave, few and many waves, shared row tiles
SHAPES = [0, 1 | 4 << 4, 2 | 2 << 4, 1 | 5 << 4 | 1 << 12, 2 | 3 << 4 | 3 << 12]
SIZES = [(1, 1, 8, 1), (31, 33, 40, 3), (32, 64, 256, 2), (33, 31, 257, 3), (64, 96, 64, 3), (100, 515, 1000, 1), (130, 257, 2048, 1), (65, 1027, 2041, 1),
         (300, 768, 768, 3)]


@pytest.mark.parametrize("N, M, K, layers", SIZES)
@pytest.mark.parametrize("dt", [torch.float32, torch.half])
def test_numbers_residuals_and_bits(N, M, K, layers, dt):
    for bias in (True, False):
        x, ls = made(N, M, K, layers, dt, bias)
        if bias:
            ls[0] = ls[0][:1] + (None,) + ls[0][2:]                            # no zero point
        residual = torch.randn(N, M, device=DEV).to(dt)
        want = [formula(x, *l) for l in ls]
        xp = lk.pack_sign(x.contiguous(), None if ls[0][1] is None else ls[0][1])
        for shape in SHAPES:
            for got, y in zip(lk.linear_rows_forward(x, packed(ls), shape=shape), want):
                assert torch.equal(got, y)
            for got, y in zip(lk.linear_rows_forward(x, packed(ls), residual=residual, shape=shape), want):
                assert torch.equal(got, y + residual)
            assert torch.equal(lk.linear_rows_forward(xp, packed(ls[:1]), residual=residual, shape=shape)[0], want[0] + residual)
            if lk.linear_rows_supported(N, M, K, layers, OUT[dt, True]):
                for got, y in zip(lk.linear_rows_forward(x, packed(ls), bits=True, shape=shape), want):
                    bits = lk.logical_from_tiled(got)
                    expected = lk.logical_from_tiled(lk.pack_sign(y))
                    assert torch.equal(bits, expected)
                into = [lk.zeros_packed(N, M, 1, DEV) for _ in ls]             # of ones: the padding of the columns is written, too
                for p in into:
                    p.data.fill_(-1)
                for got, y in zip(lk.linear_rows_forward(x, packed(ls), bits=True, shape=shape, bits_out=into), want):
                    whole = N // 32 * -(-M // 256) * 256
                    assert torch.equal(got.data[:, :whole], lk.pack_sign(y).data[:, :whole])


@pytest.mark.parametrize("dt", [torch.float32, torch.half])
@pytest.mark.parametrize("N, M", [(1, 33), (33, 64), (40, 97), (95, 31)])
def test_nothing_is_written_past_the_output(N, M, dt):
    """The last row tile and column tile end where the output does; the next layer's zero point is taken off the bits."""
    K = 100
    x, ls = made(N, M, K, 1, dt, True)
    x = x.contiguous()
    room = torch.full(((N + 64) * M + 2048,), 7.0, dtype=dt, device=DEV)       # a further row tile would fit
    out = room[1024:1024 + N * M]
    (w, zp, sw, sa, bias), = packed(ls)
    layer = (_lib.RowsLayer * 1)()
    layer[0].W_tiled, layer[0].zero_point, layer[0].sw, layer[0].sa = w.data.data_ptr(), zp.data_ptr(), sw.data_ptr(), sa.data_ptr()
    layer[0].bias, layer[0].out = bias.data_ptr(), out.data_ptr()
    src = _lib.SRC_F32 if dt == torch.float32 else _lib.SRC_F16
    _lib.check(_lib.lib().bgemm_linear_rows_forward(x.data_ptr(), src, K, N, M, K, 1, layer, OUT[dt, False], None, 0, None))
    assert torch.equal(out.view(N, M), formula(x, *ls[0]))
    assert bool((room[:1024] == 7).all()) and bool((room[1024 + N * M:] == 7).all())
    bits, following = lk.zeros_packed(N, M), torch.full((1,), 0.25, dtype=dt, device=DEV)
    layer[0].out, layer[0].next_zero_point = bits.data.data_ptr(), following.data_ptr()
    _lib.check(_lib.lib().bgemm_linear_rows_forward(x.data_ptr(), src, K, N, M, K, 1, layer, OUT[dt, True], None, 0, None))
    assert torch.equal(lk.logical_from_tiled(bits), lk.logical_from_tiled(lk.pack_sign(formula(x, *ls[0]), following)))


@pytest.mark.parametrize("dt", [torch.float32, torch.half])
@pytest.mark.parametrize("scale", [0.0, -0.0, -1.0, float("inf"), 2.0 ** -24, 60000.0])
def test_scales_that_are_not_ordinary(scale, dt):
    x, ls = made(40, 70, 96, 1, dt, False)
    w, zp, sw, sa, _ = ls[0]
    sw[::3] = scale
    sw[1::7] = float("nan")
    got, want = lk.linear_rows_forward(x, packed([(w, zp, sw, sa, None)]))[0], formula(x, w, zp, sw, sa, None)
    assert torch.equal(got.isnan(), want.isnan())
    ints = {torch.float32: torch.int32, torch.half: torch.int16}[dt]
    assert torch.equal(got.view(ints)[~want.isnan()], want.view(ints)[~want.isnan()])      # signs of zeros, too


@pytest.mark.parametrize("dt", [torch.float32, torch.half])
@pytest.mark.parametrize("scale", [0.0, -0.0, -1.0, float("inf"), -float("inf"), 2.0 ** -24, 60000.0])
def test_bits_of_scales_that_are_not_ordinary(scale, dt):
    """Wherever the centred number is one (the sign of a NaN is not defined)."""
    for shape in (0, 1 | 5 << 4 | 1 << 12, 2 | 2 << 4 | 2 << 12):
        x, ls = made(40, 70, 96, 1, dt, True)
        w, zp, sw, sa, bias = ls[0]
        sw[::3] = scale
        sw[1::7] = float("nan")
        bias[::5] = -scale
        following = torch.full((1,), 0.25, dtype=dt, device=DEV)
        got, = lk.linear_rows_forward(x, packed(ls), bits=True, next_zero_point=following, shape=shape)
        words = lk.logical_from_tiled(got)
        bits = (words[:, torch.arange(70, device=DEV) // 32] >> (31 - torch.arange(70, device=DEV) % 32)) & 1
        want = formula(x, *ls[0]) - following
        assert torch.equal(bits[~want.isnan()] != 0, torch.signbit(want[~want.isnan()])) and bool((~want.isnan()).any())


@pytest.mark.parametrize("dt", [torch.float32, torch.half])
@pytest.mark.parametrize("B, S, H, d", [(1, 1, 1, 32), (2, 33, 5, 64), (3, 70, 3, 96), (1, 130, 7, 128), (2, 64, 8, 32)])
def test_context_as_bits(B, S, H, d, dt):
    g = torch.Generator(device=DEV).manual_seed(S + d)
    q, k, v = (lk.pack_sign(torch.randn(B * S, H * d, generator=g, device=DEV)) for _ in range(3))
    scores, context = lk.attention_forward(q, k, v, B, H, dt)
    for zp in (0.0, 2.0, -1.0):
        zp = torch.full((1,), zp, dtype=dt, device=DEV)
        scores2, bits = lk.attention_forward(q, k, v, B, H, dt, zp)
        assert torch.equal(scores, scores2)
        want = lk.pack_sign(context.view(B * S, H * d), zp)
        assert torch.equal(lk.logical_from_tiled(bits), lk.logical_from_tiled(want))
        real = (B * S) // 32 * bits.words // -(-B * S // 32)                   # whole row tiles, their padding of columns included
        assert torch.equal(bits.data[:, :real], want.data[:, :real])


# column tiles and waves (32, 16 x 32, 1024), rows (32), K-tiles (256), one column; a row far from zero against its deviation, equal outputs
@pytest.mark.parametrize("N, M, K", [(1, 1, 1), (31, 33, 40), (33, 512, 256), (64, 513, 257), (65, 768, 768), (100, 1001, 1000), (32, 1024, 1024)])
def test_layer_norm_of_rows_and_residual(N, M, K):
    for offset, bias, gamma, beta in ((0.0, True, True, True), (50.0, False, True, False), (0.0, True, False, True)):
        x, ls = made(N, M, max(K, 8), 1, torch.float32, bias, seed=int(offset))
        x, ls[0] = x[:, :K], (ls[0][0][:, :K].contiguous(),) + ls[0][1:]
        residual = torch.randn(N, M, device=DEV) + offset
        g, b = (torch.randn(M, device=DEV) if wanted else None for wanted in (gamma, beta))
        w, zp, sw, sa, bi = ls[0]
        if offset:
            sw, residual[N // 2] = sw * 0.0, offset                            # a row of equal values
        xp = lk.pack_sign(x.contiguous(), zp)
        got, = lk.linear_rows_forward(xp, [(lk.pack_sign(w), zp, sw, sa, bi)], residual=residual, norm=(g, b, 1e-12))
        z = (formula(x, w, zp, sw, sa, bi) + residual).double()
        mean, var = z.mean(1, keepdim=True), z.var(1, unbiased=False, keepdim=True)
        gd, bd = 1.0 if g is None else g.double(), 0.0 if b is None else b.double()
        want = (z - mean) / (var + 1e-12).sqrt() * gd + bd
        # a mean of at most 64 fp32 roundings of 2^-24 on values of that size, over a deviation whose relative error is no larger
        far = z.abs().amax(1, keepdim=True)
        bound = 64 * 2.0 ** -24 * ((1 + far / (var + 1e-12).sqrt()) * (torch.ones_like(z) * gd).abs() + (want - bd).abs() + abs(bd))
        assert bool(((got.double() - want).abs() <= bound).all())


@pytest.mark.parametrize("N, M", [(1, 33), (33, 64), (40, 97), (95, 31), (65, 513), (31, 1001)])
def test_the_layer_norm_writes_nothing_past_the_output_and_keeps_rows_apart(N, M):
    """The last row tile and column tile end where the output does; infinities and NaNs of one row stay in it."""
    K = 100
    x, ls = made(N, M, K, 1, torch.float32, True)
    (w, zp, sw, sa, bias), = packed(ls)
    xp, residual = lk.pack_sign(x.contiguous(), zp), torch.randn(N, M, device=DEV)
    lost = torch.arange(N, device=DEV) % 4 == 1
    for row, value in zip(lost.nonzero()[:, 0].tolist(), [float("inf"), -float("inf"), float("nan")] * N):
        residual[row, row % M] = value
    gamma, beta = torch.randn(M, device=DEV), torch.randn(M, device=DEV)
    room = torch.full(((N + 64) * M + 2048,), 7.0, device=DEV)                 # a further row tile would fit
    out = room[1024:1024 + N * M]
    layer = (_lib.RowsLayer * 1)()
    layer[0].W_tiled, layer[0].sw, layer[0].sa, layer[0].bias, layer[0].out = w.data.data_ptr(), sw.data_ptr(), sa.data_ptr(), bias.data_ptr(), out.data_ptr()
    _lib.check(_lib.lib().bgemm_linear_rows_norm_forward(xp.data.data_ptr(), N, M, K, layer, residual.data_ptr(), gamma.data_ptr(), beta.data_ptr(), 1e-12, None))
    assert bool((room[:1024] == 7).all()) and bool((room[1024 + N * M:] == 7).all())
    got = out.view(N, M)
    assert bool(got[lost].isnan().all())                                       # a mean that is not finite leaves nothing of its row
    z = (formula(x, *ls[0]) + residual)[~lost].double()
    want = torch.nn.functional.layer_norm(z, (M,), gamma.double(), beta.double(), 1e-12)
    # (as above: at most 64 roundings of 2^-24 on values of the mean's size and deviation)
    far, dev = z.abs().amax(1, keepdim=True), (z.var(1, unbiased=False, keepdim=True) + 1e-12).sqrt()
    bound = 64 * 2.0 ** -24 * ((1 + far / dev) * gamma.double().abs() + (want - beta.double()).abs() + beta.double().abs())
    assert bool(((got[~lost].double() - want).abs() <= bound).all())
