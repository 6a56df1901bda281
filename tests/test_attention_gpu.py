"""The one-launch binary self-attention against dense torch: scores bit for bit, the context wherever float64 leaves no doubt about a
probability's side of the level; the block that uses it against its own general path."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu

import _lib
import attention_demo
import bgemm_linear as bl
import lowbit_kernel as lk

DEV = "cuda:0"


def pm1(t):
    return torch.where(torch.signbit(t), -1.0, 1.0)


@pytest.mark.parametrize("dtype", [torch.float32, torch.half])
@pytest.mark.parametrize("B, S, H, d", [(1, 1, 1, 32), (3, 7, 2, 64), (1, 32, 3, 96), (2, 33, 5, 128), (2, 63, 3, 32), (1, 64, 9, 64), (1, 65, 2, 64),
                                        (2, 127, 4, 96), (5, 129, 7, 64), (4, 512, 12, 64), (1, 1000, 3, 128), (1, 2048, 2, 64), (1, 4096, 1, 32),
                                        (16, 130, 12, 32)])
def test_attention_in_one_launch(B, S, H, d, dtype):
    g = torch.Generator(device=DEV).manual_seed(S * 131 + d)
    q, k, v = (torch.randn(B * S, H * d, generator=g, device=DEV) for _ in range(3))
    q = q + 0.4 * k                                     # scores away from their mean as well
    scores, context = lk.attention_forward(lk.pack_sign(q), lk.pack_sign(k), lk.pack_sign(v), B, H, dtype)
    assert scores.shape == (B, H, S, S) and context.shape == (B, S, H * d) and context.dtype == dtype
    split = lambda t: pm1(t).view(B, S, H, d).permute(0, 2, 1, 3)
    want = (split(q) @ split(k).transpose(-1, -2).contiguous()).half() / math.sqrt(d)
    assert torch.equal(scores, want)
    p = torch.softmax(want.double(), -1)
    # fp32 exponentials, a sum of S of them and a division: within 1e-6 of p (measured bits agree far closer)
    over = [(p * (1 + e)).half().float() >= torch.tensor(1.0 / S) for e in (-1e-6, 1e-6)]
    clear = (over[0] == over[1]).all(-1)
    ref = (over[0].float() @ split(v).contiguous()).half()
    got = context.view(B, S, H, d).permute(0, 2, 1, 3)
    assert clear.float().mean() > 0.97
    assert torch.equal(got[clear], ref.to(dtype)[clear])


@pytest.mark.parametrize("hidden, heads, B, S, dtype", [(768, 12, 2, 128, torch.float32), (96, 3, 3, 77, torch.half), (640, 5, 1, 200, torch.float32)])
def test_block_fused_equals_its_general_path(hidden, heads, B, S, dtype, monkeypatch):
    torch.manual_seed(S)
    block = attention_demo.BinarySelfAttention(hidden, heads).to(DEV).to(dtype)
    x = torch.randn(B, S, hidden, device=DEV, dtype=dtype)
    calls = []
    inner = lk.attention_forward
    monkeypatch.setattr(lk, "attention_forward", lambda *a: calls.append(1) or inner(*a))
    with torch.no_grad():
        block(x)                                        # sets the scales
        assert not calls
        out, scores = block(x)
        assert len(calls) == 1
        seen = []
        handle = block.key.register_forward_hook(lambda m, i, o: seen.append(o.shape))       # a listener gets its call
        out2, scores2 = block(x)
        handle.remove()
        assert len(calls) == 1 and seen == [(B, S, hidden)]
        masked, _ = block(x, torch.zeros(B, 1, 1, S, device=DEV))
    assert out.dtype == out2.dtype and torch.equal(scores, scores2)
    # a probability on the level may fall either way with the order of the softmax's sum: few rows of the context, if any
    same = (out == out2).all(-1).float().mean()
    assert same > 0.98 and torch.equal(masked, out2), float(same)


@pytest.mark.parametrize("other", ["elastic", "bireal", "nn.Linear", "nn.Sequential", "heads", "mode"])
def test_block_with_other_parts_takes_its_general_path(other, monkeypatch):
    """Any module may stand for a projection, and whoever replaces the split into heads or watches torch's functions is asked."""
    torch.manual_seed(2)
    block = attention_demo.BinarySelfAttention(64, 2).to(DEV)
    made = {"elastic": lambda: bl.BGEMMLinear_elastic_signed(64, 64), "bireal": lambda: bl.BGEMMLinear_bireal(64, 64, bias=True),
            "nn.Linear": lambda: torch.nn.Linear(64, 64), "nn.Sequential": lambda: torch.nn.Sequential(bl.BGEMMLinear(64, 64))}
    if other in made:
        block.key = made[other]().to(DEV)
    x, calls = torch.randn(3, 10, 64, device=DEV), []
    with torch.no_grad():
        block(x)                                        # sets the scales
        if other == "heads":
            split = block.transpose_for_scores
            block.transpose_for_scores = lambda t: calls.append("heads") or split(t.flip(-1))
        if other == "mode":
            class Functions(torch.overrides.TorchFunctionMode):
                def __torch_function__(self, func, types, args=(), kwargs=None):
                    calls.append(getattr(func, "__name__", ""))
                    return func(*args, **(kwargs or {}))

            with Functions():
                out, scores = block(x)
            assert "softmax" in calls
        else:
            out, scores = block(x)
        monkeypatch.setattr(attention_demo.BinarySelfAttention, "_fusable", lambda self, t: False)
        want, want_scores = block(x)
    assert torch.equal(out, want) and torch.equal(scores, want_scores)
    assert other != "heads" or calls.count("heads") == 6


@pytest.mark.parametrize("change", ["none", "plain", "hook", "half", "other", "tensor"])
def test_block_of_many_rows_with_its_layer_norm_in_the_last_projection(change, monkeypatch):
    """From a thousand rows on the block's layer norm is part of its last launch, unless it is another module or somebody listens to it."""
    torch.manual_seed(5)
    block = attention_demo.BinarySelfAttention(96, 3).to(DEV)
    with torch.no_grad():
        block.LayerNorm.weight.uniform_(0.5, 1.5)
        block.LayerNorm.bias.normal_()
    x, seen = torch.randn(9, 130, 96, device=DEV), []
    if change == "plain":
        block.LayerNorm = torch.nn.LayerNorm(96, elementwise_affine=False)
    if change == "hook":
        block.LayerNorm.register_forward_hook(lambda m, i, o: seen.append(1))
    if change == "half":
        block, x = block.half(), x.half()
    if change == "other":
        block.LayerNorm = torch.nn.Identity()
    if change == "tensor":                                                     # as some reparametrisations leave it: no parameter, an attribute
        weight = block.LayerNorm.weight.detach().clone()
        del block.LayerNorm.weight
        block.LayerNorm.weight = weight
    with torch.no_grad():
        block(x)
        del seen[:]
        calls = []
        monkeypatch.setattr(torch.nn.functional, "layer_norm", lambda *a, f=torch.nn.functional.layer_norm: calls.append(1) or f(*a))
        out, scores = block(x)
        assert len(calls) == (1 if change in ("hook", "half", "tensor") else 0) and len(seen) == (change == "hook")
        monkeypatch.setattr(lk, "linear_rows_norm_supported", lambda *a: 1)
        want, want_scores = block(x)
    assert torch.equal(scores, want_scores) and out.dtype == want.dtype
    # two orders of a sum of 96 values of about one: some 2^-24 each
    torch.testing.assert_close(out, want, rtol=0, atol=0 if change in ("hook", "half", "other", "tensor") else 2e-5)


@pytest.mark.parametrize("native", [True, False])
@pytest.mark.parametrize("width", [128, 512])
def test_block_refuses_projections_of_another_width(width, native, monkeypatch):
    """Parameters of another width than heads x head size, the modules' own sizes left as they were: refused as by the general path, also where
    the width splits into heads that the kernel takes."""
    if not native:
        monkeypatch.setattr(_lib, "_native", None)
        monkeypatch.setattr(_lib, "_native_looked_for", True)
    block = attention_demo.BinarySelfAttention(256, 4).to(DEV)
    x = torch.randn(2, 40, 256, device=DEV)
    with torch.no_grad():
        block(x)
        for layer in (block.query, block.key, block.value):
            for name, t in (("weight", torch.randn(width, 256)), ("sw", torch.rand(width)), ("bias", torch.randn(width))):
                setattr(layer, name, torch.nn.Parameter(t.to(DEV)))
        for _ in range(2):
            with pytest.raises(RuntimeError, match="invalid for input of size"):
                block(x)
