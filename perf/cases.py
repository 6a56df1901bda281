"""What the speed of this library is measured on: the calls its users make, over the range of sizes they make them with.

Every case goes through the public entry points (the ``lowbit_kernel`` functions and the layers of ``bgemm_linear``) the
way a program that uses them does: inference layers keep their packed weights between calls, the drop-in call gets fp16
operands every time, a training step runs forward and backward and gets every gradient.  The sizes are those of the
benchmark configurations (Llama-7B projections, BERT-base layers, the 784-4096-4096-10 MLP, the 8192^3 product), of
the demos and of the ragged shapes in the tests; ``draw`` spreads cases over the ranges between and around them.
"""
import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.getcwd(), "bgemm-cuda_amd"))

import attention_demo  # noqa: E402
import bgemm_linear as bl  # noqa: E402
import lowbit_kernel as lk  # noqa: E402

DEV = "cuda:0"
DTYPES = {"fp32": torch.float32, "fp16": torch.half}
MODES = {"and": lk.MODE_AND, "xor": lk.MODE_XOR, "attn": lk.MODE_ATTN}


def listed():
    return [
        # one token of a decode step through a binary layer of Llama-7B's up projection: latency
        {"name": "decode_linear", "kind": "infer_linear", "n": 1, "k": 4096, "m": 11008, "dtype": "fp16", "bias": False},
        # sixteen decode rows with ternary activations (binary weight x ternary activation), pack included
        {"name": "decode_ternary", "kind": "ternary", "n": 16, "k": 4096, "m": 11008, "scaled": False},
        # the binarised MLP's forward at batch 128: small dependent layers with only bits between them
        {"name": "mlp_chain", "kind": "chain", "n": 128, "k": 784, "h": 4096, "m": 10, "dtype": "fp16"},
        # a BERT-base feed-forward layer in inference, 16 x 512 tokens, fp32 activations as torch hands them over
        {"name": "bert_ffn", "kind": "infer_linear", "n": 8192, "k": 768, "m": 3072, "dtype": "fp32", "bias": True},
        # the reference's own call: fp16 activations and weights, both packed inside the call
        {"name": "dropin_4096", "kind": "dropin", "n": 2048, "k": 4096, "m": 4096, "mode": "xor", "split_k": 1},
        # the same on sizes that are a multiple of nothing (rows start at odd addresses), and-popcount, split K asked for
        {"name": "dropin_ragged", "kind": "dropin", "n": 2053, "k": 4345, "m": 8195, "mode": "and", "split_k": 2},
        # a prompt of 2048 tokens with ternary activations, scaled fp16 output
        {"name": "prefill_ternary", "kind": "ternary", "n": 2048, "k": 4096, "m": 11008, "scaled": True},
        # the large square product on prepacked operands, int32 accumulators out
        {"name": "packed_8192", "kind": "packed", "n": 8192, "k": 8192, "m": 8192, "mode": "xor", "out": "int32"},
        # a BERT-base self-attention block with binary matmuls, batch 16 x 512 tokens, inference
        {"name": "attention_block", "kind": "attention", "batch": 16, "seq": 512, "heads": 12, "size": 64},
        # training both attention products on head-split views, forward and backward
        {"name": "attention_train", "kind": "attention_train", "batch": 4, "seq": 512, "heads": 12, "size": 64},
        # training a binary layer at BERT-base's feed-forward size, fp32 parameters, forward and backward
        {"name": "linear_train", "kind": "train", "layer": "linear", "n": 8192, "k": 768, "m": 3072, "dtype": "fp32", "bias": True},
        # training the learned-scale layer of the MLP demo at its batch and width: many small steps
        {"name": "elastic_train", "kind": "train", "layer": "elastic", "n": 256, "k": 128, "m": 128, "dtype": "fp32", "bias": True},
    ]


def _size(rng, low, high):
    """A size between low and high, even over its logarithm; one in three is left as it falls, the others are a multiple of 64 (of 8 below 64)."""
    v = int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))
    if rng.random() < 1 / 3:
        return max(low, min(high, v))
    step = 64 if v >= 64 else 8 if v >= 8 else 1
    return max(low, min(high, (v + step // 2) // step * step))


def draw(rng):
    kind = rng.choice(["decode", "infer", "ternary", "chain", "dropin", "packed", "attention", "attention_train", "linear_train", "elastic_train"])
    dtype = rng.choice(["fp16", "fp32"])
    if kind == "decode":
        return {"kind": "infer_linear", "n": rng.randint(1, 32), "k": _size(rng, 512, 11008), "m": _size(rng, 512, 22016), "dtype": dtype,
                "bias": rng.random() < 0.5}
    if kind == "infer":
        return {"kind": "infer_linear", "n": _size(rng, 33, 8192), "k": _size(rng, 256, 4096), "m": _size(rng, 256, 4096), "dtype": dtype,
                "bias": rng.random() < 0.5}
    if kind == "ternary":
        return {"kind": "ternary", "n": _size(rng, 1, 2048), "k": _size(rng, 512, 11008), "m": _size(rng, 512, 11008), "scaled": rng.random() < 0.5}
    if kind == "chain":
        return {"kind": "chain", "n": _size(rng, 1, 512), "k": _size(rng, 256, 1024), "h": _size(rng, 256, 4096), "m": rng.randint(2, 1000), "dtype": dtype}
    if kind == "dropin":
        return {"kind": "dropin", "n": _size(rng, 1, 4096), "k": _size(rng, 256, 8192), "m": _size(rng, 256, 11008),
                "mode": rng.choice(sorted(MODES)), "split_k": rng.choice([1, 1, 2, 4])}
    if kind == "packed":
        return {"kind": "packed", "n": _size(rng, 128, 8192), "k": _size(rng, 512, 16384), "m": _size(rng, 512, 8192),
                "mode": rng.choice(sorted(MODES)), "out": rng.choice(["int32", "fp16"])}
    if kind == "attention":
        return {"kind": "attention", "batch": rng.randint(1, 16), "seq": _size(rng, 32, 512), "heads": rng.randint(2, 12), "size": rng.choice([32, 64])}
    if kind == "attention_train":
        return {"kind": "attention_train", "batch": rng.randint(1, 4), "seq": _size(rng, 32, 512), "heads": rng.randint(2, 12), "size": rng.choice([32, 64])}
    if kind == "linear_train":
        k, m = _size(rng, 128, 3072), _size(rng, 128, 3072)
        n = _size(rng, 32, min(8192, 8192 * 768 * 3072 // (k * m)))
        return {"kind": "train", "layer": rng.choice(["linear", "bireal"]), "n": n, "k": k, "m": m, "dtype": dtype, "bias": rng.random() < 0.5}
    return {"kind": "train", "layer": "elastic", "n": _size(rng, 32, 2048), "k": _size(rng, 64, 1024), "m": _size(rng, 64, 1024), "dtype": "fp32", "bias": True}


class _Inputs:
    """Seeded tensors on the GPU."""

    def __init__(self, seed):
        self.g = torch.Generator(device=DEV).manual_seed(int(seed))

    def normal(self, *shape, dtype=torch.float32, scale=1.0):
        return torch.randn(*shape, generator=self.g, device=DEV).mul_(scale).to(dtype)

    def ternary(self, *shape):
        """fp16 activations in {-1, 0, +1}, half of them zero."""
        r = torch.randint(0, 4, shape, generator=self.g, device=DEV)
        return ((r == 0).to(torch.half) - (r == 1).to(torch.half))

    def layer(self, cls, k, m, bias, dtype=torch.float32):
        """A layer with nn.Linear's own initialisation, from this generator."""
        lin = cls(k, m, bias=bias).to(DEV)
        with torch.no_grad():
            lin.weight.uniform_(-1 / math.sqrt(k), 1 / math.sqrt(k), generator=self.g)
            if bias:
                lin.bias.uniform_(-1 / math.sqrt(k), 1 / math.sqrt(k), generator=self.g)
        return lin.to(dtype)


LAYERS = {"linear": bl.BGEMMLinear, "bireal": bl.BGEMMLinear_bireal, "elastic": bl.BGEMMLinear_elastic_signed}


def prepare(case, seed):
    inp, kind = _Inputs(seed), case["kind"]
    if kind == "infer_linear":
        dt = DTYPES[case["dtype"]]
        lin, x = inp.layer(bl.BGEMMLinear, case["k"], case["m"], case["bias"], dt), inp.normal(case["n"], case["k"], dtype=dt)
        with torch.no_grad():
            lin(inp.normal(64, case["k"], dtype=dt))      # the first call sets the layer's scales
            lin(x)                                        # packs the weight, which the layer keeps
        return {"kind": kind, "layer": lin, "x": x}
    if kind == "ternary":
        w = lk.pack_sign(inp.normal(case["m"], case["k"], dtype=torch.half))
        scale = None
        if case["scaled"]:
            scale = (inp.normal(case["m"], scale=0.01).abs_().to(torch.half), torch.full((1,), 0.5, dtype=torch.half, device=DEV), None)
        return {"kind": kind, "w": w, "x": inp.ternary(case["n"], case["k"]), "scale": scale}
    if kind == "chain":
        dt = DTYPES[case["dtype"]]
        chain = bl.BGEMMChain(inp.layer(bl.BGEMMLinear, case["k"], case["h"], True, dt), inp.layer(bl.BGEMMLinear, case["h"], case["h"], True, dt),
                              inp.layer(bl.BGEMMLinear, case["h"], case["m"], True, dt))
        x = inp.normal(case["n"], case["k"], dtype=dt)
        with torch.no_grad():
            chain(inp.normal(64, case["k"], dtype=dt))    # sets the scales
            chain(x)                                      # packs the weights, sizes the bit buffers
        return {"kind": kind, "layer": chain, "x": x}
    if kind == "dropin":
        return {"kind": kind, "x": inp.normal(case["n"], case["k"], dtype=torch.half), "w": inp.normal(case["m"], case["k"], dtype=torch.half),
                "instr": MODES[case["mode"]], "split_k": case["split_k"]}
    if kind == "packed":
        return {"kind": kind, "x": lk.pack_sign(inp.normal(case["n"], case["k"], dtype=torch.half)),
                "w": lk.pack_sign(inp.normal(case["m"], case["k"], dtype=torch.half)), "mode": MODES[case["mode"]],
                "out": torch.int32 if case["out"] == "int32" else torch.half}
    if kind == "attention":
        hidden = case["heads"] * case["size"]
        block = attention_demo.BinarySelfAttention(hidden, case["heads"]).to(DEV)
        for name in ("query", "key", "value", "dense"):
            setattr(block, name, inp.layer(bl.BGEMMLinear, hidden, hidden, True))
        x = inp.normal(case["batch"], case["seq"], hidden)
        with torch.no_grad():
            block(x)
        return {"kind": kind, "layer": block, "x": x}
    if kind == "attention_train":
        B, S, H, d = case["batch"], case["seq"], case["heads"], case["size"]

        def projection():
            return inp.normal(B, S, H * d, dtype=torch.half).requires_grad_(True)

        return {"kind": kind, "q": projection(), "k": projection(), "v": projection(), "heads": H, "size": d,
                "probs": inp.normal(B, H, S, S, dtype=torch.half).requires_grad_(True),
                "g_scores": inp.normal(B, H, S, S, dtype=torch.half, scale=0.01), "g_context": inp.normal(B, H, S, d, dtype=torch.half, scale=0.01)}
    if kind == "train":
        dt = DTYPES[case["dtype"]]
        lin = inp.layer(LAYERS[case["layer"]], case["k"], case["m"], case["bias"], dt)
        x = inp.normal(case["n"], case["k"], dtype=dt).requires_grad_(True)
        out = lin(x).detach()                             # the first step sets the scales
        # the gradient that comes back through a batch norm over these outputs: theirs over the outputs' deviation
        # (fp16: small enough for the scales' gradients, sums over the rows, to stay below the largest half)
        g = inp.normal(*out.shape, scale=0.1 if dt == torch.float32 else 0.001)
        if case["layer"] != "elastic":
            g = g / out.float().std()
        wants = [x, lin.weight, lin.sw, lin.sa] + ([lin.bias] if case["bias"] else [])
        return {"kind": kind, "layer": lin, "x": x, "g": g.to(out.dtype), "wants": wants}
    raise ValueError("unknown kind of case: %r" % kind)


def run(state):
    kind = state["kind"]
    if kind in ("infer_linear", "chain", "attention"):
        with torch.no_grad():
            return state["layer"](state["x"])
    if kind == "ternary":
        return lk.bgemm_packed_weight_forward(state["w"], state["x"], lk.MODE_BWTA, scale=state["scale"])
    if kind == "dropin":
        return lk.bgemm_linear_forward_cuda(state["x"], state["w"], state["split_k"], state["instr"])
    if kind == "packed":
        return lk.bgemm_packed_forward(state["w"], state["x"], state["mode"], state["out"])
    if kind == "attention_train":
        def split(t):
            return t.view(t.shape[0], t.shape[1], state["heads"], state["size"]).permute(0, 2, 1, 3)

        q, k, v, probs = state["q"], state["k"], state["v"], state["probs"]
        scores = bl.bgemm_matmul.apply(split(q), split(k).transpose(-1, -2))
        context = bl.bgemm_attn_matmul.apply(probs, split(v))
        grads = torch.autograd.grad([scores, context], [q, k, v, probs], [state["g_scores"], state["g_context"]])
        return [scores.detach(), context.detach(), *grads]
    out = state["layer"](state["x"])
    return [out.detach(), *torch.autograd.grad(out, state["wants"], state["g"])]


def work(case):
    kind = case["kind"]
    if kind in ("attention", "attention_train"):
        B, S, H, d = case["batch"], case["seq"], case["heads"], case["size"]
        hidden, pairs = H * d, B * H * S * S
        if kind == "attention":
            # the hidden states in and out (fp32), four packed weights, the scores (fp16), which the block returns
            return {"bytes": 8 * B * S * hidden + 4 * hidden * hidden / 8 + 2 * pairs, "flops": 8 * B * S * hidden * hidden + 4 * pairs * d}
        # q, k, v and their gradients, probabilities, scores and their gradients, the context and its gradient, all fp16
        return {"bytes": 2 * (6 * B * S * hidden + 4 * pairs + 2 * B * S * hidden), "flops": 12 * pairs * d}
    n, k, m = case["n"], case["k"], case["m"]
    if kind == "chain":
        h, e = case["h"], 4 if case["dtype"] == "fp32" else 2
        return {"bytes": n * (k + m) * e + (k * h + h * h + h * m) / 8 + 2 * (2 * h + m) * e, "flops": 2 * n * (k * h + h * h + h * m)}
    if kind == "ternary":
        return {"bytes": 2 * n * k + m * k / 8 + n * m * (2 if case["scaled"] else 4), "flops": 2 * n * k * m}
    if kind == "dropin":
        return {"bytes": 2 * (n * k + m * k + n * m), "flops": 2 * n * k * m}
    if kind == "packed":
        return {"bytes": (n * k + m * k) / 8 + n * m * (4 if case["out"] == "int32" else 2), "flops": 2 * n * k * m}
    e = 4 if case["dtype"] == "fp32" else 2
    if kind == "infer_linear":
        return {"bytes": n * k * e + m * k / 8 + n * m * e + 2 * m * e, "flops": 2 * n * k * m}
    # train: activations and weights in, their gradients out, the output out and its gradient in
    return {"bytes": e * (2 * n * k + 2 * m * k + 2 * n * m + 4 * m), "flops": 6 * n * k * m}


def tolerance(case):
    kind = case["kind"]
    if kind == "train" and case["layer"] == "elastic":
        # fp32 products; the output is rounded to fp16 once on the way (against a float64 evaluation: 1.5e-4)
        return {"rel": 6e-4}
    if kind == "train":
        # the gradients' products take fp16 operands and give fp16 results (against float64: 4.3e-4; everything in fp16: 7e-4)
        return {"rel": 2e-3 if case["dtype"] == "fp32" else 3e-3}
    if kind == "attention_train":
        return {"rel": 2e-3}          # the same, in fp16 throughout
    if kind == "attention":
        # fp16 scores; a probability exactly at the level that makes it a 1 may fall either way with the order of the softmax's sum
        return {"rel": 1e-3}
    # integer sums, rounded once (or step by step by a stated rule): every correct implementation gives the same values
    return "exact"
