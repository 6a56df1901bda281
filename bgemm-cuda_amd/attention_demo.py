"""A binarised BERT self-attention block on the binary layers and the batched attention pair.

The reference vendors a quantised BERT whose self-attention still multiplies with ``torch.matmul``
(tests/python/bert/bert.py:222-262: Q K^T at :245-246, probabilities x V at :259); its README lists
wiring the binary kernels in as open work.  This block is that wiring, forward and backward:
the four projections are ``BGEMMLinear`` layers, the scores are ``bgemm_matmul(q, k^T)`` on the
sign bits of Q and K, and the context is ``bgemm_attn_matmul(a, v)`` with the probabilities binarised
to {0,1} (1 where a probability is at least the uniform level 1/S, its row's mean) and V to {-1,+1}.  ``kernels=False``
evaluates the same block with dense torch matmuls on the de-binarised tensors, which is what the
tests compare against, bit for bit.

    python attention_demo.py            # times one BERT-base block, kernels against dense torch
"""
import math
import time

import torch
import torch.nn as nn

import _lib
import lowbit_kernel
from bgemm_linear import BGEMMLinear, GraphedInference, bgemm_attn_matmul, bgemm_matmul, fused_bits


def _pm1(t):
    """{-1,+1} by the sign bit (what the kernels read: -0.0 counts as negative)."""
    return torch.where(torch.signbit(t), -1.0, 1.0).to(t.dtype)


def _unheard(layer):
    """Whether a module is a plain BGEMMLinear whose call nothing listens to."""
    return (type(layer) is BGEMMLinear and layer.fuse_inference and not layer._forward_hooks and not layer._forward_pre_hooks
            and "forward" not in layer.__dict__ and not nn.modules.module._has_any_global_hook())


class BinarySelfAttention(nn.Module):
    """hidden -> heads x head_size attention with binary operands everywhere a matmul happens
    (bert.py:177-262 with both matmuls on the binary kernels)."""

    def __init__(self, hidden_size=768, num_attention_heads=12, kernels=True):
        super().__init__()
        if hidden_size % num_attention_heads:
            raise ValueError("hidden size %d is not a multiple of %d heads" % (hidden_size, num_attention_heads))
        self.num_attention_heads = num_attention_heads
        self.attention_head_size = hidden_size // num_attention_heads
        self.kernels = kernels
        self.query = BGEMMLinear(hidden_size, hidden_size, bias=True)
        self.key = BGEMMLinear(hidden_size, hidden_size, bias=True)
        self.value = BGEMMLinear(hidden_size, hidden_size, bias=True)
        self.dense = BGEMMLinear(hidden_size, hidden_size, bias=True)
        self.LayerNorm = nn.LayerNorm(hidden_size, eps=1e-12)

    def transpose_for_scores(self, x):
        return x.view(*x.shape[:-1], self.num_attention_heads, self.attention_head_size).permute(0, 2, 1, 3)

    def _fusable(self, x):
        """Whether bits may stand for the projections' outputs: three plain layers that split into these heads, nothing that looks in between."""
        if (torch.is_grad_enabled() or torch.is_autocast_enabled() or lowbit_kernel.watched()
                or getattr(self.transpose_for_scores, "__func__", None) is not BinarySelfAttention.transpose_for_scores):
            return False
        layers = [self._modules.get(name) for name in ("query", "key", "value")]
        hidden = self.num_attention_heads * self.attention_head_size
        if not all(_unheard(l) and l.out_features == hidden for l in layers):
            return False
        native = _lib.native_or_none()
        if native is not None and native.block_ready([l.__dict__ for l in layers], x, self.num_attention_heads, self.attention_head_size):
            return True
        return (x.dim() == 3 and x.numel() > 0 and all(l.weight.shape[0] == hidden and l._bits_fusable(x) for l in layers)
                and lowbit_kernel.attention_supported(x.shape[0], x.shape[1], self.num_attention_heads, self.attention_head_size))

    def _dense_fusable(self, x, rows, hidden):
        """Whether the last projection may read the context's bits and add the residual: a plain layer of this block's size."""
        layer = self._modules.get("dense")
        return (_unheard(layer) and layer.out_features == hidden and layer.weight.shape == (hidden, hidden) and x.shape[-1] == hidden and layer._bits_fusable(x)
                and lowbit_kernel.linear_rows_supported(rows, hidden, hidden, 1, lowbit_kernel.OUT_F32_SCALED if x.dtype == torch.float32
                                                        else lowbit_kernel.OUT_F16_SCALED))

    def _norm(self, x, rows, hidden):
        """The layer norm as ``linear_rows_forward`` takes it; None where it is not a plain fp32 one over these features whose call nothing listens to."""
        norm = self._modules.get("LayerNorm")
        if (type(norm) is not nn.LayerNorm or norm.normalized_shape != (hidden,) or norm._forward_hooks or norm._forward_pre_hooks
                or "forward" in norm.__dict__ or x.dtype != torch.float32 or "weight" not in norm._parameters or "bias" not in norm._parameters):
            return None          # (one that is not registered, not even as None, has been replaced by something else)
        parameters = norm._parameters["weight"], norm._parameters["bias"]
        for t in parameters:
            if t is not None and (type(t) is not nn.Parameter or t.dtype != torch.float32 or t.device != x.device or t.shape != (hidden,) or not t.is_contiguous()):
                return None
        return (*parameters, norm.eps) if lowbit_kernel.linear_rows_norm_supported(rows, hidden, hidden) == 2 else None

    def forward(self, hidden_states, attention_mask=None):
        if self.kernels and attention_mask is None and self._fusable(hidden_states):
            # nothing but the projections' signs is read: they leave their GEMMs as bits, and one kernel does the rest
            bits = fused_bits([self.query, self.key, self.value], hidden_states)
            batch, seq, _ = hidden_states.shape
            rows, hidden = batch * seq, bits[0].K
            if self._dense_fusable(hidden_states, rows, hidden):
                # of the context, too, the last projection reads its signs only, and it adds the residual as it stores
                zero_point = self.dense.zpa
                if zero_point.dtype != hidden_states.dtype:
                    zero_point = zero_point.detach().to(hidden_states.dtype)
                scores, context = lowbit_kernel.attention_forward(*bits, batch, self.num_attention_heads, hidden_states.dtype, zero_point)
                native, norm = _lib.native_or_none(), self._norm(hidden_states, rows, hidden)
                out = None if native is None else native.rows_residual(self.dense.__dict__, context.data, hidden_states, norm)
                if out is None:
                    residual = hidden_states.reshape(rows, hidden).contiguous()
                    out = lowbit_kernel.linear_rows_forward(context, [self.dense._rows_layer(hidden_states.dtype)], residual=residual, norm=norm)[0].view(batch, seq, hidden)
                return out if norm is not None else self.LayerNorm(out), scores
            scores, context = lowbit_kernel.attention_forward(*bits, batch, self.num_attention_heads, hidden_states.dtype)
            return self.LayerNorm(self.dense(context) + hidden_states), scores
        q = self.transpose_for_scores(self.query(hidden_states))
        k = self.transpose_for_scores(self.key(hidden_states))
        v = self.transpose_for_scores(self.value(hidden_states))
        if self.kernels:
            scores = bgemm_matmul.apply(q, k.transpose(-1, -2))
        else:
            scores = torch.matmul(_pm1(q.half()).float(), _pm1(k.half()).float().transpose(-1, -2)).half()
        # the scores are small integers held in fp16 (the kernel's output type); the elementwise work between the
        # two matmuls stays in fp16 storage, which is a third of the memory traffic of an fp32 round trip
        scores = scores / math.sqrt(self.attention_head_size)
        if attention_mask is not None:
            scores = scores + attention_mask.to(scores.dtype)
        probs = torch.softmax(scores, dim=-1)
        centred = probs - 1.0 / probs.shape[-1]                     # {0,1}: at least the uniform level 1/S
        if self.kernels:
            context = bgemm_attn_matmul.apply(centred, v)
        else:
            context = torch.matmul((~torch.signbit(centred.half())).float(), _pm1(v.half()).float()).half()
        context = context.permute(0, 2, 1, 3).reshape(*hidden_states.shape[:-1], -1).to(hidden_states.dtype)
        out = self.dense(context)
        return self.LayerNorm(out + hidden_states), scores


def main():
    dev = torch.device("cuda:0")
    torch.manual_seed(0)
    block = BinarySelfAttention().to(dev)
    x = torch.randn(16, 512, 768, device=dev)
    with torch.no_grad():
        block(x)                                     # initialises the layers' scales
        for kernels in (True, False):
            block.kernels = kernels
            for _ in range(3):
                block(x)
            torch.cuda.synchronize()
            t0 = time.perf_counter()
            for _ in range(20):
                block(x)
            torch.cuda.synchronize()
            print("%-28s %.2f ms per block forward (batch 16, 512 tokens, BERT-base sizes)"
                  % ("binary kernels:" if kernels else "dense torch on +-1 tensors:", (time.perf_counter() - t0) / 20 * 1e3))
        block.kernels = True
        fast = GraphedInference(lambda t: block(t)[0], x)          # the same forward as one captured graph
        for _ in range(3):
            fast(x)
        torch.cuda.synchronize()
        t0 = time.perf_counter()
        for _ in range(20):
            fast(x)
        torch.cuda.synchronize()
        print("%-28s %.2f ms per block forward" % ("binary kernels, one graph:", (time.perf_counter() - t0) / 20 * 1e3))


if __name__ == "__main__":
    main()
