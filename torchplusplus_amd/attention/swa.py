"""Sliding-window attention (reference: torchpp/attention/swa.py:8-93):
causal attention limited to the last `window_size` keys,
flash_attn_func(..., window_size=(window_size - 1, 0)) (swa.py:85-89).
Same fixes as MultiHeadAttention (module init, head_dim QK-norm)."""
from __future__ import annotations

import torch

from torchplusplus_amd._native import ext as _ext
from torchplusplus_amd.attention._common import norm_rope_qk
from torchplusplus_amd.attention.flash import flash_attn_func
from torchplusplus_amd.attention.mha import MultiHeadAttention
from torchplusplus_amd.dlops.linear import linear

_C = _ext()


class SlidingWindowAttention(MultiHeadAttention):
    def __init__(self, window_size: int, embed_dim: int, n_heads: int, qknorm: bool = True,
                 dtype: torch.dtype = torch.float16, device=None):
        super().__init__(embed_dim, n_heads, qknorm, dtype, device)
        self.window_size = window_size

    def forward(self, x: torch.Tensor, cos, sin):
        bsz, seq, _ = x.shape
        q, k, v = (self._heads(t, bsz, seq) for t in
                   _C.linear3(x, self.Wq.weight, self.Wk.weight, self.Wv.weight))
        q, k = norm_rope_qk(q, k, self.q_norm, self.k_norm, cos, sin)
        o = flash_attn_func(q, k, v, causal=True, window_size=(self.window_size - 1, 0))
        return linear(o.reshape(bsz, seq, self.embed_dim), self.out_projection.weight,
                      self.out_projection.bias)
