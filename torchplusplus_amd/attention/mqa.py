"""Multi-query attention (reference: torchpp/attention/mqa.py:9-93): Hq query
heads share one K/V head. Attention runs on the single KV head directly
(no broadcast copy). Fix: K is rotated from K (the reference rotates Q into
K, mqa.py:81)."""
from __future__ import annotations

import torch
import torch.nn as nn

from torchplusplus_amd._native import ext as _ext
from torchplusplus_amd.attention._common import norm_rope_qk
from torchplusplus_amd.attention.flash import flash_attn_func
from torchplusplus_amd.dlops.linear import linear

_C = _ext()


class MultiQueryAttention(nn.Module):
    def __init__(self, num_q_heads: int, embed_dim: int, qk_norm: bool = True,
                 dtype: torch.dtype = torch.float16, device=None):
        super().__init__()
        self.embed_dim = embed_dim
        self.num_q_head = num_q_heads
        self.head_dim = embed_dim // num_q_heads
        kw = dict(dtype=dtype, device=device, bias=False)
        self.Wq = nn.Linear(embed_dim, embed_dim, **kw)
        self.Wk = nn.Linear(embed_dim, self.head_dim, **kw)
        self.Wv = nn.Linear(embed_dim, self.head_dim, **kw)
        self.out_projection = nn.Linear(embed_dim, embed_dim, **kw)
        self.qk_norm = qk_norm
        self.q_norm = nn.RMSNorm(self.head_dim, eps=1e-6, dtype=dtype, device=device)
        self.k_norm = nn.RMSNorm(self.head_dim, eps=1e-6, dtype=dtype, device=device)

    def forward(self, x, cos, sin):
        bsz, seq, _ = x.shape
        q, k, v = _C.linear3(x, self.Wq.weight, self.Wk.weight, self.Wv.weight)
        q = q.view(bsz, seq, self.num_q_head, self.head_dim)
        k, v = k.view(bsz, seq, 1, self.head_dim), v.view(bsz, seq, 1, self.head_dim)
        norms = (self.q_norm, self.k_norm) if self.qk_norm else (None, None)
        q, k = norm_rope_qk(q, k, *norms, cos, sin)
        o = flash_attn_func(q, k, v, causal=True)
        return linear(o.reshape(bsz, seq, self.embed_dim), self.out_projection.weight)
