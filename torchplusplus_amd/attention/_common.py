"""Shared pieces of the non-GQA attention modules."""
from __future__ import annotations

import torch

from torchplusplus_amd._native import ext as _ext

_C = _ext()


def head_rmsnorm(x: torch.Tensor, norm) -> torch.Tensor:
    """nn.RMSNorm over head_dim on [B, S, H, D] through the fused kernel."""
    if norm is None:
        return x
    eps = norm.eps if norm.eps is not None else 1e-6
    return _C.rmsnormFused(x, norm.weight, eps)


def rope_bshd(x: torch.Tensor, cos: torch.Tensor, sin: torch.Tensor) -> torch.Tensor:
    """rope_apply on a [B, S, H, D] tensor: the kernel works on [B, H, S, D]."""
    xt = x.transpose(1, 2).contiguous()
    _C.rope_apply_(xt, cos, sin)
    return xt.transpose(1, 2)


def norm_rope_qk(q: torch.Tensor, k: torch.Tensor, q_norm, k_norm, cos: torch.Tensor,
                 sin: torch.Tensor):
    """Per-head norm (a module or None) and rotation of freshly projected q and
    k, [B, S, H, D]: one in-place launch where the kernel takes them (head_dim
    64, 128 or 256, 16-byte alignment), the separate norm and rotation
    otherwise."""
    norms = (q_norm, k_norm)
    if all(n is None or n.weight is not None for n in norms):
        weights = [None if n is None else n.weight for n in norms]
        eps = [1e-6 if n is None or n.eps is None else n.eps for n in norms]
        if _C.qk_norm_rope_(q, k, *weights, *eps, cos, sin):
            return q, k
    q, k = head_rmsnorm(q, q_norm), head_rmsnorm(k, k_norm)
    return rope_bshd(q, cos, sin), rope_bshd(k, cos, sin)
