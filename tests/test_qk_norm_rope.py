"""Per-head norm + rotation of Q and K in one in-place launch, against the
oracle's norm and rotation (each rounded to the storage type: atol 2e-2 /
rtol 1e-2, the tolerance of every 16-bit output here)."""
import pytest
import torch

import oracle
from tests.conftest import close

pytestmark = pytest.mark.gpu


def _rand(shape, dtype, seed):
    return torch.randn(*shape, generator=torch.Generator().manual_seed(seed)).to(dtype)


def _want(x, w, eps, cos, sin):
    if w is not None:
        x = oracle.rmsnorm(x, w, eps)
    return oracle.rope(x.transpose(1, 2).contiguous(), cos, sin).transpose(1, 2)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("tables", [torch.float16, torch.float32, torch.bfloat16])
@pytest.mark.parametrize("b,s,hq,hk,d,norms", [(1, 1, 1, 1, 64, "qk"), (2, 17, 4, 4, 64, "qk"),
                                               (3, 70, 6, 1, 128, ""), (1, 33, 4, 2, 256, "k"),
                                               (2, 1000, 16, 16, 64, "q"), (2, 129, 8, 3, 128, "qk")])
def test_qk_norm_rope(dev, dtype, tables, b, s, hq, hk, d, norms):
    from torchplusplus_amd._native import ext
    cos, sin = (t.to(tables) for t in oracle.compute_rope_params(d, 1e6, s))
    q, k = _rand((b, s, hq, d), dtype, 1), _rand((b, s, hk, d), dtype, 2)
    qw = 1 + _rand((d,), dtype, 3) / 8 if "q" in norms else None
    kw = 1 + _rand((d,), dtype, 4) / 8 if "k" in norms else None
    up = lambda t: None if t is None else t.to(dev)  # noqa: E731
    # rows of one wider projection: token stride larger than the heads
    buf = torch.zeros(b, s, (hq + hk) * d + 8, dtype=dtype, device=dev)
    qd = buf[..., :hq * d].view(b, s, hq, d)
    kd = buf[..., hq * d:(hq + hk) * d].view(b, s, hk, d)
    qd.copy_(q.to(dev)), kd.copy_(k.to(dev))
    assert ext().qk_norm_rope_(qd, kd, up(qw), up(kw), 1e-6, 1e-5, up(cos), up(sin))
    close(qd, _want(q, qw, 1e-6, cos, sin), what="q")
    close(kd, _want(k, kw, 1e-5, cos, sin), what="k")
    assert torch.count_nonzero(buf[..., (hq + hk) * d:]) == 0


def test_qk_norm_rope_leaves_other_layouts_to_the_general_path(dev):
    """Head sizes, strides and alignments outside the kernel's are not touched
    and the layers' general path gives the oracle's result for them."""
    from torchplusplus_amd._native import ext
    from torchplusplus_amd.attention._common import norm_rope_qk
    for d, shift in ((96, 0), (32, 0), (64, 1)):
        cos, sin = (t.to(dev) for t in oracle.compute_rope_params(d, 1e6, 20))
        q, k = _rand((2, 20, 4, d), torch.bfloat16, 5), _rand((2, 20, 2, d), torch.bfloat16, 6)
        w = torch.zeros(d + 1, dtype=torch.bfloat16, device=dev)[shift:shift + d]  # shift: unaligned
        w.copy_(1 + _rand((d,), torch.bfloat16, 7).to(dev) / 8)
        qd, kd = q.to(dev), k.to(dev)
        assert not ext().qk_norm_rope_(qd, kd, w, w, 1e-6, 1e-6, cos, sin)
        assert torch.equal(qd.cpu(), q)
        norm = torch.nn.RMSNorm(d, eps=1e-6, dtype=torch.bfloat16, device=dev)
        norm.weight = torch.nn.Parameter(w, requires_grad=False)
        got = norm_rope_qk(qd, kd, norm, norm, cos, sin)
        for g, x in zip(got, (q, k)):
            close(g, _want(x, w.cpu(), 1e-6, cos.cpu(), sin.cpu()), what=f"d {d} shift {shift}")
    q = _rand((2, 4, 20, 64), torch.bfloat16, 8).to(dev).transpose(1, 2)  # head-major storage
    cos, sin = (t.to(dev) for t in oracle.compute_rope_params(64, 1e6, 20))
    assert not ext().qk_norm_rope_(q, q.clone(), None, None, 1e-6, 1e-6, cos, sin)
