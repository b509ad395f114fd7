"""Layer calls that run whole in the binding: the same results as the separate
calls they replace, and the same refusals."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _rand(shape, dtype, seed):
    return torch.randn(*shape, generator=torch.Generator().manual_seed(seed)).to(dtype)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("b,s,start,rows", [(1, 1, 0, 1), (3, 1, 130, 5), (2, 17, 0, 2), (2, 33, 95, 4)])
def test_gqa_attend_equals_separate_calls(dev, dtype, b, s, start, rows):
    """Bit-exact against qkv_rope_cache with a positions tensor + attention
    (and attn_decode_fused with lengths), caches allocated for more sequences
    than the call has; without a cache the same at start 0."""
    from torchplusplus_amd._native import ext
    C, hq, hkv, d, cap = ext(), 4, 2, 64, 256
    qkv = _rand((b, s, (hq + 2 * hkv) * d), dtype, 1).to(dev)
    qw, kw = (1 + _rand((d,), dtype, i).to(dev) / 8 for i in (2, 3))
    cos, sin = (_rand((cap, d), torch.float16, i).to(dev) for i in (4, 5))
    base = [_rand((rows, hkv, cap, d), dtype, i).to(dev) for i in (6, 7)]
    got_c, want_c = [t.clone() for t in base], [t[:b].clone() for t in base]
    got = C.gqa_attend(qkv, qw, kw, 1e-6, cos, sin, *got_c, start, hq, hkv, d)
    if s == 1:
        lens = torch.full((b,), start + 1, dtype=torch.int32, device=dev)
        want = C.attn_decode_fused(qkv, qw, kw, cos, sin, 1e-6, *want_c, lens)
    else:
        q = torch.empty(b, s, hq, d, dtype=dtype, device=dev)
        pos = torch.full((b,), start, dtype=torch.int32, device=dev)
        C.qkv_rope_cache(qkv, q, *want_c, qw, kw, cos, sin, pos, 1e-6)
        want = C.flash_attn_func(q, *(t[:, :, :start + s].transpose(1, 2) for t in want_c), True)
    assert torch.equal(got, want.reshape(b, s, hq * d))
    for g, w, o in zip(got_c, want_c, base):
        assert torch.equal(g[:b], w) and torch.equal(g[b:], o[b:])
    if s > 1:
        plain = C.gqa_attend(qkv, qw, kw, 1e-6, cos, sin, None, None, 0, hq, hkv, d)
        fresh = [torch.zeros(b, hkv, s, d, dtype=dtype, device=dev) for _ in range(2)]
        assert torch.equal(plain, C.gqa_attend(qkv, qw, kw, 1e-6, cos, sin, *fresh, 0, hq, hkv, d))
    with pytest.raises(RuntimeError):
        C.gqa_attend(qkv, qw, kw, 1e-6, cos, sin, *got_c, cap, hq, hkv, d)  # past the cache


@pytest.mark.parametrize("qk_norm", [True, False])
def test_gqa_sequences_at_their_own_positions(dev, qk_norm):
    """rope_cache and decode_fused with a position per sequence: each sequence
    gets the cache rows (bit-exact) and the output that a call of its own at
    that position gives."""
    from tests.conftest import close
    from torchplusplus_amd.attention import GroupedQueryAttention
    from torchplusplus_amd.llmops.kvcache import KVCache
    hq, hkv, d, cap, dtype = 4, 2, 64, 256, torch.bfloat16
    mod = GroupedQueryAttention(256, hq, hkv, d, qk_norm=qk_norm, dtype=dtype, device=dev).eval()
    cos, sin = (_rand((cap, d), torch.float16, i).to(dev) for i in (4, 5))
    base = [_rand((2, hkv, cap, d), dtype, i).to(dev) for i in (6, 7)]
    starts = [5, 131]
    pos = torch.tensor(starts, dtype=torch.int32, device=dev)
    for s in (1, 20):
        qkv = _rand((2, s, (hq + 2 * hkv) * d), dtype, s).to(dev)
        got = [t.clone() for t in base]
        with torch.no_grad():
            if s == 1:
                out = mod.decode_fused(qkv, cos, sin, *got, pos + 1).reshape(2, 1, hq * d)
            else:
                mod.rope_cache(qkv, cos, sin, *got, pos)
            for b, start in enumerate(starts):
                cache = KVCache(cap, hkv, d, dtype, dev, 1)
                cache.update(base[0][b:b + 1], base[1][b:b + 1])
                alone = mod.attend(qkv[b:b + 1].contiguous(), cos, sin, cache, start)
                assert torch.equal(got[0][b], cache.k_cache[0]) and torch.equal(got[1][b], cache.v_cache[0])
                if s == 1:
                    close(out[b:b + 1], alone, what=f"sequence {b} at {start}")


@pytest.mark.parametrize("rows", [1, 16, 17, 40])
def test_ffn_and_projections_equal_separate_calls(dev, rows):
    from torchplusplus_amd._native import ext
    C = ext()
    x = _rand((1, rows, 256), torch.bfloat16, 1).to(dev)
    w_gu, w_down = _rand((1024, 256), torch.bfloat16, 2).to(dev) / 16, _rand((256, 512), torch.bfloat16, 3).to(dev) / 16
    h = C.gemv_swiglu(x, w_gu) if rows <= 16 else C.linear_swiglu(x, w_gu)
    want = C.gemv(h, w_down) if rows <= 16 else C.linear(h, w_down)
    assert torch.equal(C.ffn_forward(x, w_gu, w_down), want)
    for got, w in zip(C.linear3(x, w_gu, w_gu[:64], w_gu[64:96]), (w_gu, w_gu[:64], w_gu[64:96])):
        assert torch.equal(got, C.linear_any(x, w))


def test_source_key_follows_edits(dev):
    """In-place edits, other storage, other shapes and inference tensors all
    give another key; reading does not."""
    from torchplusplus_amd._native import ext
    key = ext().source_key
    w = torch.zeros(8, 8, device=dev)
    k0 = key([w, w])
    w.sum()
    assert key([w, w]) == k0 and key([w]) != k0
    w.add_(1)
    assert key([w, w]) != k0
    assert key([w]) != key([w.clone()]) and key([w]) != key([w.view(4, 16)])
    with torch.inference_mode():
        i = torch.zeros(8, 8, device=dev)
        assert key([i]) == key([i])
