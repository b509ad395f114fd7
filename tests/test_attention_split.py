"""Prefill attention with few work items: the key-split kernel, one chunk and
several (partials merged by a second launch), against the CPU oracle (atol
2e-2 / rtol 1e-2, the tolerance of every 16-bit output here)."""
import pytest
import torch

import oracle
from tests.conftest import close

pytestmark = pytest.mark.gpu


def _qkv(b, sq, sk, hq, hkv, d, dtype, seed=0):
    g = torch.Generator().manual_seed(seed)
    return [torch.randn(b, s, h, d, generator=g).to(dtype) for s, h in ((sq, hq), (sk, hkv), (sk, hkv))]


def _workspace(b, sq, sk, hq, hkv, d, causal, window):
    import ctypes
    from torchplusplus_amd._native import lib
    f = lib().tpp_attn_prefill_workspace_size
    f.restype = ctypes.c_size_t
    i64 = ctypes.c_int64
    return f(i64(b), i64(sq), i64(sk), i64(hq), i64(hkv), i64(d), int(causal), window[0], window[1])


# one key; tile and query-tile edges (32 / 64 keys, 32 / 64 queries, one past);
# groups of 1, 2, 3, 4 and 8 heads per KV head; Sq > Sk (rows without a key);
# windows that begin inside a tile; pair counts that split over the XCDs or not
ONE_CHUNK = [(1, 1, 1, 2, 1, 128, True, (-1, -1)), (1, 17, 33, 4, 2, 128, True, (-1, -1)),
             (2, 32, 32, 8, 8, 128, True, (-1, -1)), (1, 33, 64, 16, 8, 128, False, (-1, -1)),
             (1, 65, 129, 3, 3, 64, True, (-1, -1)), (1, 64, 65, 6, 2, 64, False, (-1, -1)),
             (1, 100, 40, 8, 2, 128, True, (-1, -1)), (1, 230, 230, 16, 8, 128, True, (-1, -1)),
             (2, 200, 300, 16, 2, 64, True, (70, 0)), (1, 300, 300, 8, 4, 128, True, (33, 0)),
             (1, 90, 200, 4, 4, 128, False, (20, 50)), (1, 600, 700, 16, 8, 128, True, (-1, -1))]
CHUNKS = [(1, 1, 3000, 8, 8, 64, False, (-1, -1)), (1, 33, 4001, 16, 8, 128, True, (-1, -1)),
          (1, 200, 3001, 16, 8, 128, True, (-1, -1)), (2, 40, 2500, 4, 1, 64, True, (-1, -1)),
          (1, 70, 2050, 3, 1, 128, True, (2000, 0)), (1, 17, 5000, 12, 4, 64, False, (-1, -1))]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("b,sq,sk,hq,hkv,d,causal,window", ONE_CHUNK + CHUNKS)
def test_split_prefill(dev, dtype, b, sq, sk, hq, hkv, d, causal, window):
    from torchplusplus_amd.attention import flash_attn_func
    shape = (b, sq, sk, hq, hkv, d, causal, window)
    assert (_workspace(*shape) > 0) == (shape in CHUNKS)
    q, k, v = _qkv(b, sq, sk, hq, hkv, d, dtype, seed=sq + sk)
    # k and v as views of a cache [B, H, L, D] with rows past Sk that must not be read
    cache = torch.full((2, b, hkv, sk + 3, d), float("nan"), dtype=dtype, device=dev)
    cache[0, :, :, :sk], cache[1, :, :, :sk] = k.transpose(1, 2).to(dev), v.transpose(1, 2).to(dev)
    kd, vd = (c[:, :, :sk].transpose(1, 2) for c in cache)
    o = flash_attn_func(q.to(dev), kd, vd, causal=causal, window_size=window)
    close(o, oracle.attention(q, k, v, causal=causal, window=window), what=f"split prefill {shape}")
    again = flash_attn_func(q.to(dev), kd, vd, causal=causal, window_size=window)
    assert torch.equal(o, again)


# windows whose widest query tile is not the first, middle or last one: key
# tiles of 64 against 32 queries (odd and even tiles differ), a middle tile cut
# at key 0 beside a short last one, bounds on both sides; one chunk and several
WINDOWS = [(1, 300, 300, 16, 8, 64, True, (200, 0)), (1, 700, 700, 16, 8, 64, True, (200, 0)),
           (1, 400, 400, 8, 8, 128, True, (199, 0)), (1, 340, 340, 16, 16, 128, True, (199, 0)),
           (1, 900, 1100, 8, 4, 128, True, (1000, 0)), (1, 784, 784, 24, 8, 64, False, (601, 77)),
           (1, 260, 260, 16, 8, 128, False, (199, 50)), (1, 177, 2495, 24, 6, 64, False, (1392, 78)),
           (1, 521, 821, 4, 4, 128, True, (700, 0))]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("b,sq,sk,hq,hkv,d,causal,window", WINDOWS)
def test_split_prefill_windows(dev, dtype, b, sq, sk, hq, hkv, d, causal, window):
    from torchplusplus_amd.attention import flash_attn_func
    q, k, v = _qkv(b, sq, sk, hq, hkv, d, dtype, seed=sq)
    o = flash_attn_func(q.to(dev), k.to(dev), v.to(dev), causal=causal, window_size=window)
    close(o, oracle.attention(q, k, v, causal=causal, window=window), what=f"window {window} of {sq} x {sk}")


@pytest.mark.parametrize("embed,heads,seq", [(1024, 8, 400), (1024, 16, 340), (512, 8, 700)])
def test_sliding_window_layer_of_200(dev, embed, heads, seq):
    """A window that is no power of two, through the layer (oracle/modules.py)."""
    from oracle import modules as om
    from tests.test_modules import _randomize, _tables, _x
    from torchplusplus_amd.attention import SlidingWindowAttention
    mod = SlidingWindowAttention(200, embed, heads, dtype=torch.bfloat16, device=dev)
    p, x = _randomize(mod, 3), _x((1, seq, embed), torch.bfloat16, 4)
    c, s, cd, sd = _tables(embed // heads, seq, dev)
    with torch.no_grad():
        got = mod(x.to(dev), cd, sd)
    close(got, om.mha(x, p, c, s, heads, window_size=200), what=f"SWA 200 over {seq}")


def test_split_prefill_captured(dev):
    """Several chunks inside a graph: every replay equals the eager result."""
    from torchplusplus_amd.attention import flash_attn_func
    q, k, v = (t.to(dev) for t in _qkv(1, 33, 4001, 16, 8, 128, torch.bfloat16, seed=9))
    want = flash_attn_func(q, k, v, causal=True)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        o = flash_attn_func(q, k, v, causal=True)
    for _ in range(3):
        o.zero_()
        graph.replay()
        assert torch.equal(o, want)
        assert torch.equal(flash_attn_func(q, k, v, causal=True), want)


def test_split_prefill_nan_stays_in_its_row(dev):
    """A NaN query makes its own rows NaN in both forms, and no other."""
    from torchplusplus_amd.attention import flash_attn_func
    for sq, sk in ((100, 100), (33, 4001)):
        q, k, v = _qkv(1, sq, sk, 4, 2, 128, torch.bfloat16, seed=4)
        q[0, 20, 3] = float("nan")
        o = flash_attn_func(q.to(dev), k.to(dev), v.to(dev), causal=True).cpu()
        assert torch.isnan(o[0, 20, 3]).all()
        o[0, 20, 3] = 0
        q[0, 20, 3] = 0
        want = oracle.attention(q, k, v, causal=True)
        want[0, 20, 3] = 0
        close(o, want, what="rows without the NaN")


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("b,hq,hkv,d,cap,window", [
    (8, 16, 8, 128, 3000, -1),   # splits merged in the kernel
    (3, 6, 3, 64, 2500, -1),     # merge kernel, groups of two
    (2, 8, 2, 128, 5000, -1),    # groups of four
    (8, 16, 8, 128, 3000, 200),  # a window, from inside a batch
    (1, 8, 1, 64, 4097, 700), (16, 8, 8, 128, 130, -1)])
def test_decode_lengths_far_below_the_capacity(dev, dtype, b, hq, hkv, d, cap, window):
    """Sequences of every length in one batch (none, one key, a batch of keys
    and one more, all of the capacity, past it): the keys are dealt to the
    splits by each sequence's length. The workspace starts as NaN past its
    counters, so a slot that no split wrote must not be read."""
    import ctypes
    from torchplusplus_amd._native import lib
    g = torch.Generator().manual_seed(cap)
    q = torch.randn(b, 1, hq, d, generator=g).to(dtype)
    k, v = (torch.randn(b, hkv, cap, d, generator=g).to(dtype) for _ in range(2))
    pool = [0, 1, 129, cap, cap + 5, 128, 511, 2 * cap // 3, 64, 65, 700, 2, cap - 1, 257, 300, 1000]
    lens = torch.tensor([min(x, cap + 5) for x in pool[:b]] if b > 1 else [300], dtype=torch.int32)
    lb, ptr, i64 = lib(), ctypes.c_void_p, ctypes.c_int64
    lb.tpp_attn_decode_workspace_size.restype = ctypes.c_size_t
    size = lb.tpp_attn_decode_workspace_size(*map(i64, (b, hq, hkv, d, cap)))
    ws = torch.full((size // 4 + 64,), float("nan"), dtype=torch.float32, device=dev)
    ws[:16384] = 0
    qd, kd, vd, ld = q.to(dev), k.to(dev), v.to(dev), lens.to(dev)
    o = torch.full_like(qd, float("nan"))
    s3 = lambda *a: (i64 * 3)(*a)  # noqa: E731
    for _ in range(2):  # the second call finds the counters at zero again
        rc = lb.tpp_attn_decode(
            ptr(qd.data_ptr()), ptr(kd.data_ptr()), ptr(vd.data_ptr()), ptr(o.data_ptr()),
            s3(hq * d, hq * d, d), s3(hkv * cap * d, d, cap * d), s3(hkv * cap * d, d, cap * d),
            s3(hq * d, hq * d, d), ptr(ld.data_ptr()), i64(b), i64(hq), i64(hkv), i64(d), i64(cap),
            ctypes.c_float(0), ctypes.c_int(window), ctypes.c_int(0 if dtype == torch.float16 else 1),
            ptr(ws.data_ptr()), ctypes.c_size_t(size), ptr(torch.cuda.current_stream().cuda_stream))
        assert rc == 0
        want = oracle.decode_attention(q, k, v, lens.clamp(max=cap), window_left=window)
        close(o, want, what=f"decode lens {lens.tolist()} cap {cap} window {window}")
        o.fill_(float("nan"))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("b,hq,hkv,d,lens,cap,window", [
    (1, 3, 1, 128, [1], 40, -1), (2, 4, 1, 128, [31, 33], 64, -1), (2, 10, 2, 64, [64, 65], 300, -1),
    (3, 8, 1, 128, [0, 129, 500], 512, -1), (8, 32, 8, 128, [5, 700, 128, 1500, 2000, 2, 256, 999], 2000, -1),
    (4, 24, 4, 64, [3000, 1, 257, 1024], 4000, -1), (8, 8, 1, 128, [900] * 8, 1000, 300),
    (1, 28, 4, 64, [2100], 2100, 65), (4, 16, 8, 128, [1, 33, 640, 900], 1000, -1),
    (1, 2, 1, 64, [4000], 4096, 50)])
def test_decode_groups(dev, dtype, b, hq, hkv, d, lens, cap, window):
    """Two to eight query heads per KV head (the matrix-core kernel): wave
    and tile edges, empty sequences, windows, one split and several; rows past
    each length hold NaN and must not be read."""
    from torchplusplus_amd.attention import decode_attention
    g = torch.Generator().manual_seed(hq + cap)
    q = torch.randn(b, 1, hq, d, generator=g).to(dtype)
    k, v = (torch.randn(b, hkv, cap, d, generator=g).to(dtype) for _ in range(2))
    sl = torch.tensor(lens, dtype=torch.int32)
    kd, vd = k.to(dev), v.to(dev)
    for i, n in enumerate(lens):
        if n:
            kd[i, :, n:], vd[i, :, n:] = float("nan"), float("nan")
    o = decode_attention(q.to(dev), kd, vd, sl.to(dev), window_left=window)
    close(o, oracle.decode_attention(q, k, v, sl, window_left=window), what=f"group of {hq // hkv}, lens {lens}")


def test_decode_group_keeps_infinities(dev):
    """An infinite value in V makes its column infinite, not NaN, and no other."""
    from torchplusplus_amd.attention import decode_attention
    g = torch.Generator().manual_seed(3)
    q = torch.randn(1, 1, 4, 128, generator=g).bfloat16()
    k, v = (torch.randn(1, 1, 300, 128, generator=g).bfloat16() for _ in range(2))
    v[0, 0, 50, 7], v[0, 0, 131, 100] = float("inf"), float("-inf")
    sl = torch.tensor([290], dtype=torch.int32)
    o = decode_attention(q.to(dev), k.to(dev), v.to(dev), sl.to(dev)).cpu()
    want = oracle.decode_attention(q, k, v, sl)
    assert torch.equal(torch.isinf(o), torch.isinf(want)) and not torch.isnan(o).any()
    fin = torch.isfinite(want)
    close(o[fin], want[fin], what="finite columns")


def _decode_64(q, k, v, n):
    """64-bit decode attention of one sequence, one KV head: q [1, 1, H, D]."""
    s = q[0, 0].double() @ k[0, 0, :n].double().t() / q.shape[-1] ** 0.5
    return torch.softmax(s, dim=-1) @ v[0, 0, :n].double()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("bits,value", [(20, 3.0), (26, 500.0), (40, 30000.0)])
def test_decode_group_keeps_small_probabilities(dev, dtype, d, bits, value):
    """One key of weight 1 whose V is zero, and 3000 of about 2^-bits: their
    sum is all there is. The result is rounded to T once; fp32 sums of 3000
    equal terms add less than that (2^-24 * 3000 / 2 < 2^-13). V stays below the
    largest half (65504), the results above the smallest normal one (2^-14)."""
    from torchplusplus_amd.attention import decode_attention
    q, k, v = (torch.zeros(1, s, h, d).to(dtype) for s, h in ((1, 4), (1, 3001), (1, 3001)))
    q[..., 0] = 16
    k[0, 0, 777, 0] = bits * 0.6931 * d ** 0.5 / 16
    v[0, 0] = value * (1 + torch.arange(d) / d).to(dtype)
    v[0, 0, 777] = 0
    o = decode_attention(q.to(dev), k.to(dev), v.to(dev), torch.tensor([3001], dtype=torch.int32, device=dev))
    want = _decode_64(q, k, v, 3001)
    rel = 2.0 ** (-8 if dtype == torch.bfloat16 else -11) + 2.0 ** -13
    err = (o[0, 0].double().cpu() - want).abs() / want
    assert err.max() <= rel, f"weights 2^-{bits}: relative error {err.max():.2e}"


@pytest.mark.parametrize("d", [64, 128])
def test_decode_group_keeps_24_bits_of_a_probability(dev, d):
    """A weight w in (0.5, 1) against its two leading bfloat16 parts, taken off
    by two keys of weight 1: what is left, w - hi - mid, is near 2^-18 and has
    the error of fp32 alone (2^-24 each for the weight and three sums: 2^-22,
    a sixteenth of it)."""
    from torchplusplus_amd.attention import decode_attention
    steps = torch.arange(1, 200, dtype=torch.float64) / 512
    kb = (-steps).bfloat16()
    w = torch.exp(16 * kb.double() / d ** 0.5)
    hi = w.bfloat16()
    mid = (w - hi.double()).bfloat16()
    left = (w - hi.double() - mid.double()).abs()
    best = int(torch.where(w > 0.5, left, torch.zeros_like(left)).argmax())
    assert left[best] > 2.0 ** -19
    q, k, v = (torch.zeros(1, s, h, d).bfloat16() for s, h in ((1, 4), (1, 300), (1, 300)))
    q[..., 0] = 16
    k[0, 0, :, 0] = -8
    k[0, 0, 17:20, 0] = torch.stack([torch.zeros_like(kb[best]), torch.zeros_like(kb[best]), kb[best]])
    for row, value in ((17, -hi[best]), (18, -mid[best]), (19, torch.ones(()))):
        v[0, 0, row] = value
    o = decode_attention(q.to(dev), k.to(dev), v.to(dev), torch.tensor([300], dtype=torch.int32, device=dev))
    want = _decode_64(q, k, v, 300)
    err = ((o[0, 0].double().cpu() - want) / want).abs().max()
    assert err <= 2.0 ** -22 / left[best] + 2.0 ** -8, f"relative error {err:.2e}"
