"""GEMMs of few outputs (below 256 tiles of 128 x 128): the K-split tiles and
the small DMA tiles, at the edges of tiles, of the K chunks and of the tile
rule, against the oracle (atol 2e-2 / rtol 1e-2, the tolerance of every
16-bit output here)."""
import ctypes
import os
import shutil
import subprocess

import pytest
import torch

import oracle
from tests.conftest import close
from tests.test_asm_waits import CSRC, ROOT, scan

ACTS = {"none": 0, "gelu": 1, "silu": 2, "relu": 3}


def _mk(m, n, k, dtype, seed=0, wstd=0.05):
    g = torch.Generator().manual_seed(seed)
    x = torch.randn(m, k, generator=g).to(dtype)
    w = (wstd * torch.randn(n, k, generator=g)).to(dtype)
    return x, w, (wstd * torch.randn(n, generator=g)).to(dtype)


# (m, n, k): one output and one chunk; a wave without a chunk (k < 256); every
# remainder of the last chunk's 8-wide units; the 32x32, 64x32, 64x64 (4 and 2
# waves), 128x64 and 128x128 tiles with ragged edges, N no multiple of 8
SHAPES = [(17, 1, 8), (17, 33, 64), (31, 64, 72), (32, 96, 200), (33, 100, 248), (77, 1024, 3072),
          (65, 1003, 1000), (230, 1024, 2048), (300, 2048, 1000), (510, 1024, 1024),
          (230, 4096, 1024), (600, 1028, 520), (2000, 1024, 1024), (1990, 1030, 320),
          (1000, 3072, 1024), (1000, 4100, 64), (1024, 4095, 128), (513, 4000, 192),
          (6700, 570, 128), (2451, 1590, 64)]


@pytest.mark.gpu
@pytest.mark.parametrize("act,bias", [("none", False), ("gelu", True), ("silu", False)])
@pytest.mark.parametrize("m,n,k", SHAPES)
def test_linear_few_outputs(dev, m, n, k, act, bias):
    from torchplusplus_amd._native import ext
    dtype = torch.float16 if m % 2 else torch.bfloat16
    x, w, b = _mk(m, n, k, dtype, seed=m + k)
    b = b if bias else None
    y = ext().linear(x.to(dev), w.to(dev), None if b is None else b.to(dev), ACTS[act])
    close(y, oracle.linear_act(x, w, b, act), what=f"linear {act} {m}x{n}x{k}")


@pytest.mark.gpu
@pytest.mark.parametrize("m,i,k", [(17, 32, 64), (40, 96, 1000), (230, 3072, 1024), (512, 3072, 1024),
                                   (129, 2048, 768), (1000, 1024, 136)])
def test_swiglu_few_outputs(dev, m, i, k):
    from torchplusplus_amd._native import ext
    from torchplusplus_amd.dlops.linear import interleave_gate_up
    x, wg, _ = _mk(m, i, k, torch.bfloat16, seed=3)
    _, wu, _ = _mk(m, i, k, torch.bfloat16, seed=4)
    y = ext().linear_swiglu(x.to(dev), interleave_gate_up(wg, wu).to(dev))
    g = oracle.linear_act(x, wg, None, "silu").float()
    u = oracle.linear_act(x, wu, None, "none").float()
    close(y, (g * u).to(x.dtype), what=f"swiglu {m}x{i}x{k}")


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k", [(40, 96, 1000), (230, 1024, 264), (2000, 1024, 192)])
def test_linear_reads_nothing_past_a_row(dev, m, n, k):
    """Rows with a pitch: NaNs between them must not reach an output, and the
    output's own gap stays untouched."""
    from torchplusplus_amd._native import lib
    x, w, _ = _mk(m, n, k, torch.bfloat16, seed=5)
    xp = torch.full((m, k + 8), float("nan"), dtype=x.dtype, device=dev)
    xp[:, :k] = x.to(dev)
    out = torch.zeros(m, n + 8, dtype=x.dtype, device=dev)
    wd, i64, ptr = w.to(dev), ctypes.c_int64, ctypes.c_void_p
    rc = lib().tpp_linear_act(ptr(xp.data_ptr()), ptr(wd.data_ptr()), None, ptr(out.data_ptr()),
                              i64(m), i64(n), i64(k), i64(k + 8), i64(n + 8), ctypes.c_int(0),
                              ctypes.c_int(1), ptr(torch.cuda.current_stream().cuda_stream))
    assert rc == 0
    close(out[:, :n], oracle.linear_act(x, w, None, "none"), what="pitched rows")
    assert torch.count_nonzero(out[:, n:]) == 0


@pytest.mark.gpu
def test_linear_few_outputs_keeps_infinities(dev):
    """An infinity in the last K unit of a K that is no multiple of 64 reaches
    its row and no other (the units past K are zeros, not copies of it)."""
    from torchplusplus_amd._native import ext
    x, w, _ = _mk(40, 64, 1000, torch.bfloat16, seed=6)
    x[7, 999] = float("inf")
    y = ext().linear(x.to(dev), w.to(dev), None, 0).cpu()
    want = oracle.linear_act(x, w, None, "none")
    assert torch.equal(torch.isinf(y), torch.isinf(want)) and not torch.isnan(y).any()
    rows = [i for i in range(40) if i != 7]
    close(y[rows], want[rows], what="rows without the infinity")


@pytest.mark.skipif(shutil.which("hipcc") is None, reason="hipcc not installed")
def test_gemm_fragment_reads_waited_for(tmp_path):
    """The K-split kernel's asm fragment reads: no compiler-made instruction
    touches their registers before the wait."""
    out = str(tmp_path / "gemm.s")
    subprocess.run(["hipcc", "--offload-arch=gfx950", "-O3", "-std=c++17", "-Xclang", "-target-feature",
                    "-Xclang", "-packed-fp32-ops", "-ffp-contract=fast", f"-I{os.path.join(ROOT, 'include')}",
                    "--cuda-device-only", "-S", os.path.join(CSRC, "gemm.hip"), "-o", out],
                   check=True, stdout=subprocess.DEVNULL, stderr=subprocess.DEVNULL, timeout=600)
    loads, bad = scan(open(out).read())
    assert loads > 0 and not bad, "\n".join(bad[:10])


# (m, n, k, act, bias): 256x256 tiles over whole rounds and 128x128 tiles over
# the remaining rows (one row block and several, ragged M and N, one K step and
# more, one round and two)
@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k,act,bias", [(6227, 3072, 128, "gelu", True), (4100, 4000, 64, "relu", True),
                                            (5633, 3072, 64, "none", True), (9990, 3076, 192, "silu", False)])
def test_linear_mixed_tiles(dev, m, n, k, act, bias):
    from torchplusplus_amd._native import ext
    dtype = torch.float16 if m % 2 else torch.bfloat16
    x, w, b = _mk(m, n, k, dtype, seed=m)
    b = b if bias else None
    y = ext().linear(x.to(dev), w.to(dev), None if b is None else b.to(dev), ACTS[act])
    close(y, oracle.linear_act(x, w, b, act), what=f"mixed {act} {m}x{n}x{k}")


@pytest.mark.gpu
def test_swiglu_mixed_tiles(dev):
    from torchplusplus_amd._native import ext
    from torchplusplus_amd.dlops.linear import interleave_gate_up
    x, wg, _ = _mk(2900, 3072, 512, torch.bfloat16, seed=3)
    _, wu, _ = _mk(1, 3072, 512, torch.bfloat16, seed=4)
    y = ext().linear_swiglu(x.to(dev), interleave_gate_up(wg, wu).to(dev))
    g = oracle.linear_act(x, wg, None, "silu").float()
    close(y, (g * oracle.linear_act(x, wu, None, "none").float()).to(x.dtype), what="mixed swiglu")


THREE = [(17, (64, 64, 64), 72), (36, (1024, 128, 128), 1024), (100, (1024, 1024, 1024), 1024),
         (300, (1000, 33, 1), 520), (600, (512, 512, 100), 256), (1045, (1024, 1024, 1024), 192),
         (2000, (1024, 1024, 1024), 128), (2000, (1024, 64, 64), 64),
         (5000, (1024, 1024, 1030), 64), (3000, (1024, 1024, 1024), 1000), (321, (1024, 1024, 1024), 1024),
         (330, (1024, 1000, 1030), 200), (1366, (1024, 1024, 1024), 64), (2689, (1024, 1024, 1024), 128),
         (3300, (1024, 64, 64), 64), (3301, (1024, 70, 60), 192)]


@pytest.mark.gpu
@pytest.mark.parametrize("m,ns,k", THREE)
def test_three_projections(dev, m, ns, k):
    """Three outputs of one launch, at every tile it has: ragged rows and
    columns, a K tail, outputs narrower than a tile; bit-equal repeats."""
    from torchplusplus_amd._native import ext
    dtype = torch.float16 if m % 2 else torch.bfloat16
    x, _, _ = _mk(m, 1, k, dtype, seed=m)
    ws = [_mk(1, n, k, dtype, seed=n + i)[1] for i, n in enumerate(ns)]
    xd, wd = x.to(dev), [w.to(dev) for w in ws]
    got = ext().linear3(xd, *wd)
    for y, w, again in zip(got, ws, ext().linear3(xd, *wd)):
        close(y, oracle.linear_act(x, w, None, "none"), what=f"three {m}x{tuple(w.shape)}")
        assert torch.equal(y, again)


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k", [(2049, 2100, 8), (2049, 2100, 136), (4096, 4096, 72), (4090, 4099, 200),
                                   (4300, 4096, 72), (4300, 4099, 120), (6000, 1500, 1000)])
def test_k_tail_large(dev, m, n, k):
    """Large outputs whose K is a multiple of 8 but not of 64: 128x128 tiles,
    256x256 tiles and both, one and several K tiles, with every epilogue."""
    from torchplusplus_amd._native import ext
    from torchplusplus_amd.dlops.linear import interleave_gate_up
    dtype = torch.float16 if m % 2 else torch.bfloat16
    x, w, b = _mk(m, n, k, dtype, seed=k)
    xd, wd, bd = x.to(dev), w.to(dev), b.to(dev)
    close(ext().linear(xd, wd), oracle.linear_act(x, w, None, "none"), what=f"plain {m}x{n}x{k}")
    close(ext().linear(xd, wd, bd, ACTS["silu"]), oracle.linear_act(x, w, b, "silu"), what=f"silu {m}x{n}x{k}")
    i = n // 64 * 32
    wg, wu = w[:i], w[i:2 * i]
    y = ext().linear_swiglu(xd, interleave_gate_up(wg, wu).to(dev))
    g = oracle.linear_act(x, wg, None, "silu").float()
    close(y, (g * oracle.linear_act(x, wu, None, "none").float()).to(dtype), what=f"swiglu {m}x{i}x{k}")


def _tile(m, ns, k, fused=False, swiglu=False):
    """(rows, columns, waves that share K, rows of 256x256 tiles ahead)."""
    from torchplusplus_amd._native import lib
    out = (ctypes.c_int32 * 4)()
    rc = lib().tpp_linear_tiles(ctypes.c_int64(m), (ctypes.c_int64 * len(ns))(*ns), len(ns), ctypes.c_int64(k),
                                int(fused), int(swiglu), out)
    assert rc == 0
    return tuple(out)


SMALL = {(32, 32, 4, 0), (64, 32, 4, 0), (64, 64, 4, 0), (64, 64, 2, 0), (128, 64, 0, 0), (128, 128, 0, 0)}


def test_shapes_reach_every_tile():
    """The shapes above take every tile of the launches they are for (host
    arithmetic, 256 CUs): a retuned rule must not empty a case unseen."""
    for fused in (False, True):
        assert {_tile(m, [n], k, fused) for m, n, k in SHAPES} == SMALL
    separate = (0, 0, 0, 0)
    assert {_tile(m, ns, k) for m, ns, k in THREE} == SMALL | {
        (128, 192, 0, 0), (128, 256, 0, 0), (256, 256, 0, 0), separate}
    for m, n, k in ((6227, 3072, 128), (4100, 4000, 64), (5633, 3072, 64), (9990, 3076, 192)):
        assert _tile(m, [n], k, fused=True)[3] > 0
    assert _tile(2900, [6144], 512, swiglu=True)[3] > 0
