"""The four-wave kernel's tiles of 256 rows x 192 columns: the sums are the per-tile kernel's, in its order, so its bits are the
reference: waves whose 96 columns lie in one block of weight scales, in two of them, in the last one and past it; row tiles and
column tiles of one row or column group; few and many tiles per block.  The fused QKV projection: exact cases."""
import pytest
import torch

import modular_amd as mx
from modular_amd import _lib, synth
from test_gpu_qkv import run_case
from test_gpu_qkv_four_wave import BLOCK, RAGGED, ROW

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,N,K", [(256, 192, 512), (257, 200, 512), (65, 96, 768), (511, 104, 512), (300, 224, 1024), (161, 1544, 768),
                                   (255, 384, 512), (4096, 2112, 1024), (2011, 6144, 512), (8192, 9000, 512)])
@pytest.mark.parametrize("kind", ["block", "row"])
def test_bits_of_the_per_tile_kernel(dev, tune, M, N, K, kind):
    a, b = synth.random_fp8((M, K), M).to(dev), synth.random_fp8((N, K), N + 1).to(dev)
    if kind == "block":
        sa, sb = synth.random_scales((K // 128, M), 3).to(dev), synth.random_scales((-(-N // 128), K // 128), 4).to(dev)
        gran, g, a_ld, b_ld = (_lib.GRAN_BLOCK, _lib.GRAN_BLOCK), (1, 128, 128), M, K // 128
    else:
        sa, sb = synth.random_scales((1, M), 3, lo=0.01, hi=0.1).to(dev), synth.random_scales((N, 1), 4, lo=0.001, hi=0.01).to(dev)
        gran, g, a_ld, b_ld = (_lib.GRAN_COLWISE, _lib.GRAN_ROWWISE), (-1, -1, -1), M, 1
    stream = torch.cuda.current_stream(dev).cuda_stream

    def run(c):
        assert 0 == _lib.lib().maxfp8_matmul_dynamic_scaled_fp8(
            c.data_ptr(), a.data_ptr(), b.data_ptr(), sa.data_ptr(), sb.data_ptr(), M, N, K, K, K, N, *gran, *g, a_ld, b_ld,
            _lib.BF16, _lib.F32, _lib.ALGO_TILED, None, 0, stream), _lib.last_error()

    tune(MAXFP8_TILE="1", MAXFP8_W4="8")
    assert _lib.matmul_tall(M, N, K, kind == "block", False)
    guard = torch.full((M + 2, N), -7.0, dtype=torch.bfloat16, device=dev)
    again = torch.empty((M, N), dtype=torch.bfloat16, device=dev)
    run(guard[1:M + 1])
    run(again)
    tune(MAXFP8_TILE="1", MAXFP8_W4=None, MAXFP8_PERSIST="0")
    want = torch.empty((M, N), dtype=torch.bfloat16, device=dev)
    run(want)
    assert torch.equal(guard[1:M + 1].view(torch.int16), want.view(torch.int16))
    assert torch.equal(again.view(torch.int16), want.view(torch.int16))
    assert bool((guard[0] == -7.0).all()) and bool((guard[M + 1] == -7.0).all())


def test_where_they_are_taken():
    assert _lib.matmul_tall(2011, 6144, 4096) and _lib.matmul_tall(2048, 24576, 7168, False)
    # (as many tiles of 192 x 256 and a long K; half a round; row tiles mostly padding; K not an even number of slabs)
    assert not any(_lib.matmul_tall(*s) for s in ((16384, 8192, 28672), (2048, 2112, 4096), (260, 24576, 4096), (2011, 6144, 4096 + 128)))


# (Q, K and V meet inside a wave's columns; no Q at all; heads whose ends are tiles' ends)
@pytest.mark.parametrize("heads", [dict(Hq=21, H=7, D=16), dict(Hq=0, H=21, D=16, k_only=True), dict(Hq=6, H=2, D=64), dict(Hq=3, H=1, D=128)])
@pytest.mark.parametrize("mnk", [BLOCK, ROW])
@pytest.mark.parametrize("prompt,cached,page", RAGGED)
def test_fused_qkv_exact(dev, tune, heads, mnk, prompt, cached, page):
    tune(MAXFP8_W4="8")
    run_case(dev, prompt, cached, K=512, mnk=mnk, page=page, layers=2, layer=1, nblocks=40, seed=8, algo="tiled", exact=True,
             bias="k_only" not in heads, **heads)


# (the first tile's rows: the starts of up to 63 sequences sit in a wave's lanes, those of more are searched in memory; empty ones among them)
@pytest.mark.parametrize("batch", [1, 2, 62, 63, 64, 130])
@pytest.mark.parametrize("tm", ["4", "8"])
def test_fused_qkv_sequences(dev, tune, tm, batch):
    tune(MAXFP8_W4=tm)
    prompt, cached = [(5 * i + 3) % 8 * (40 if batch < 3 else 1) for i in range(batch)], [(7 * i) % 50 for i in range(batch)]
    run_case(dev, prompt, cached, Hq=6, H=2, D=64, K=512, mnk=ROW, page=16, layers=1, layer=0, nblocks=1100, seed=batch,
             algo="tiled", exact=True)


@pytest.mark.parametrize("kind", ["block", "row"])
@pytest.mark.parametrize("out", [torch.bfloat16, torch.float32])
def test_the_same_without_the_workspace_that_is_not_asked_for(dev, kind, out):
    """A plan that cuts a tail, behind tiles of 256 x 192: whatever the result's type, a workspace changes nothing."""
    M, N, K = 1216, 28672, 4096
    L = _lib.lib()
    need = L.maxfp8_matmul_workspace_bytes(M, N, K)
    assert L.maxfp8_matmul_auto_workspace_bytes(M, N, K) == 0 < need
    a, b = synth.random_fp8((M, K), 1).to(dev), synth.random_fp8((N, K), 2).to(dev)
    if kind == "block":
        sa, sb = synth.random_scales((K // 128, M), 3).to(dev), synth.random_scales((N // 128, K // 128), 4).to(dev)
        how = (_lib.GRAN_BLOCK, _lib.GRAN_BLOCK, 1, 128, 128, M, K // 128)
    else:
        sa, sb = synth.random_scales((1, M), 3, lo=0.01, hi=0.1).to(dev), synth.random_scales((N, 1), 4, lo=0.001, hi=0.01).to(dev)
        how = (_lib.GRAN_COLWISE, _lib.GRAN_ROWWISE, -1, -1, -1, M, 1)
    workspace = torch.empty(need, dtype=torch.uint8, device=dev)
    results = []
    for ws, size in ((workspace.data_ptr(), need), (None, 0)):
        c = torch.full((M, N), float("nan"), dtype=out, device=dev)
        assert 0 == L.maxfp8_matmul_dynamic_scaled_fp8(c.data_ptr(), a.data_ptr(), b.data_ptr(), sa.data_ptr(), sb.data_ptr(), M, N, K, K, K, N, *how,
                                                       _lib.BF16 if out == torch.bfloat16 else _lib.F32, _lib.F32, _lib.ALGO_AUTO, ws, size,
                                                       torch.cuda.current_stream(dev).cuda_stream), _lib.last_error()
        results.append(c)
    assert bool(torch.isfinite(results[0].float()).all()) and torch.equal(*results)
