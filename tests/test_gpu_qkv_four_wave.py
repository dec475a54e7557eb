"""The fused QKV projection on the four-wave kernel (whole tiles of 128, 160 and 192 rows, and tiles cut along K), and on the
three-stage tiles: edges of tiles inside and between Q, K and V, rows of several sequences in a wave's part, pages shorter
and longer than it, rows past the last one."""
import pytest
import torch

import modular_amd as mx
from modular_amd import synth
from test_gpu_qkv import run_case

pytestmark = pytest.mark.gpu

BLOCK, ROW, TENSOR = (1, 128, 128), (1, 1, -1), (-1, -1, -1)
# prompts, cached lengths, page size: one sequence per wave's part with a page edge in it; short sequences and pages (the search
# row by row); an empty sequence, and a last tile of a few rows
RAGGED = [([210, 190], [100, 37], 128), ([7, 60, 1, 0, 33, 90, 5], [3, 0, 40, 9, 31, 64, 2], 16), ([385, 0, 8], [0, 5, 250], 256)]


@pytest.mark.parametrize("tm", [4, 5, 6])
@pytest.mark.parametrize("mnk", [BLOCK, ROW])
@pytest.mark.parametrize("prompt,cached,page", RAGGED)
def test_whole_tiles_exact(dev, tune, tm, mnk, prompt, cached, page):
    tune(MAXFP8_W4=str(tm))
    # q_dim 336, K and V 112 wide: all three meet inside the 64-column steps of the second column tile
    run_case(dev, prompt, cached, Hq=21, H=7, D=16, K=512, mnk=mnk, page=page, layers=2, layer=1, nblocks=40, seed=tm,
             algo="tiled", bias=True, exact=True)


@pytest.mark.parametrize("mnk", [BLOCK, ROW])
@pytest.mark.parametrize("kv_dim", [1, 2])
def test_key_cache_only(dev, tune, mnk, kv_dim):
    """No Q at all: every column of every tile goes to the pages, C is null with rows of no length (the K-cache matmul)."""
    tune(MAXFP8_W4="5")
    run_case(dev, [210, 0, 190], [100, 3, 37], Hq=0, H=21, D=16, K=512, mnk=mnk, page=128, layers=2, layer=1, nblocks=40, seed=8,
             algo="tiled", k_only=True, kv_dim=kv_dim, exact=True)


@pytest.mark.parametrize("mnk", [BLOCK, ROW, TENSOR])
def test_whole_tiles(dev, tune, mnk):
    tune(MAXFP8_W4="6")
    run_case(dev, [300, 1, 129], [5, 0, 127], Hq=6, H=2, D=64, K=1024, mnk=mnk, page=128, layers=1, layer=0, nblocks=12, seed=2,
             algo="tiled", bias=True)


@pytest.mark.parametrize("tile", ["2", "4"])
@pytest.mark.parametrize("mnk", [BLOCK, ROW])
def test_three_stage_tiles_exact(dev, tune, tile, mnk):
    tune(MAXFP8_TILE=tile)
    run_case(dev, [130, 1, 0, 260], [3, 0, 2, 9], Hq=6, H=2, D=64, K=640, mnk=mnk, page=64, layers=3, layer=1, nblocks=16, seed=3,
             algo="tiled", bias=True, exact=True)
    run_case(dev, [130, 1, 0, 260], [3, 0, 2, 9], Hq=3, H=2, D=16, K=640, mnk=mnk, page=64, layers=3, layer=1, nblocks=16, seed=4,
             algo="tiled", bias=True, exact=True)


@pytest.mark.parametrize("T", [192, 500])
@pytest.mark.parametrize("scaling", ["row", "block"])
def test_cut_tiles(dev, tune, scaling, T):
    """Every tile cut, its pieces' sums exchanged: with row scaling and whole-number inputs every sum is exact in any order, so
    the bits are those of whole tiles; block scaling folds a product of scales in per slab, a bf16 step apart."""
    H, heads, kv_heads, D = 2048, 8, 2, 128
    cfg = mx.rowwise_fp8_config() if scaling == "row" else mx.blockwise_fp8_config()
    N = (heads + 2 * kv_heads) * D
    g = torch.Generator().manual_seed(T)
    x = torch.randint(-1, 2, (T, H), generator=g).to(torch.bfloat16)
    x[:, 0] = 1.0  # (every row has the same scale)
    w = torch.randint(-1, 2, (N, H), generator=g).float().to(torch.float8_e4m3fn).to(dev)
    ws = torch.ones((N, 1)) if scaling == "row" else synth.random_scales((N // 128, H // 128), 1)
    params = mx.KVCacheParams(torch.bfloat16, kv_heads, D, 1, 128)
    offsets = torch.tensor([0, T // 3, T], dtype=torch.int32).to(dev)
    table = torch.arange(12, dtype=torch.int32).reshape(2, 6).to(dev)
    outs = []
    for switches in ({"MAXFP8_W4": "0"}, {"MAXFP8_W4": "4"}, {"MAXFP8_W4": "4", "MAXFP8_W4_SPLIT": "1"}):
        tune(**switches)
        for _ in range(2):  # (the flags are put back by the launch that used them)
            blocks = torch.zeros(params.blocks_shape(12), dtype=torch.bfloat16, device=dev)
            cache = mx.PagedCacheValues(blocks, torch.tensor([100, 7], dtype=torch.int32).to(dev), table)
            q = mx.quantized_fused_qkv_matmul(params, x.to(dev), w, cache, 0, offsets, heads, cfg, ws.to(dev))
        outs.append((q.float(), blocks.float()))
    for other in outs[1:]:
        for a, b in zip(outs[0], other):
            if scaling == "row":
                assert torch.equal(a, b)
            else:
                # one bf16 step is at most 2^-7 of a value; sums that cancel: of the rms
                rms = a[a != 0].square().mean().sqrt()
                assert bool(((a - b).abs() <= 2.0 ** -7 * torch.maximum(a.abs(), rms)).all()) and torch.equal(a == 0, b == 0)
