"""The matmul kernel for tens to a few hundred tokens (small tiles, K split over the block's waves): every tile shape forced on
ragged sizes, exact where the arithmetic is; the shape the estimates choose against the oracle on both sides of every edge; and
its fused QKV epilogue against the decode kernel's."""
import numpy as np
import pytest
import torch

import modular_amd as mx
import oracle
from modular_amd import _lib, synth
from mid_cases import SHAPES as BUILT, exact_case
from qkv_cases import make_cache_case, make_operands
from util import assert_rel, f32_np, fp8_bytes

pytestmark = pytest.mark.gpu
NT = oracle.default_threads()
CFG = {"block": mx.blockwise_fp8_config(), "row": mx.rowwise_fp8_config()}
SHAPES = [10 * mt + nt for mt in (2, 3, 4) for nt in (1, 2, 3, 4)]


def run(a, b, sa, sb, kind, dev, out_type, algo="auto"):
    return mx.dynamic_scaled_matmul(a.to(dev), b.to(dev), sa.to(dev), sb.to(dev), CFG[kind].input_scale, CFG[kind].weight_scale,
                                    out_type=out_type, algo=algo)


@pytest.mark.parametrize("kind", ["block", "row"])
@pytest.mark.parametrize("shape", SHAPES)
def test_every_tile_shape_is_exact(dev, tune, kind, shape):
    mt, nt = divmod(shape, 10)
    tune(MAXFP8_MID=shape)
    # one slab (three waves idle), slabs that do not divide by four, a K tail, ragged last tiles of rows and columns, N not
    # a multiple of 8, more tiles than the eight XCDs divide evenly
    for i, (M, N, K) in enumerate([(16 * mt, 16 * nt, 128), (16 * mt + 1, 16 * nt * 9 + 8, 640), (5, 16 * nt * 3 - 3, 1040),
                                   (3 * 16 * mt - 7, 16 * nt * 11, 2048)]):
        case = exact_case(M, N, K, kind, 100 * shape + i)
        for out_type in (torch.bfloat16, torch.float32):
            y, want = run(*case, kind, dev, out_type), run(*case, kind, dev, out_type, algo="naive")
            assert torch.equal(y, want), f"shape {shape}, {M} x {N} x {K}, {out_type}"


@pytest.mark.parametrize("kind", ["block", "row"])
@pytest.mark.parametrize("M,N,K", [(17, 10240, 2176), (33, 576, 7168), (64, 4096, 4096), (65, 4096, 4096), (117, 6144, 4096),
                                   (256, 1536, 7168), (320, 576, 7168)])
def test_chosen_shapes_against_the_oracle(dev, kind, M, N, K):
    assert "K split over the block's waves" in _lib.matmul_describe(M, N, K)
    a, b = synth.random_fp8((M, K), M), synth.random_fp8((N, K), N)
    if kind == "block":
        sa, sb = synth.random_scales((K // 128, -(-M // 4) * 4), 3), synth.random_scales((-(-N // 128), K // 128), 4)
    else:
        sa, sb = synth.random_scales((1, M), 3), synth.random_scales((N, 1), 4)
    y = run(a, b, sa, sb, kind, dev, torch.bfloat16)
    again = run(a, b, sa, sb, kind, dev, torch.bfloat16)
    assert torch.equal(y, again), "same bits from launch to launch"
    cols = np.r_[0:40, N // 2:N // 2 + 24, N - 40:N]
    if kind == "block":
        full = oracle.matmul_blockwise(fp8_bytes(a), fp8_bytes(b), sa.numpy(), sb.numpy(), gmnk=(1, 128, 128), threads=NT)
    else:
        full = oracle.matmul_rowwise(fp8_bytes(a), fp8_bytes(b), sa.numpy().reshape(-1), sb.numpy().reshape(-1), threads=NT)
    assert_rel(f32_np(y)[:, cols], full[:, cols], 1e-2, "mid")
    assert np.isfinite(f32_np(y)).all() and y.shape == (M, N)


@pytest.mark.parametrize("mnk", [(-1, -1, -1), (1, 1, -1), (1, 128, 128)])
@pytest.mark.parametrize("shape", BUILT)
@pytest.mark.parametrize("bias", [False, True])
def test_fused_qkv_epilogue_matches_the_decode_kernel(dev, tune, mnk, shape, bias):
    """Every built shape: Q and both caches, bit for bit, on exactly representable data: sequences that start inside a page, pages scattered
    over the pool, a row without a page."""
    lens, cached, page, heads, kv_heads, D = [3, 1, 20, 9], [5, 127, 0, 60], 16, 4, 2, 64
    T, K, q_dim = sum(lens), 768, heads * D
    N = q_dim + 2 * kv_heads * D
    ro, cl, lut = make_cache_case(lens, cached, page, 64, seed=1)
    lut[3, -1] = 64                                    # no block behind the last page of sequence 3
    a, w, sa, sb = make_operands(T, N, K, mnk, seed=2)
    g = torch.Generator().manual_seed(7)
    a = torch.randint(-2, 3, (T, K), generator=g).float().to(torch.float8_e4m3fn)
    w = torch.randint(-2, 3, (N, K), generator=g).float().to(torch.float8_e4m3fn)
    sa, sb = torch.exp2(torch.round(torch.log2(sa))), torch.exp2(torch.round(torch.log2(sb)))
    b = torch.randn(N, generator=g).to(torch.bfloat16).to(dev) if bias else None
    kv = mx.KVCacheParams(torch.bfloat16, kv_heads, D, num_layers=2, page_size=page)

    def once(algo):
        blocks = torch.full(kv.blocks_shape(64), 3.0, dtype=torch.bfloat16, device=dev)
        as_dev = lambda t: torch.from_numpy(t.astype(np.int64)).to(torch.uint32).to(dev)
        cache = mx.PagedCacheValues(blocks, as_dev(cl), as_dev(lut))
        q = mx.kernels._qkv_cache_matmul(kv, a.to(dev), as_dev(ro), w.to(dev), sa.to(dev), sb.to(dev), cache, 1, q_dim, mnk, b, algo)
        torch.cuda.synchronize()
        return q, blocks

    tune(MAXFP8_MID=shape)
    q, blocks = once("auto")
    want_q, want_blocks = once("skinny")
    assert torch.equal(q, want_q) and torch.equal(blocks, want_blocks)
