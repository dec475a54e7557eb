"""Which kernel a fused QKV matmul runs on, by its tokens, scaling and size, read from a profile; and the same Q, K and V from each."""
import numpy as np
import pytest
import torch

import modular_amd as mx
from qkv_cases import make_cache_case

pytestmark = pytest.mark.gpu
HEAD, PAGE = 128, 128


def projection(dev, T, hidden, heads, kv_heads, mnk, seed):
    """a fused QKV matmul as a function of the algorithm, its caches filled anew by every call"""
    g = torch.Generator(device=dev).manual_seed(seed)
    N, q_dim = (heads + 2 * kv_heads) * HEAD, heads * HEAD
    ints = lambda rows: torch.randint(-2, 3, (rows, hidden), generator=g, device=dev).float().to(torch.float8_e4m3fn)
    a, w = ints(T), ints(N)
    power = lambda *shape: 2.0 ** torch.randint(-2, 1, shape, generator=g, device=dev).float()
    if mnk == (1, 128, 128):
        sa, sb = power(hidden // 128, -(-T // 4) * 4), power(N // 128, hidden // 128)
    else:
        sa, sb = power(1, T), power(N, 1)
    lens = [1] * T if T <= 64 else [T // 3, T - T // 3]
    ro, cl, lut = make_cache_case(lens, [7] * len(lens), PAGE, 200, seed=seed)
    kv = mx.KVCacheParams(torch.bfloat16, kv_heads, HEAD, num_layers=1, page_size=PAGE)
    as_dev = lambda t: torch.from_numpy(t.astype(np.int64)).to(torch.uint32).to(dev)
    ro, cl, lut = as_dev(ro), as_dev(cl), as_dev(lut)

    def run(algo="auto"):
        blocks = torch.zeros(kv.blocks_shape(200), dtype=torch.bfloat16, device=dev)
        q = mx.kernels._qkv_cache_matmul(kv, a, ro, w, sa, sb, mx.PagedCacheValues(blocks, cl, lut), 0, q_dim, mnk, None, algo)
        return q, blocks
    return run


# tokens, hidden size, heads, K / V heads, row scales: kernel
CASES = [(16, 4096, 32, 8, True, "gemm_skinny"), (18, 4096, 32, 8, True, "gemm_skinny"), (18, 4096, 32, 8, False, "gemm_mid"), (30, 2048, 32, 4, True, "gemm_skinny"),
         (24, 8192, 64, 8, True, "gemm_mid"), (33, 4096, 32, 8, True, "gemm_mid"), (200, 3584, 28, 4, True, "gemm_mid"), (491, 2048, 16, 4, True, "gemm_tiled"),
         # little more than half a round of four-wave tiles: not with K and V to store; with row scales from seven eighths of one on
         (526, 6144, 48, 8, True, "gemm_tiled"), (639, 5120, 40, 8, False, "gemm_tiled"), (939, 4096, 32, 8, True, "gemm_tiled"), (966, 5120, 40, 8, True, "gemm_w4")]


@pytest.mark.parametrize("T,hidden,heads,kv_heads,row,kernel", CASES)
def test_kernel_and_result(dev, T, hidden, heads, kv_heads, row, kernel):
    from torch.profiler import ProfilerActivity, profile

    run = projection(dev, T, hidden, heads, kv_heads, (1, 1, -1) if row else (1, 128, 128), seed=T)
    with profile(activities=[ProfilerActivity.CUDA]) as seen:
        q, blocks = run()
        torch.cuda.synchronize()
    ran = [e.name for e in seen.events() if "maxfp8::gemm_" in e.name]
    assert len(ran) == 1 and kernel in ran[0], ran
    # (small integers and powers of two: every sum is exact)
    want_q, want_blocks = run("tiled")
    assert torch.equal(q, want_q) and torch.equal(blocks, want_blocks)
