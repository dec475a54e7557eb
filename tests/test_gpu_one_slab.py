"""The batched kernel for one slab of K: exact data against the oracle at the edges of its chunks of 16 to 64 tokens, of its walk over several chunks, of
its column groups, with strided operands between guard rows; and where it leaves the call to the other kernels."""
import numpy as np
import pytest
import torch

import modular_amd as mx
import oracle
from util import f32_np, fp8_bytes

pytestmark = pytest.mark.gpu
BLK = mx.blockwise_fp8_config()


# one chunk of every height, full and not; two chunks; 300 matrices, whose blocks (more than four per CU) walk 2 and 5 chunks;
# a wave without columns, two scale blocks of columns
@pytest.mark.parametrize("B,M,N", [(2, 1, 32), (2, 16, 64), (3, 17, 160), (2, 32, 96), (2, 33, 128), (2, 48, 512), (2, 49, 288), (3, 64, 32), (2, 65, 128),
                                   (300, 100, 512), (300, 257, 544), (1, 70, 64), (2, 70, 40)])
def test_exact(dev, B, M, N):
    g = torch.Generator().manual_seed(B + M + N)
    K, m_pad = 128, -(-M // 4) * 4
    a = torch.randint(-3, 4, (B, M, K), generator=g).float().to(torch.float8_e4m3fn)
    b = torch.randint(-3, 4, (B, N, K), generator=g).float().to(torch.float8_e4m3fn)
    sa = 2.0 ** torch.randint(-2, 3, (B, 1, m_pad), generator=g).float()
    sb = 2.0 ** torch.randint(-2, 3, (B, -(-N // 128), 1), generator=g).float()
    wide = torch.zeros((M, B, K + 128), dtype=torch.uint8, device=dev).view(torch.float8_e4m3fn)
    wide[:, :, :K] = a.transpose(0, 1).to(dev)
    out = torch.full((M + 2, B, N + 8), 7.0, dtype=torch.bfloat16, device=dev)
    y = mx.batched_dynamic_scaled_fp8_matmul(wide[:, :, :K].transpose(0, 1), b.to(dev), sa.to(dev), sb.to(dev), BLK.input_scale, BLK.weight_scale,
                                             out=out[1:M + 1, :, :N].transpose(0, 1))
    torch.cuda.synchronize()
    for i in {0, B // 2, B - 1}:
        want = oracle.matmul_blockwise(fp8_bytes(a[i]), fp8_bytes(b[i]), sa[i].numpy(), sb[i].numpy(), gmnk=(1, 128, 128), threads=oracle.default_threads())
        assert np.array_equal(f32_np(y[i]), torch.from_numpy(want).to(torch.bfloat16).float().numpy()), i
    tiles = mx.batched_dynamic_scaled_fp8_matmul(wide[:, :, :K].transpose(0, 1), b.to(dev), sa.to(dev), sb.to(dev), BLK.input_scale, BLK.weight_scale, algo="tiled")
    assert torch.equal(y.contiguous().view(torch.int16), tiles.view(torch.int16))     # (signs of zeros included)
    assert bool((out[0] == 7).all()) and bool((out[M + 1] == 7).all()) and bool((out[:, :, N:] == 7).all())


@pytest.mark.parametrize("M,K,stride", [(1, 128, 0), (33, 128, 64), (200, 384, 0), (65, 256, 128), (130, 128, 0)])
def test_quantiser_of_short_rows(dev, M, K, stride):
    """Rows of fewer than four groups: a thread's items are rows.  The oracle's bytes and scales, from strided heads."""
    x = torch.randn((M, 3, K + stride), generator=torch.Generator().manual_seed(M)).to(torch.bfloat16)
    x[0, :, :K] = 0
    q, s = mx.batched_quantize_dynamic_scaled_fp8(x.to(dev)[:, :, :K].transpose(0, 1), 128)
    for h in range(3):
        bits = x[:, h, :K].contiguous().view(torch.int16).numpy().view(np.uint16)
        want_q, want_s = oracle.quantize_dynamic_scaled_fp8(bits, 128)
        assert np.array_equal(q[h].cpu().view(torch.uint8).numpy(), want_q) and np.array_equal(s[h].cpu().numpy()[:, :M], want_s)


# (matrices, walkers and column blocks that do not divide by the XCDs; several chunks per walker, the last one's short)
@pytest.mark.parametrize("B,M,N", [(9, 3000, 160), (70, 500, 96), (5, 90, 1056), (7, 1, 32), (600, 65, 128)])
def test_walkers(dev, B, M, N):
    test_exact(dev, B, M, N)


@pytest.mark.parametrize("B,M,N", [(128, 1000, 512), (32, 2048, 1024), (128, 80, 512)])
def test_no_slower_than_the_tiles(dev, B, M, N):
    """Results of 131, 134 and 10 MB, four in turn: 28, 28 and 5.5 us; the tiles take 42, 40 and 8, and an earlier form of this kernel took 51, 50 and 9.5."""
    sets = [(torch.zeros((B, M, 128), dtype=torch.float8_e4m3fn, device=dev), torch.zeros((B, N, 128), dtype=torch.float8_e4m3fn, device=dev),
             torch.ones((B, 1, -(-M // 4) * 4), device=dev), torch.ones((B, -(-N // 128), 1), device=dev)) for _ in range(4)]
    outs = [torch.empty((B, M, N), dtype=torch.bfloat16, device=dev) for _ in sets]

    def milliseconds(algo):
        call = lambda: [mx.batched_dynamic_scaled_fp8_matmul(*s, BLK.input_scale, BLK.weight_scale, algo=algo, out=o) for s, o in zip(sets, outs)]
        call()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            call()
        times = []
        for _ in range(5):
            start, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            start.record()
            for _ in range(5):
                graph.replay()
            end.record()
            torch.cuda.synchronize()
            times.append(start.elapsed_time(end))
        return min(times)

    assert milliseconds("auto") < milliseconds("tiled")


# (rows form: a few rows of many matrices, a last block of few rows, two groups in blocks that are nearly full; groups form: blocks a fifth empty, three groups)
@pytest.mark.parametrize("B,M,K,rows", [(200, 50, 128, True), (3, 2753, 128, True), (5, 2001, 256, True), (130, 65, 256, False), (129, 66, 384, False), (16, 200, 128, False), (1, 1, 128, False)])
def test_quantiser_of_many_short_rows(dev, B, M, K, rows):
    from torch.profiler import ProfilerActivity, profile

    x = torch.randn((M, B, K + 64), generator=torch.Generator().manual_seed(M)).to(torch.bfloat16)
    x[M // 2, :, :K] = 0
    on = x.to(dev)[:, :, :K].transpose(0, 1)
    with profile(activities=[ProfilerActivity.CUDA]) as seen:
        q, s = mx.batched_quantize_dynamic_scaled_fp8(on, 128)
        torch.cuda.synchronize()
    names = [e.name for e in seen.events() if "quant_g128_bf16_kernel<" in e.name]
    assert [", true>" in n for n in names] == [rows], names
    for h in {0, B // 2, B - 1}:
        bits = x[:, h, :K].contiguous().view(torch.int16).numpy().view(np.uint16)
        want_q, want_s = oracle.quantize_dynamic_scaled_fp8(bits, 128)
        assert np.array_equal(q[h].cpu().view(torch.uint8).numpy(), want_q) and np.array_equal(s[h].cpu().numpy()[:, :M], want_s)
