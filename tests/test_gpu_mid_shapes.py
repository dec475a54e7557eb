"""Every built shape of the kernel whose blocks split K among their waves, by its tile and its blocks per CU: exact where the arithmetic is, on
ragged sizes, K tails, shares of K without a slab and grids of one, several and many blocks; and the heights and cuts the planner
takes for matmuls of little more than half a round of tiles."""
import re

import pytest
import torch

import modular_amd as mx
from modular_amd import _lib
from mid_cases import SHAPES, describe_of, exact_case, exact_operands, exact_scales

CFG = {"block": mx.blockwise_fp8_config(), "row": mx.rowwise_fp8_config()}


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["block", "row"])
@pytest.mark.parametrize("shape", SHAPES)
def test_every_built_shape_is_exact(dev, tune, kind, shape):
    blocks, mt, nt = shape // 100, shape // 10 % 10, shape % 10
    tune(MAXFP8_MID=shape)
    assert all(part in _lib.matmul_describe(20, 512, 512) for part in describe_of(shape))
    waves = 8 if blocks == 1 else 4
    # one slab; a slab more than the waves; a K tail; the longest share of a wave; several rounds of blocks; more tokens than the
    # choice by estimates takes below the tiles
    for i, (M, N, K) in enumerate([(16 * mt, 16 * nt, 128), (16 * mt + 1, 16 * nt * 9 + 8, 128 * (waves + 1)), (5, 16 * nt * 3 - 3, 1040),
                                   (17, 16 * nt, 64 * waves * 128 if waves == 4 else 32768), (3 * 16 * mt - 7, 16 * nt * 601, 256), (1030, 16 * nt * 2, 640)]):
        case = exact_case(M, N, K, kind, 100 * shape + i)
        on = [t.to(dev) for t in case]
        run = lambda algo: mx.dynamic_scaled_matmul(*on, CFG[kind].input_scale, CFG[kind].weight_scale, algo=algo)
        assert torch.equal(run("auto"), run("naive")), f"shape {shape}, {M} x {N} x {K}"


@pytest.fixture(scope="module")
def large(dev):
    """64 MB of weights and a few tokens: what the kernel reads past the caches; and the naive kernel's results"""
    M, N, K = 50, 262152, 256
    a, b, g = exact_operands(M, N, K, 5, dev)
    scales, want = {}, {}
    for kind in CFG:
        scales[kind] = exact_scales(M, N, K, kind, g, dev)
        want[kind] = mx.dynamic_scaled_matmul(a, b, *scales[kind], CFG[kind].input_scale, CFG[kind].weight_scale, algo="naive")
    return a, b, scales, want


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["block", "row"])
@pytest.mark.parametrize("shape", SHAPES)
def test_weights_that_are_read_once_are_exact(large, tune, kind, shape):
    """One row tile and 2^26 bytes of weights or more: the form with non-temporal loads.  The last column tile is ragged."""
    a, b, scales, want = large
    M = min(16 * (shape // 10 % 10) - 3, 50)
    assert b.numel() >= 1 << 26
    sa, sb = scales[kind]
    sa = sa[:, :-(-M // 4) * 4] if kind == "block" else sa[:, :M]
    tune(MAXFP8_MID=shape)
    y = mx.dynamic_scaled_matmul(a[:M], b, sa.contiguous(), sb, CFG[kind].input_scale, CFG[kind].weight_scale)
    assert torch.equal(y, want[kind][:M])


def test_heights_and_cuts_of_little_more_than_half_a_round():
    # one row tile of 192 instead of two of 128: 144 tiles on 256 CUs
    assert _lib.matmul_describe(166, 36864, 7168) == "192x256 x144 persistent, four waves"
    # two row tiles of 192 in four pieces instead of three of 128 in two; where 128-row tiles do not pay, K splits as before
    assert _lib.matmul_describe(338, 8192, 28672, False) == "192x256 x64 persistent, four waves, every tile cut in pieces of 56 slabs"
    assert "K split" in _lib.matmul_describe(164, 8192, 28672, False) and "K split 3" in _lib.matmul_describe(2048, 2304, 16384)
    # row scales: taller tiles whose row tiles share the weights, not 504 tiles of 128 x 128; where they fill too little of the chip, not
    assert _lib.matmul_describe(1072, 7168, 18432, False) == "160x256 x196 persistent, four waves"
    assert _lib.matmul_describe(1352, 5856, 15104, False) == "160x256 x207 persistent, four waves"
    assert "four waves" not in _lib.matmul_describe(776, 7168, 18432, False)
    assert _lib.matmul_describe(598, 12128, 10496, False) == "128x256 x240 persistent, four waves"
    # ... and cut tiles rather than whole ones of little more than half a round
    assert _lib.matmul_describe(600, 7168, 5120, False) == "160x256 x112 persistent, four waves, every tile cut in pieces of 20 slabs"
    # cut tiles against a short round of whole ones, with the workspace and without
    assert "every tile cut" in _lib.matmul_describe(1929, 1536, 7168) and "cut" not in _lib.matmul_describe(1929, 1536, 7168, True, False)


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["block", "row"])
def test_the_name_is_that_of_the_kernel_that_runs(dev, kind):
    from torch.profiler import ProfilerActivity, profile

    sizes = [(8, 4096, 4096), (16, 6144, 4096), (17, 1536, 7168), (18, 2048, 4880), (20, 4096, 4096), (28, 4096, 14336), (32, 28672, 4096),
             (48, 8192, 28672), (64, 4096, 4096), (64, 32768, 512), (117, 6144, 4096), (1500, 4096, 4096)]

    def call(M, N, K):
        a, b = (torch.ones(rows, K, device=dev).to(torch.float8_e4m3fn) for rows in (M, N))
        ones = lambda *shape: torch.ones(shape, device=dev)
        scales = (ones(-(-K // 128), -(-M // 4) * 4), ones(-(-N // 128), -(-K // 128))) if kind == "block" else (ones(1, M), ones(N, 1))
        mx.dynamic_scaled_matmul(a, b, *scales, CFG[kind].input_scale, CFG[kind].weight_scale)
    with profile(activities=[ProfilerActivity.CUDA]) as seen:
        for size in sizes:
            call(*size)
        torch.cuda.synchronize()
    ran = sorted((e.time_range.start, e.name) for e in seen.events() if "maxfp8::gemm_" in e.name)
    assert len(ran) == len(sizes)
    for (M, N, K), (_, name) in zip(sizes, ran):
        text = _lib.matmul_describe(M, N, K, kind == "block")
        small = [shape for shape in SHAPES if all(part in text for part in describe_of(shape))]
        if small:
            blocks, mt, nt = small[0] // 100, small[0] // 10 % 10, small[0] % 10
            assert re.search(rf"gemm_mid_kernel<{mt}, {nt}, \w+, \d+, {blocks}, ", name), (text, name)
        elif text == "skinny":
            assert "gemm_skinny_kernel" in name, (text, name)
        else:
            assert ("gemm_w4_kernel" if "four waves" in text else "gemm_tiled_kernel") in name, (text, name)
