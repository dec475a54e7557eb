"""The sums of the kernel whose blocks split K among their waves, bit for bit with block scales: a wave folds its slabs in order, each product of a slab
times the two scales by one fused multiply-add, and the waves' sums are added in order -- however long its share of K is, and so whichever copy of the loop
a slab meets.  (The operands are small integers and the scales have 12 bits: a slab's product, the scales' and a sum before its rounding are exact in 64 bits.)"""
import numpy as np
import pytest
import torch

import modular_amd as mx
from mid_cases import SHAPES, exact_operands

pytestmark = pytest.mark.gpu
CFG = mx.blockwise_fp8_config()


def wanted(a, b, sa, sb, waves):
    (M, K), N = a.shape, b.shape[0]
    slabs = -(-K // 128)
    share = -(-slabs // waves)
    column_block = np.arange(N) // 128
    total = None
    for w in range(waves):
        acc = np.zeros((M, N), np.float32)
        for s in range(w * share, min((w + 1) * share, slabs)):
            k = slice(128 * s, 128 * (s + 1))
            scale = sa[s, :M, None] * sb[column_block, s][None, :]
            assert np.array_equal(scale.astype(np.float32), scale)
            acc = (acc + (a[:, k] @ b[:, k].T) * scale).astype(np.float32)
        total = acc if total is None else total + acc
    return total


@pytest.mark.parametrize("shape", SHAPES)
def test_order_and_rounding_of_the_sums(dev, tune, shape):
    blocks, mt, nt = shape // 100, shape // 10 % 10, shape % 10
    waves = 8 if blocks == 1 else 4
    tune(MAXFP8_MID=shape)
    M, N = 16 * mt + 2, 16 * nt * 9 + 4
    # shares of one to seven slabs, of which the last wave's is shorter
    for share in range(1, 8):
        K = 128 * (waves * share - (share > 1))
        a, b, g = exact_operands(M, N, K, 10 * shape + share)
        scale = lambda *size: 1.0 + torch.randint(0, 2048, size, generator=g).float() / 2048
        sa, sb = scale(K // 128, -(-M // 4) * 4), scale(-(-N // 128), K // 128)
        got = mx.dynamic_scaled_matmul(*[t.to(dev) for t in (a, b, sa, sb)], CFG.input_scale, CFG.weight_scale, out_type=torch.float32)
        want = wanted(*[t.double().numpy() for t in (a, b, sa, sb)], waves)
        assert np.array_equal(got.cpu().numpy(), want), f"shape {shape}, a share of {share} slabs: {np.count_nonzero(got.cpu().numpy() != want)} differ"
