"""The batched kernel for short K (latent attention in decode): equal to the oracle where the arithmetic is exact, equal to the
oracle's tolerance elsewhere, at the edges of its range -- one and four slabs, 1 / 16 / 17 / 32 tokens, one 32-column group and
a ragged last block of them, strided operands -- and on both sides of its rule."""
import numpy as np
import pytest
import torch

import modular_amd as mx
import oracle
from modular_amd import synth
from util import assert_rel, f32_np, fp8_bytes

pytestmark = pytest.mark.gpu
BLK = mx.blockwise_fp8_config()


def reference(a, b, sa, sb):
    return np.stack([oracle.matmul_blockwise(fp8_bytes(a[i]), fp8_bytes(b[i]), sa[i].numpy(), sb[i].numpy(), gmnk=(1, 128, 128),
                                             threads=oracle.default_threads()) for i in range(a.shape[0])])


@pytest.mark.parametrize("B,M,N,K", [(2, 1, 32, 128), (3, 16, 160, 128), (5, 17, 512, 128), (2, 32, 96, 256), (3, 20, 288, 384),
                                     (2, 17, 128, 512), (2, 31, 64, 512), (70, 5, 128, 512), (2, 33, 128, 128), (3, 12, 40, 128),
                                     (40, 20, 288, 384), (40, 17, 128, 512), (70, 31, 64, 512)])
@pytest.mark.parametrize("exact", [True, False])
def test_short_k_batches(dev, B, M, N, K, exact):
    g = torch.Generator().manual_seed(B + M + N + K)
    m_pad = -(-M // 4) * 4
    if exact:  # small integers and powers of two: every sum is exact in any order, and so is its bf16 rounding
        a = torch.randint(-3, 4, (B, M, K), generator=g).float().to(torch.float8_e4m3fn)
        b = torch.randint(-3, 4, (B, N, K), generator=g).float().to(torch.float8_e4m3fn)
        sa = 2.0 ** torch.randint(-2, 3, (B, K // 128, m_pad), generator=g).float()
        sb = 2.0 ** torch.randint(-2, 3, (B, -(-N // 128), K // 128), generator=g).float()
    else:
        a, b = synth.random_fp8((B, M, K), M), synth.random_fp8((B, N, K), N)
        sa, sb = synth.random_scales((B, K // 128, m_pad), 3), synth.random_scales((B, -(-N // 128), K // 128), 4)
    # activations and results as views of [token, batch, channel] buffers, between guard rows
    wide = torch.zeros((M, B, K + 128), dtype=torch.uint8, device=dev).view(torch.float8_e4m3fn)
    wide[:, :, :K] = a.transpose(0, 1).to(dev)
    out = torch.full((M + 2, B, N + 8), 7.0, dtype=torch.bfloat16, device=dev)
    view = out[1:M + 1, :, :N].transpose(0, 1)
    y = mx.batched_dynamic_scaled_fp8_matmul(wide[:, :, :K].transpose(0, 1), b.to(dev), sa.to(dev), sb.to(dev), BLK.input_scale,
                                             BLK.weight_scale, out=view)
    torch.cuda.synchronize()
    want = reference(a, b, sa, sb)
    if exact:
        assert np.array_equal(f32_np(y), torch.from_numpy(want).to(torch.bfloat16).float().numpy())
    else:
        assert_rel(f32_np(y).reshape(B * M, N), want.reshape(B * M, N), 1e-2, "short K")
    assert bool((out[0] == 7).all()) and bool((out[M + 1] == 7).all()) and bool((out[:, :, N:] == 7).all())


@pytest.mark.parametrize("B,M,N,K,decode", [(32, 48, 128, 512, True), (48, 48, 128, 512, False), (16, 33, 256, 256, True), (24, 64, 256, 256, False),
                                            (2, 64, 1024, 384, True), (32, 32, 128, 512, True), (48, 32, 128, 512, False)])
def test_decode_kernel_up_to_one_block_per_cu(dev, B, M, N, K, decode):
    """From two slabs on the decode kernel runs while its 16-row blocks are at most one per CU (more than 16 tokens).  Seen in the
    bits: it rounds a slab's scaled sum before it adds it, the others add in one fused step -- two float32 results in five differ,
    and of the 131072 and more bf16 ones of 32 tokens (whose kernel has no float32 form) half a dozen."""
    out_type = torch.float32 if M > 32 else torch.bfloat16
    a, b = synth.random_fp8((B, M, K), 1).to(dev), synth.random_fp8((B, N, K), 2).to(dev)
    sa, sb = synth.random_scales((B, K // 128, -(-M // 4) * 4), 3).to(dev), synth.random_scales((B, -(-N // 128), K // 128), 4).to(dev)
    run = lambda algo: mx.batched_dynamic_scaled_fp8_matmul(a, b, sa, sb, BLK.input_scale, BLK.weight_scale, out_type, algo=algo)
    assert torch.equal(run("auto"), run("skinny")) == decode
    if M > 32:
        assert torch.equal(run("auto"), run("tiled")) != decode
