"""silu(gate) * up with the quantisation behind it in one kernel: the bytes and scales of the two kernels it stands for, at the
edges of its vectors and row lengths, with rows beyond row_offsets[-1] left alone."""
import pytest
import torch

import modular_amd as mx
from modular_amd.moe_kernels import silu_quantize, silu_quantize_group

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,used,inter,per_row", [
    (1, 1, 128, False), (17, 17, 384, False), (300, 257, 1408, False), (9, 0, 256, False),
    (1, 1, 256, True), (5, 5, 4096, True), (33, 20, 4224, True), (3, 3, 8320, True), (2, 2, 16512, True), (2, 2, 32768, True)])
@pytest.mark.parametrize("round_activation", [False, True])
def test_same_bytes_as_the_two_kernels(dev, rows, used, inter, per_row, round_activation):
    cfg = mx.rowwise_fp8_config() if per_row else mx.blockwise_fp8_config()
    group = inter if per_row else 128
    assert silu_quantize_group(cfg, 128, inter) == group
    g = torch.Generator().manual_seed(rows + inter)
    x = torch.randn((rows, 2 * inter), generator=g) * torch.exp(2.0 * torch.randn((rows, 1), generator=g))
    x[0, :128] = 0                                     # a group (or part of a row) of zeros
    x = x.to(torch.bfloat16).to(dev)
    offsets = torch.tensor([0, used], dtype=torch.int64).to(torch.uint32).to(dev)
    q, s = silu_quantize(x, offsets, group, round_activation=round_activation)
    h = mx.fused_silu(x, offsets, round_activation=round_activation)
    want_q, want_s = mx.quantize_dynamic_scaled_float8(h, cfg.input_scale, cfg.weight_scale, scales_type=torch.float32)
    torch.cuda.synchronize()
    assert q.shape == want_q.shape and s.shape == want_s.shape
    assert torch.equal(q[:used].view(torch.uint8), want_q[:used].view(torch.uint8)) and torch.equal(s[:, :used], want_s[:, :used])


def test_rows_beyond_the_offsets_are_not_written(dev):
    x = torch.randn((8, 512), generator=torch.Generator().manual_seed(1)).to(torch.bfloat16).to(dev)
    lib = mx.kernels._lib.lib()
    for group in (128, 256):
        out, scales = torch.full((8, 256), 99, dtype=torch.uint8, device=dev), torch.full((2, 8), -1.0, device=dev)
        for used, past in ((3, 3), (1 << 30, 8)):     # (an offset beyond the buffers is held to their rows)
            off = torch.tensor([0, used], dtype=torch.int64).to(torch.uint32).to(dev)
            assert lib.maxfp8_silu_quantize_dynamic_scaled_fp8(out.data_ptr(), scales.data_ptr(), x.data_ptr(), off.data_ptr(), 2, 8, 256,
                                                               512, 256, group, 8, 0, 0, 1200.0, 0) == 0
            torch.cuda.synchronize()
            assert bool((out[past:] == 99).all()) and bool((scales[:2 if group == 128 else 1, past:] == -1).all())
            assert bool((scales[0, :past] != -1).all())
