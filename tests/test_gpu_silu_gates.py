"""silu(gate) * up: every bf16 gate against 64 bits, in order and shuffled (a gate beyond the range of the exponential, an infinity
or a NaN leaves its neighbours alone), and the tiles of 32 rows x 2 groups at their remainders."""
import pytest
import torch

import modular_amd as mx
from modular_amd.moe_kernels import silu_quantize

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("round_activation", [False, True])
@pytest.mark.parametrize("shuffled", [False, True])
def test_every_gate(dev, shuffled, round_activation):
    bits = torch.arange(65536, dtype=torch.int32)
    if shuffled:
        bits = bits[torch.randperm(65536, generator=torch.Generator().manual_seed(5))]
    gate = bits.to(torch.int16).view(torch.bfloat16).reshape(32, 2048)
    x = torch.cat([gate, torch.ones_like(gate)], dim=1).to(dev)
    got = mx.fused_silu(x, torch.tensor([0, 32], dtype=torch.int64).to(torch.uint32).to(dev), round_activation=round_activation).double().cpu()
    g = gate.double()
    want = g / (1.0 + torch.exp(-g))
    assert torch.equal(torch.isnan(got), torch.isnan(want))
    # the rounding to bf16, whose 8 bits are off by 2^-8 of the value at most (half of 2^-7, the step at a power of two), and some 30
    # steps of 2^-24 before it; exp(-gate) leaves float32's range below -88
    ok = (got - want).abs() <= want.abs() * (2.0 ** -8 + 30 * 2.0 ** -24) + 2.0 ** -120
    ok |= torch.isnan(want) | (got == want)
    assert bool(ok.all()), (g[~ok][:5], got[~ok][:5], want[~ok][:5])
    zero = g == 0
    assert torch.equal(torch.signbit(got[zero]), torch.signbit(g[zero]))


@pytest.mark.parametrize("rows,used,inter", [(1031, 1029, 1408), (4096, 4065, 128), (65, 64, 16640), (33, 1, 16512)])
@pytest.mark.parametrize("round_activation", [False, True])
def test_tiles_of_32_rows(dev, rows, used, inter, round_activation):
    """The bytes and scales of the product in bf16, quantised by the quantiser, and nothing past the rows in use."""
    cfg = mx.blockwise_fp8_config()
    x = torch.randn((rows, 2 * inter), generator=torch.Generator().manual_seed(rows)).to(torch.bfloat16).to(dev)
    off = torch.tensor([0, used], dtype=torch.int64).to(torch.uint32).to(dev)
    q, s = silu_quantize(x, off, 128, round_activation=round_activation)
    h = mx.fused_silu(x, off, round_activation=round_activation)
    # (the same rows one by one, as tiles of 16 rows x 1 group)
    for r in (0, used // 2, used - 1):
        one = mx.fused_silu(x[r:r + 1], torch.tensor([0, 1], dtype=torch.int64).to(torch.uint32).to(dev), round_activation=round_activation)
        assert torch.equal(one[0].view(torch.int16), h[r].view(torch.int16))
    want_q, want_s = mx.quantize_dynamic_scaled_float8(h[:used].contiguous(), cfg.input_scale, cfg.weight_scale, scales_type=torch.float32)
    assert torch.equal(q[:used].view(torch.uint8), want_q.view(torch.uint8)) and torch.equal(s[:, :used], want_s[:, :used])
