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


# ---- bit for bit ---------------------------------------------------------------------------------------------------------------------
# A lane computes eight outputs, all of them by expf and the IEEE division where one of its gates is beyond the range of the short form: so the same gate, at the
# same place, with and without such a neighbour, is that form beside the reference.
def every_finite_gate():
    bits = torch.arange(65536, dtype=torch.int32)
    gate = bits.to(torch.int16).view(torch.bfloat16)
    return gate[gate.float().abs() < 86]


@pytest.mark.parametrize("round_activation", [False, True])
def test_every_gate_has_the_bits_of_the_division(dev, round_activation):
    gates = every_finite_gate()
    n = gates.numel()
    got = []
    for neighbour in (0.0, 100.0):
        x = torch.full((-(-n // 16), 16, 8), neighbour, dtype=torch.bfloat16)
        x.view(-1, 8)[:n, 3] = gates
        x = x.reshape(x.shape[0], 128)
        rows = torch.tensor([0, x.shape[0]], dtype=torch.int64).to(torch.uint32).to(dev)
        y = mx.fused_silu(torch.cat([x, torch.ones_like(x)], dim=1).to(dev), rows, round_activation=round_activation)
        got.append(y.cpu().reshape(-1, 8)[:n, 3].view(torch.int16))
    assert torch.equal(*got)


# (a power of two shows the float32 activation by the scale, largest value / 448, up to two neighbours that round alike; three more factors part those)
@pytest.mark.parametrize("mantissa", [1.0, 1.25, 1.5, 1.75])
def test_every_gate_has_the_float32_of_the_division(dev, mantissa):
    gates = every_finite_gate()
    n, cfg = gates.numel(), mx.blockwise_fp8_config()
    g = gates.double()
    size = (g / (1.0 + torch.exp(-g))).abs()
    up = (mantissa * 2.0 ** torch.where(size > 0, -torch.floor(torch.log2(size)), torch.zeros_like(size)).clamp(-120, 120)).to(torch.bfloat16)
    place = torch.arange(n) % 128
    scales, codes = [], []
    for neighbour in (0.0, 100.0):                       # (times 0: the group's largest value is the gate's)
        x, u = torch.zeros((n, 128), dtype=torch.bfloat16), torch.zeros((n, 128), dtype=torch.bfloat16)
        x[torch.arange(n), place ^ 1] = neighbour
        x[torch.arange(n), place], u[torch.arange(n), place] = gates, up
        rows = torch.tensor([0, n], dtype=torch.int64).to(torch.uint32).to(dev)
        q, s = mx.fused_silu_quantized(torch.cat([x, u], dim=1).to(dev), rows, cfg)
        scales.append(s.cpu()[0].view(torch.int32))
        codes.append(q.cpu().view(torch.uint8)[torch.arange(n), place])
    assert torch.equal(*scales) and torch.equal(*codes)
    shown = size * up.double() >= 1e-4
    assert shown.sum() > 30000 and bool(((scales[0].view(torch.float32).double() * 448 - size * up.double()).abs() <= 2.0 ** -20 * size * up.double())[shown].all())
