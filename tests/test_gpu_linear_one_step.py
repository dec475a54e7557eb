"""The one-step operators (native module: quantisation and matmul, the feed-forward block, the experts, the fused QKV linear) give
the bits of the step-by-step wrappers, inside and outside the decode kernel's own quantisation, and leave to the wrappers
what they do not take."""
import os

import pytest
import torch

import modular_amd as mx
from modular_amd import _lib, synth

pytestmark = pytest.mark.gpu
CFG = {"block": mx.blockwise_fp8_config(), "row": mx.rowwise_fp8_config()}


def weight(N, K, kind, dev, seed):
    w = synth.weights_f32(N, K, seed=seed)
    q, s = synth.quantize_weight_block(w) if kind == "block" else synth.quantize_weight_rowwise(w)
    return q.to(dev), s.to(dev)


def steps(x, w, ws, kind):
    cfg = CFG[kind]
    q, s = mx.quantize_dynamic_scaled_float8(x, cfg.input_scale, cfg.weight_scale, scales_type=torch.float32)
    return mx.dynamic_scaled_matmul(q, w, s, ws, cfg.input_scale, cfg.weight_scale)


# (M, N, K): decode shapes with 16, 32 and 64 weight rows per block, one slab, fewer slabs than waves, a share that ends
# inside a 512-element load, the last token count that is quantised inside and the first that is not, larger ones
SHAPES = [(1, 16, 128), (1, 4096, 4096), (2, 250, 384), (3, 1000, 640), (4, 2048, 2048), (8, 2048, 2048), (9, 512, 1152), (1, 10240, 8192),
          (1, 28672, 4096), (2, 28672, 4096), (16, 4096, 512), (1, 24576, 1536), (117, 512, 1024), (300, 384, 256)]


@pytest.mark.parametrize("kind", ["block", "row"])
@pytest.mark.parametrize("M,N,K", SHAPES)
def test_linear_has_the_bits_of_its_steps(dev, kind, M, N, K):
    w, ws = weight(N, K, kind, dev, seed=N)
    wide = synth.activations(M, K + 64, seed=M, device=dev)
    wide[0, :128] = 0                                 # a group of zeros
    for x in (wide[:, :K], wide[:, :K].contiguous()):  # strided and packed rows
        done = _lib.native().linear(x, w, ws, _lib.GRAN_BLOCK if kind == "block" else _lib.GRAN_ROWWISE, 1200.0)
        assert torch.equal(done, steps(x, w, ws, kind)), f"{kind} {M} x {N} x {K}"
    assert torch.equal(mx.quantized_matmul(wide[:, :K], w, ws, None, CFG[kind]), done)


def test_the_quantisation_moves_into_the_decode_kernel_for_few_activations(dev):
    L = _lib.lib()
    for gran in (_lib.GRAN_BLOCK, _lib.GRAN_ROWWISE):
        assert L.maxfp8_linear_workspace_bytes(1, 4096, 4096, gran) == 0 < L.maxfp8_linear_workspace_bytes(16, 4096, 4096, gran)
    x, (w, ws) = synth.activations(1, 4096, seed=1, device=dev), weight(4096, 4096, "block", dev, 2)
    os.environ["MAXFP8_SKINNY_QUANT"] = "0"
    _lib.tuning_reload()
    try:
        assert L.maxfp8_linear_workspace_bytes(1, 4096, 4096, _lib.GRAN_BLOCK) > 0
        two = mx.quantized_matmul(x, w, ws, None, CFG["block"])
    finally:
        os.environ.pop("MAXFP8_SKINNY_QUANT")
        _lib.tuning_reload()
    assert torch.equal(two, mx.quantized_matmul(x, w, ws, None, CFG["block"]))


@pytest.mark.parametrize("M,N,K", [(1, 4096, 4096), (5, 300, 768), (64, 512, 1024), (700, 1024, 512)])
def test_static_linear_has_the_bits_of_its_steps(dev, M, N, K):
    x = synth.activations(M, K, seed=M, device=dev)
    w = synth.random_fp8((N, K), 3, std=0.5).to(dev)
    si, sw = torch.tensor(0.37), torch.tensor(0.011)
    done = _lib.native().linear_static(x, w, si, sw)
    want = mx.matmul_static_scaled_float8(mx.quantize_static_scaled_float8(x, si), w, si, sw)
    assert torch.equal(done, want)


@pytest.mark.parametrize("kind", ["block", "row"])
@pytest.mark.parametrize("M,H,F", [(1, 256, 512), (48, 512, 1024), (130, 256, 384)])
def test_mlp_has_the_bits_of_its_steps(dev, kind, M, H, F):
    layer = mx.MLP(H, F, CFG[kind], device=dev)
    for proj, n, k in ((layer.gate_proj, F, H), (layer.up_proj, F, H), (layer.down_proj, H, F)):
        w, ws = weight(n, k, kind, dev, seed=n + k)
        proj.weight.copy_(w)
        proj.weight_scale.copy_(ws)
    x = synth.activations(M, H, seed=4, device=dev)
    both = steps(x, layer.gate_up_weight, layer.gate_up_weight_scale, kind)
    h = mx.fused_silu(both, layer._all_rows(M, x.device), round_activation=True)
    assert torch.equal(layer(x), steps(h, layer.down_proj.weight, layer.down_proj.weight_scale, kind))
    assert torch.equal(layer(x.reshape(1, M, H)), layer(x).reshape(1, M, H))


def test_experts_have_the_bits_of_their_steps(dev):
    seq, k, E, H, F = 37, 3, 7, 256, 384
    cfg = CFG["block"]
    gu, sgu = (torch.stack(t) for t in zip(*[weight(2 * F, H, "block", dev, 10 + e) for e in range(E)]))
    d, sd = (torch.stack(t) for t in zip(*[weight(H, F, "block", dev, 50 + e) for e in range(E)]))
    x = synth.activations(seq, H, seed=5, device=dev)
    router = torch.randn((seq, E), generator=torch.Generator().manual_seed(6)).topk(k, dim=1).indices.to(dev)
    y = mx.expert_matmuls_fp8(x, router, gu, sgu, d, sd, cfg)
    assert torch.equal(y, mx.expert_matmuls_fp8(x, router.to(torch.int32), gu, sgu, d, sd, cfg, host_sync=False))
    order, start, restore, ids, stats = mx.moe_create_indices(router.reshape(-1).to(torch.int32), E)
    q, s = mx.quantize_dynamic_scaled_float8(x, cfg.input_scale, cfg.weight_scale, scales_type=torch.float32, row_index=order, index_div=k)
    mm = lambda q, s, w, ws, **kw: mx.grouped_dynamic_scaled_fp8_matmul(q, w, s, ws, start, ids, stats.cpu(), cfg.input_scale, cfg.weight_scale, **kw)
    h = mx.fused_silu(mm(q, s, gu, sgu), start)
    hq, hs = mx.quantize_dynamic_scaled_float8(h, cfg.input_scale, cfg.weight_scale, scales_type=torch.float32)
    assert torch.equal(y.reshape(seq * k, H), mm(hq, hs, d, sd, out_row_index=order))


# a few tokens, more sequences, more tokens; a projection whose tiles are cut along K (150 tokens fill its two row tiles badly, 200 well)
@pytest.mark.parametrize("kind", ["block", "row"])
@pytest.mark.parametrize("bias", [False, True])
@pytest.mark.parametrize("lens,shape", [([1], (4, 2, 64, 512)), ([1, 1, 1], (4, 2, 64, 512)), ([2, 30, 1, 40], (4, 2, 64, 512)),
                                        ([60, 1, 89], (32, 8, 128, 8192)), ([130, 70], (32, 8, 128, 8192))])
def test_qkv_linear_has_the_bits_of_its_steps(dev, kind, bias, lens, shape):
    heads, kv_heads, D, K = shape
    page, cached = 16, 9
    T, N = sum(lens), (heads + 2 * kv_heads) * D
    if T == 200:
        assert _lib.lib().maxfp8_fused_qkv_matmul_workspace_bytes(T, N, K, int(kind == "block")) > 0, "tiles cut along K"
    w, ws = weight(N, K, kind, dev, seed=1)
    x = synth.activations(T, K, seed=2, device=dev)
    kv = mx.KVCacheParams(torch.bfloat16, kv_heads, D, num_layers=2, page_size=page)
    pages = max(-(-(cached + n) // page) for n in lens)
    table = torch.randperm(len(lens) * pages, generator=torch.Generator().manual_seed(3)).to(torch.int32).reshape(len(lens), pages).to(dev)
    offsets = torch.tensor([0] + list(torch.tensor(lens).cumsum(0)), dtype=torch.int32, device=dev)
    b = torch.randn(N, generator=torch.Generator().manual_seed(4)).to(torch.bfloat16).to(dev) if bias else None
    cfg = CFG[kind]

    def cache():
        return mx.PagedCacheValues(torch.full(kv.blocks_shape(len(lens) * pages), 2.0, dtype=torch.bfloat16, device=dev),
                                   torch.full((len(lens),), cached, dtype=torch.int32, device=dev), table)
    one, two = cache(), cache()
    q = mx.quantized_fused_qkv_matmul(kv, x, w, one, 1, offsets, heads, cfg, ws, bias=b)
    xq, xs = mx.quantize_dynamic_scaled_float8(x, cfg.input_scale, cfg.weight_scale, scales_type=torch.float32)
    want = mx.fused_qkv_ragged_matmul_scaled_float8(kv, xq, offsets, w, two, 1, heads, xs, ws, bias=b, quant_config=cfg)
    assert torch.equal(q, want) and torch.equal(one.kv_blocks, two.kv_blocks)
    # an operand that the native operator leaves to the wrapper: channels that are not contiguous
    three = cache()
    q = mx.quantized_fused_qkv_matmul(kv, x.t().contiguous().t(), w, three, 1, offsets, heads, cfg, ws, bias=b)
    assert torch.equal(q, want) and torch.equal(three.kv_blocks, two.kv_blocks)


def test_what_the_native_operators_leave_to_the_wrappers(dev):
    n = _lib.native()
    x, (w, ws) = synth.activations(4, 256, seed=1, device=dev), weight(128, 256, "block", dev, 2)
    assert n.linear(x.float(), w, ws, _lib.GRAN_BLOCK, 1200.0) is None                # another dtype
    assert n.linear(x[:, 1:], w[:, 1:], ws, _lib.GRAN_BLOCK, 1200.0) is None          # rows that are not 16-byte aligned
    assert n.linear(x.t().contiguous().t(), w, ws, _lib.GRAN_BLOCK, 1200.0) is None   # channels that are not contiguous
    assert n.linear(x[:0], w, ws, _lib.GRAN_BLOCK, 1200.0) is None                    # nothing to do
    assert n.linear(x, w.cpu(), ws, _lib.GRAN_BLOCK, 1200.0) is None                  # another device
    assert n.linear(x, w, ws[:, :1], _lib.GRAN_BLOCK, 1200.0) is None                 # scales that do not fit
    assert n.linear(x, None, ws, _lib.GRAN_BLOCK, 1200.0) is None
    with pytest.raises(ValueError):
        mx.quantized_matmul(x, w[:, :128].contiguous(), ws, None, CFG["block"])
    with pytest.raises(TypeError):
        n.linear(x, w)
    assert mx.quantized_matmul(x[:0], w, ws, None, CFG["block"]).shape == (0, 128)
    y = mx.quantized_matmul(x.t().contiguous().t(), w, ws, None, CFG["block"])
    assert torch.equal(y, mx.quantized_matmul(x, w, ws, None, CFG["block"]))
