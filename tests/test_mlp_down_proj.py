"""The feed-forward block calls its `down_proj` wherever that is more than the scaled matmul of the block's own config."""
import pytest
import torch

import modular_amd as mx
from modular_amd import linear


class _Double(torch.nn.Module):
    def forward(self, x):
        return 2 * x[:, :256]


def _bias(mlp):
    mlp.down_proj.bias = torch.ones(256, dtype=torch.bfloat16)


def _hook(mlp):
    mlp.down_proj.register_forward_hook(lambda module, args, out: out + 1)


def _pre_hook(mlp):
    mlp.down_proj.register_forward_pre_hook(lambda module, args: (args[0] + 1,))


def _other_module(mlp):
    mlp.down_proj = _Double()


def _other_config(mlp):
    mlp.down_proj = mx.Linear(512, 256, mx.rowwise_fp8_config())


def _scales_elsewhere(mlp):
    mlp.down_proj.weight_scale = mlp.down_proj.weight_scale.to("meta")


def _plain(mlp):
    pass


def _stand_ins(monkeypatch):
    """On the CPU the kernels are stand-ins: what counts is which of them the block asks."""
    class Native:
        def mlp(self, x, *_):
            return torch.zeros((x.shape[0], 256), dtype=torch.bfloat16)

    asked = []
    monkeypatch.setattr(linear._lib, "native", Native)
    monkeypatch.setattr(linear, "fused_silu", lambda both, rows, round_activation: torch.ones_like(both[:, :512]))

    def quantized_matmul(x, weight, scale, input_scale, config):
        asked.append((tuple(weight.shape), config))
        return torch.zeros((x.shape[0], weight.shape[0]), dtype=torch.bfloat16)

    monkeypatch.setattr(linear, "quantized_matmul", quantized_matmul)
    return asked


@pytest.mark.parametrize("change, called", [(_plain, False), (_bias, True), (_hook, True), (_pre_hook, True), (_other_module, True),
                                            (_other_config, True), (_scales_elsewhere, True)])
def test_down_proj_is_called(monkeypatch, change, called):
    asked = _stand_ins(monkeypatch)
    mlp = mx.MLP(256, 512, mx.blockwise_fp8_config())
    change(mlp)
    y = mlp(torch.zeros((3, 256), dtype=torch.bfloat16))
    assert y.shape == (3, 256)
    assert [shape for shape, _ in asked][:1] == ([(1024, 256)] if called else [])
    if change in (_bias, _hook):
        assert (y == 1).all()
    if change is _other_module:
        assert (y == 2).all()
    if change is _other_config:
        assert asked[1] == ((256, 512), mlp.down_proj.quant_config)


@pytest.mark.parametrize("register", ["register_module_forward_hook", "register_module_forward_pre_hook"])
def test_hooks_of_every_module_see_down_proj(monkeypatch, register):
    _stand_ins(monkeypatch)
    mlp = mx.MLP(256, 512, mx.blockwise_fp8_config())
    seen = []
    handle = getattr(torch.nn.modules.module, register)(lambda module, *_: seen.append(module))
    try:
        mlp(torch.zeros((3, 256), dtype=torch.bfloat16))
    finally:
        handle.remove()
    assert mlp in seen and mlp.down_proj in seen
    seen.clear()
    mlp(torch.zeros((3, 256), dtype=torch.bfloat16))
    assert not seen
