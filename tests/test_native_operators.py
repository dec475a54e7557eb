"""The native operators' argument checks, without a GPU: what they cannot take is left to the Python wrappers or raises, and
never ends the process."""
import dataclasses
import os
import subprocess
import sys

import pytest
import torch
from torch._subclasses.fake_tensor import FakeTensorMode

import modular_amd as mx
from modular_amd import _lib, moe, quant_ops

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_tensor_without_memory_raises():
    """Inside torch.func.vmap a tensor has no memory to point to: asking for it is a C++ exception."""
    with FakeTensorMode():
        x = torch.empty((3, 4, 256), dtype=torch.bfloat16, device="cuda")
    native = _lib.native()
    for call in (lambda t: native.quantize(t, 128, True, 1200.0), lambda t: native.rms_norm_quantize(t, t[0], 1e-5, 0.0, 1200.0),
                 lambda t: native.linear(t, t, t, _lib.GRAN_BLOCK, 1200.0)):
        with pytest.raises(RuntimeError):
            torch.func.vmap(call)(x)


def test_cpu_tensors_are_left_to_the_wrappers():
    x = torch.zeros((4, 256), dtype=torch.bfloat16)
    assert _lib.native().quantize(x, 128, True, 1200.0) is None
    assert _lib.native().quantize(x.to_sparse(), 128, True, 1200.0) is None


STATIC_SCALES = """
import sys
import torch
torch._C._cuda_getCurrentRawStream = lambda index: 0   # (found by the module when it is loaded; nothing is launched)
from torch._subclasses.fake_tensor import FakeTensorMode
import modular_amd as mx
from modular_amd import _lib

native = _lib.native()
with FakeTensorMode():
    x = torch.empty((4, 256), dtype=torch.bfloat16, device="cuda")
    w = torch.empty((128, 256), dtype=torch.float8_e4m3fn, device="cuda")
    scale = torch.empty((), dtype=torch.float32) if sys.argv[1] == "fake" else torch.empty((), dtype=torch.float32, device="meta")
    assert native.linear_static(x, w, scale, scale) is None
    try:
        mx.quantize_static_scaled_float8(x, scale)
    except Exception as e:
        print("raised", type(e).__name__)
"""


@pytest.mark.parametrize("kind", ["fake", "meta"])
def test_static_scales_without_a_value(kind):
    """Scales of a traced program, or of a layer built on the meta device and not loaded yet: left to the wrapper, which raises.
    In a process of its own, because what goes wrong here ends it."""
    done = subprocess.run([sys.executable, "-c", STATIC_SCALES, kind], capture_output=True, text=True, cwd=ROOT)
    assert done.returncode == 0, done.stderr[-2000:]
    assert done.stdout.startswith("raised"), done.stdout


class Recorder:
    """In the place of the native module: every operator takes its operands and says what it was given."""

    def __init__(self):
        self.calls = []

    def __getattr__(self, name):
        def operator(*args):
            self.calls.append((name, args))
            return torch.zeros(1)
        return operator


def test_experts_with_scales_of_another_dtype_are_left_to_the_steps(monkeypatch):
    """A config of bfloat16 scales with float32 scale tensors: the steps quantise with bfloat16 scales and refuse to mix them."""
    native = Recorder()
    monkeypatch.setattr(moe._lib, "native", lambda: native)
    cfg = mx.blockwise_fp8_config()
    x, ids = torch.zeros((4, 128), dtype=torch.bfloat16), torch.zeros((4, 2), dtype=torch.int32)
    w, s = torch.zeros((3, 256, 128), dtype=torch.uint8).view(torch.float8_e4m3fn), torch.zeros((3, 2, 1))
    moe.expert_matmuls_fp8(x, ids, w, s, w, s, cfg)
    assert [name for name, _ in native.calls] == ["moe_experts"]
    native.calls.clear()
    cfg = dataclasses.replace(cfg, weight_scale=dataclasses.replace(cfg.weight_scale, dtype=torch.bfloat16))
    with pytest.raises(RuntimeError):  # (the steps, which run on the GPU only)
        moe.expert_matmuls_fp8(x, ids, w, s, w, s, cfg)
    assert "moe_experts" not in [name for name, _ in native.calls]


@pytest.mark.parametrize("layer", [1, 1.0, torch.tensor(1)])
def test_layer_index_of_another_type(monkeypatch, layer):
    """The fused QKV projection's layer is whatever int() takes, as in the wrapper behind the native operator."""
    native = Recorder()
    monkeypatch.setattr(quant_ops._lib, "native", lambda: native)
    kv = mx.KVCacheParams(torch.bfloat16, 1, 64, num_layers=2, page_size=16)
    u32 = torch.zeros(2, dtype=torch.int32)
    cache = mx.PagedCacheValues(torch.zeros(kv.blocks_shape(1), dtype=torch.bfloat16), u32[:1], u32[:1].reshape(1, 1))
    w, s = torch.zeros((384, 128), dtype=torch.uint8).view(torch.float8_e4m3fn), torch.zeros((3, 1))
    mx.quantized_fused_qkv_matmul(kv, torch.zeros((1, 128), dtype=torch.bfloat16), w, cache, layer, u32, 4, mx.blockwise_fp8_config(), s)
    (name, args), = native.calls
    assert name == "qkv_linear" and type(args[10]) is int and args[10] == 1


@pytest.mark.parametrize("path", ["LIB_PATH", "NATIVE_PATH"])
def test_argument_errors_come_before_a_missing_library(monkeypatch, path):
    """Without the built files the wrappers still say what is wrong with their operands; a call for the GPU says what is missing."""
    monkeypatch.setattr(_lib, "_native", None)
    monkeypatch.setattr(_lib, path, "/nowhere/lib.so")
    cfg = mx.blockwise_fp8_config()
    x = torch.zeros((4, 256), dtype=torch.bfloat16)
    with pytest.raises(ValueError, match="rank 2"):
        mx.quantize_dynamic_scaled_float8(x[0], cfg.input_scale, cfg.weight_scale, scales_type=torch.float32)
    with pytest.raises(RuntimeError, match="GPU only"):
        mx.quantize_dynamic_scaled_float8(x, cfg.input_scale, cfg.weight_scale, scales_type=torch.float32)
    with FakeTensorMode(), pytest.raises(_lib.LibraryMissing, match="/nowhere/lib.so"):
        mx.quantize_dynamic_scaled_float8(torch.empty((4, 256), dtype=torch.bfloat16, device="cuda"), cfg.input_scale, cfg.weight_scale,
                                          scales_type=torch.float32)
