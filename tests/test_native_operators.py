"""The native operators' argument checks, without a GPU: what they cannot take is left to the Python wrappers or raises, and
never ends the process."""
import os
import subprocess
import sys

import pytest
import torch
from torch._subclasses.fake_tensor import FakeTensorMode

from modular_amd import _lib

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
