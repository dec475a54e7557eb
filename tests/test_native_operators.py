"""The native operators' argument checks, without a GPU: what they cannot take is left to the Python wrappers or raises, and
never ends the process."""
import pytest
import torch
from torch._subclasses.fake_tensor import FakeTensorMode

from modular_amd import _lib


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
