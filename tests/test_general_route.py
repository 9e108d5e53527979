"""Which calls of the general path stay with its library product (CPU only): those whose product something
else sees. The general kernel would give autocast's result another type, leave no operation for a mode or a
tensor subclass to see, and no gradient or tangent of x."""

import contextlib

import pytest
import torch
from torch.autograd import forward_ad
from torch.overrides import TorchFunctionMode
from torch.utils._python_dispatch import TorchDispatchMode

from mlx_tree_spec_amd.qmm import _general_kernel_ok

M, N, K, BITS = 5, 33, 256, 8


def taken(x):
    return _general_kernel_ok(x, M, N, K, BITS)


def rows():
    return torch.zeros((M, K), dtype=torch.bfloat16)


class _FunctionMode(TorchFunctionMode):
    def __torch_function__(self, func, types, args=(), kwargs=None):
        return func(*args, **(kwargs or {}))


class _DispatchMode(TorchDispatchMode):
    def __torch_dispatch__(self, func, types, args=(), kwargs=None):
        return func(*args, **(kwargs or {}))


@contextlib.contextmanager
def _autocast(device, dtype):
    """torch.autocast's flags (it leaves a GPU's off where there is none)."""
    was = torch.is_autocast_enabled(device), torch.get_autocast_dtype(device)
    torch.set_autocast_enabled(device, True)
    torch.set_autocast_dtype(device, dtype)
    try:
        yield
    finally:
        torch.set_autocast_enabled(device, was[0])
        torch.set_autocast_dtype(device, was[1])


@contextlib.contextmanager
def _device_and_function_mode():
    with torch.device("cpu"), _FunctionMode():
        yield


@pytest.mark.parametrize("context,kernel", [
    (contextlib.nullcontext, True), (torch.no_grad, True), (torch.inference_mode, True),
    (lambda: _autocast("cuda", torch.bfloat16), True),   # the kernel's own result type
    (lambda: _autocast("cpu", torch.float16), True),
    (lambda: torch.device("cpu"), True),                 # a default device is a function mode too
    (lambda: _autocast("cuda", torch.float16), False), (lambda: _autocast("cuda", torch.float32), False),
    (_FunctionMode, False), (_device_and_function_mode, False), (_DispatchMode, False), (forward_ad.dual_level, False),
])
def test_modes(context, kernel):
    x = rows()
    with context():
        assert taken(x) is kernel
    assert taken(x)


def test_forms_of_x():
    assert taken(torch.nn.Parameter(rows(), requires_grad=False))
    assert not taken(rows().as_subclass(type("Sub", (torch.Tensor,), {})))
    x = rows().requires_grad_()
    assert not taken(x)
    with torch.no_grad():
        assert taken(x)
