"""Which calls of the general path stay with its library product (CPU only): the sizes at which it is the faster
form, and calls whose product something else sees. The general kernel would give autocast's result another type, leave no operation for a mode or a
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


# Sizes at either side of the rule's lines, with the form that was measured as the faster one (us of the
# kernel / the library product, 4-bit groups of 64).
@pytest.mark.parametrize("m,k,n,kernel", [
    (32, 256, 151937, True),     # 30 / 48
    (33, 256, 151937, False),    # 62 / 52 (groups of 32)
    (33, 64, 65537, True),       # 23 / 37
    (64, 1024, 65537, True), (65, 1024, 65537, False),
    (128, 5120, 17409, True), (129, 5120, 17409, False), (256, 5120, 17409, False),  # 77 / 95, 103 / 109, 135 / 121
    (256, 8192, 8191, True),     # 88 / 111
    (160, 4096, 11009, False), (192, 512, 16385, True),
    (256, 64, 65537, False),     # 85 / 38
    (512, 1024, 513, True), (2048, 256, 2047, True), (400, 320, 16001, False), (300, 64, 65537, False),
    (4096, 128, 4095, False),    # 88 / 42
    (524288, 64, 3, False),      # 80 / 38
    (320, 17408, 513, False),    # past 256 rows only small products
])
def test_sizes(m, k, n, kernel):
    x = torch.empty((1, 1), dtype=torch.bfloat16).expand(m, k)
    assert _general_kernel_ok(x, m, n, k, 4) is kernel
