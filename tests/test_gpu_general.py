"""The general quantized matmul kernel at its edges: rows around its 16/32/64-row blocks, columns around
its 16- and 32-column blocks, K of fewer units (64 k) than the 8 waves that split it, slices that
start inside a group of 128, and more than one scale segment (8 units) per wave."""

import numpy as np
import pytest
import torch
from torch.utils.flop_counter import FlopCounterMode

from mlx_tree_spec_amd import dequantize, quantized_matmul
from mlx_tree_spec_amd.qmm import _general_kernel_ok
from oracle import qmm4_oracle as O

pytestmark = pytest.mark.gpu

CASES = [  # m, k, n, bits, group
    (1, 64, 1, 8, 32), (15, 128, 15, 4, 128), (16, 192, 17, 2, 64), (17, 256, 33, 4, 32), (32, 704, 31, 8, 64),
    (33, 640, 47, 2, 32), (64, 1152, 16, 8, 128), (65, 4672, 5, 8, 32), (100, 5120, 49, 4, 64), (257, 896, 63, 2, 128),
    (7, 1024, 8193, 4, 32), (24, 512, 8200, 8, 64),
]


def _inputs(m, k, n, bits, group, seed):
    rng = np.random.default_rng(seed)
    x = O.f32_to_bf16_bits(rng.standard_normal((m, k)).astype(np.float32))
    w = rng.integers(0, 2**32, size=(n, k * bits // 32), dtype=np.uint32)
    s = O.f32_to_bf16_bits((np.abs(rng.standard_normal((n, k // group))) * 0.004 + 1e-4).astype(np.float32))
    b = O.f32_to_bf16_bits((-(2.0 ** (bits - 1)) * O.bf16_bits_to_f32(s)
                            + rng.standard_normal((n, k // group)) * 1e-3).astype(np.float32))
    return x, w, s, b


def _dev(a, dt):
    return torch.from_numpy(np.ascontiguousarray(a).view(dt)).cuda()


@pytest.mark.parametrize("m,k,n,bits,group", CASES)
def test_general_kernel_edges(m, k, n, bits, group):
    x, w, s, b = _inputs(m, k, n, bits, group, seed=m + k + n)
    xd, wd = _dev(x, np.int16).view(torch.bfloat16), _dev(w, np.int32)
    sd, bd = _dev(s, np.int16).view(torch.bfloat16), _dev(b, np.int16).view(torch.bfloat16)
    assert _general_kernel_ok(xd, m, n, k, bits)
    y = quantized_matmul(xd, wd, sd, bd, group_size=group, bits=bits).float().cpu().numpy().astype(np.float64)
    xf = O.bf16_bits_to_f32(x).astype(np.float64)
    wf = O.bf16_bits_to_f32(O.dequantize(w, s, b, group, bits)).astype(np.float64)
    ref = xf @ wf.T
    # One bf16 rounding of the result, and K fp32 additions in some order (each within 2^-24 of the sum
    # of magnitudes).
    bound = 2.0**-8 * np.abs(ref) + k * 2.0**-24 * (np.abs(xf) @ np.abs(wf).T)
    assert np.all(np.abs(y - ref) <= bound), float(np.max(np.abs(y - ref) / bound))


def test_general_path_keeps_the_gradient_of_x():
    """x that asks for a gradient takes the dequantize + library form, which is differentiable in x."""
    x, w, s, b = _inputs(5, 256, 33, 8, 64, seed=3)
    xd = _dev(x, np.int16).view(torch.bfloat16).requires_grad_()
    wd = _dev(w, np.int32)
    sd, bd = _dev(s, np.int16).view(torch.bfloat16), _dev(b, np.int16).view(torch.bfloat16)
    y = quantized_matmul(xd, wd, sd, bd, group_size=64, bits=8)
    y.backward(torch.ones_like(y))
    wf = dequantize(wd, sd, bd, group_size=64, bits=8).float()
    want = wf.sum(0).expand(5, -1)
    # Sums of 33 bf16 weights rounded to bf16.
    assert torch.allclose(xd.grad.float(), want, rtol=2.0**-7, atol=1e-3)


def test_general_path_shows_its_product_to_modes():
    """Autocast to another type, function and dispatch modes and forward-mode derivatives see the general path's
    product, in the native form of the call and behind it."""
    x, w, s, b = _inputs(5, 256, 33, 8, 32, seed=4)
    xd, wd = _dev(x, np.int16).view(torch.bfloat16), _dev(w, np.int32)
    sd, bd = _dev(s, np.int16).view(torch.bfloat16), _dev(b, np.int16).view(torch.bfloat16)
    call = lambda t: quantized_matmul(t, wd, sd, bd, group_size=32, bits=8)  # noqa: E731
    wf = dequantize(wd, sd, bd, group_size=32, bits=8)
    want = xd.float() @ wf.float().T.contiguous()
    for dtype in (torch.float16, torch.float32, torch.bfloat16):
        with torch.autocast("cuda", dtype):
            y = call(xd)
        assert y.dtype == dtype and torch.allclose(y.float(), want, rtol=2.0**-7, atol=2.0**-7 * want.abs().max())
    seen = []

    class Functions(torch.overrides.TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            seen.append(func)
            return func(*args, **(kwargs or {}))

    with Functions():
        call(xd)
    assert torch.nn.functional.linear in seen
    with FlopCounterMode(display=False) as flops:
        call(xd)
    assert flops.get_total_flops() == 2 * 5 * 256 * 33
    sub = type("Sub", (torch.Tensor,), {})
    assert type(call(xd.as_subclass(sub))) is sub
    with torch.autograd.forward_ad.dual_level():
        dual = torch.autograd.forward_ad.make_dual(xd, torch.ones_like(xd))
        tangent = torch.autograd.forward_ad.unpack_dual(call(dual)).tangent
    # Sums of 256 bf16 weights rounded to bf16.
    assert torch.allclose(tangent.float(), wf.float().sum(1).expand(5, -1), rtol=2.0**-7, atol=1e-3)
