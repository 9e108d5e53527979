"""Stream-K GEMM launches in units of 4 K steps: workgroup ranges that start and end in the middle of a
block of 8 scales, over 128 x 128 and 128 x 256 tiles, and with scales outside the fast form's range
(test_plans.py checks that the shapes take those units)."""

import pytest
import torch

from mlx_tree_spec_amd import dequantize, quantized_matmul
from route_cases import GEMM_HALF_UNIT_CASES

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("big_scale", [False, True])
@pytest.mark.parametrize("m,k,n", [case[:3] for case in GEMM_HALF_UNIT_CASES])
def test_half_unit_ranges(m, k, n, big_scale):
    g = torch.Generator(device=DEV).manual_seed(m + k + n)
    x = torch.randn(m, k, generator=g, device=DEV).bfloat16()
    w = torch.randint(-2**31, 2**31, (n, k // 8), generator=g, device=DEV, dtype=torch.int64).to(torch.int32)
    s = (torch.randn(n, k // 64, generator=g, device=DEV).abs() * 0.004 + 1e-4).bfloat16()
    if big_scale:  # |s| >= 2^104 takes the general dequantization; x is zero there, so the sums stay finite
        s[::7, 5::8] = 2.0**105
        x.view(m, k // 64, 64)[:, 5::8] = 0
    b = (-8 * s.float() + torch.randn(n, k // 64, generator=g, device=DEV) * 1e-3).bfloat16()
    y = quantized_matmul(x, w, s, b).double()
    wd = dequantize(w, s, b).double()
    ref = x.double() @ wd.T.contiguous()
    mag = x.double().abs() @ wd.abs().T.contiguous()
    # One bf16 rounding of the result, and K fp32 additions in some order.
    assert bool(((y - ref).abs() <= 2.0**-8 * ref.abs() + k * 2.0**-24 * mag).all())
    assert torch.equal(quantized_matmul(x, w, s, b).double(), y)
