"""The row-split kernel's activation staging and K-slice merge at 5-16 rows: x of at most 4 pieces of 16 bytes per
thread (one batch of 4) or more (batches of 10), and 1, 2, 4 and 8 K slices. test_plans.py checks that each
shape takes the slices that it names."""

import pytest
import torch

from mlx_tree_spec_amd import dequantize, gate_up_silu, quantized_matmul
from route_cases import ROWSPLIT_BATCH_CASES

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("m,k,n,fused,slices", ROWSPLIT_BATCH_CASES)
def test_rowsplit_batches(m, k, n, fused, slices):
    g = torch.Generator(device=DEV).manual_seed(m + k + n)
    x = torch.randn(m, k, generator=g, device=DEV).bfloat16()
    w = torch.randint(-2**31, 2**31, (n, k // 8), generator=g, device=DEV, dtype=torch.int64).to(torch.int32)
    s = (torch.randn(n, k // 64, generator=g, device=DEV).abs() * 0.004 + 1e-4).bfloat16()
    b = (-8 * s.float() + torch.randn(n, k // 64, generator=g, device=DEV) * 1e-3).bfloat16()
    call = gate_up_silu if fused else quantized_matmul
    y = call(x, w, s, b)
    wd = dequantize(w, s, b)
    rows = 1 << 15  # weight rows at a time in 64 bits
    ref, mag = [], []
    for i in range(0, n, rows):
        d = wd[i:i + rows].double()
        ref.append(x.double() @ d.T.contiguous())
        mag.append(x.double().abs() @ d.abs().T.contiguous())
    # fp32 sums of K terms in some order, then one bf16 rounding.
    ref, err = torch.cat(ref, 1), torch.cat(mag, 1) * (k * 2.0**-24)
    if not fused:
        bound = err + 2.0**-8 * ref.abs()
    else:
        # silu's relative change is at most 1 + |g| times its argument's; four more bf16 roundings.
        gate, up = ref.chunk(2, 1)
        ge, ue = err.chunk(2, 1)
        sig = torch.sigmoid(gate)
        ref = gate * sig * up
        bound = 2.0**-8 * (6 + gate.abs()) * ref.abs() + 1.2 * (ge * up.abs() + ue * (gate * sig).abs() + ge * ue) + 1e-30
    assert bool(((y.double() - ref).abs() <= bound).all())
    assert all(torch.equal(call(x, w, s, b), y) for _ in range(2))  # whichever slice arrives last
