"""The native form of the package's calls against their Python form: the same bits for every form of
the arguments that it takes, and None (the Python form runs) for every other."""

import pytest
import torch

from mlx_tree_spec_amd import (QuantizedLinear, _lib, add_rms_norm_, gate_up_silu, install, quantized_matmul)
from mlx_tree_spec_amd.fused_ops import add_rms_norm_qmm_

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


class _Declines:
    """Stands in for the native module: every function declines, so the Python form runs."""

    def __getattr__(self, name):
        return lambda *args: None


def both(monkeypatch, call):
    got = call()
    with monkeypatch.context() as m:
        m.setattr(_lib, "native", lambda: _Declines())
        want = call()
    got, want = (got, want) if isinstance(got, tuple) else ((got,), (want,))
    assert len(got) == len(want)
    for a, b in zip(got, want):
        assert a.shape == b.shape and a.dtype == b.dtype and a.is_contiguous() and not a.requires_grad
        assert torch.equal(a.view(torch.int16), b.view(torch.int16))


def weights(n, k, bits=4, group=64, seed=0):
    g = torch.Generator(device=DEV).manual_seed(seed)
    w = torch.randint(-2**31, 2**31, (n, k * bits // 32), generator=g, device=DEV, dtype=torch.int64).to(torch.int32)
    s = (torch.randn(n, k // group, generator=g, device=DEV).abs() * 0.004 + 1e-4).bfloat16()
    b = (torch.randn(n, k // group, generator=g, device=DEV) * 1e-2).bfloat16()
    return w, s, b


def rows(*shape, seed=1):
    g = torch.Generator(device=DEV).manual_seed(seed)
    return torch.randn(*shape, generator=g, device=DEV).bfloat16()


@pytest.mark.parametrize("lead", [(), (1,), (5,), (2, 3), (1, 1, 7)])
def test_native_matches_python_form(monkeypatch, lead):
    w, s, b = weights(96, 256)
    x, r, nw = rows(*lead, 256), rows(*lead, 256, seed=2), rows(256, seed=3)
    both(monkeypatch, lambda: quantized_matmul(x, w, s, b))
    both(monkeypatch, lambda: quantized_matmul(x, w.view(torch.uint32), s, b))
    both(monkeypatch, lambda: gate_up_silu(x, w, s, b))
    both(monkeypatch, lambda: add_rms_norm_(x, r, torch.nn.Parameter(nw), 1e-6))
    for silu in (False, True):
        both(monkeypatch, lambda: add_rms_norm_qmm_(x, r, nw, 1e-6, w, s, b, silu_mul=silu))
    w8, s8, b8 = weights(33, 256, 8, 32)
    both(monkeypatch, lambda: quantized_matmul(x, w8, s8, b8, group_size=32, bits=8))


def test_native_declines_what_it_does_not_take(monkeypatch):
    w, s, b = weights(96, 256)
    wide = rows(6, 520)
    native = _lib.native()
    for x in (wide[:, :256], wide[:3, 4:260], rows(256, 6).T, wide.flatten()[1:1 + 3 * 256].view(3, 256)):
        assert native.qmm(x, w, s, b, 64, 4, False) is None and native.gate_up(x, w, s, b) is None
        both(monkeypatch, lambda: quantized_matmul(x, w, s, b))
        both(monkeypatch, lambda: add_rms_norm_(x, x, rows(256), 1e-6))
    x = rows(3, 256)
    for bad in (x.float(), x.cpu(), x[:0], x.as_subclass(type("Sub", (torch.Tensor,), {}))):
        assert native.qmm(bad, w, s, b, 64, 4, False) is None
    assert native.qmm(x, w, s[:, :3], b, 64, 4, False) is None and native.qmm(x, w.long(), s, b, 64, 4, False) is None
    assert native.norm(x, rows(2, 256), rows(256), 1e-6) is None and native.norm(x, x, rows(128), 1e-6) is None
    with pytest.raises(ValueError):
        quantized_matmul(x.float(), w, s, b)
    assert native.gate_up(x, *weights(48, 256)) is None  # gate and up halves of whole blocks
    assert native.qmm(x, *weights(40, 256), 64, 4, False) == _lib.QMM4_ERR_INVALID  # the library's own refusal


def test_native_linear_follows_replaced_buffers():
    mod = QuantizedLinear.from_quantized(*weights(64, 256))
    install(torch.nn.ModuleList([mod]), verbose=False)
    x = rows(4, 256)
    w2 = weights(64, 256, seed=9)
    assert torch.equal(mod(x), quantized_matmul(x, mod.weight, mod.scales, mod.biases))
    mod.weight, mod.scales, mod.biases = w2
    assert torch.equal(mod(x), quantized_matmul(x, *w2))
    mod.weight.data = weights(64, 256, seed=10)[0]
    assert torch.equal(mod(x), quantized_matmul(x, mod.weight, mod.scales, mod.biases))


def test_native_raises_under_a_transform_of_its_outputs():
    """Inside torch.func.grad new tensors are wrappers without storage: the calls raise, as their Python form does,
    with the interpreter's lock held."""
    w, s, b = weights(96, 256)
    mod = QuantizedLinear.from_quantized(w, s, b)
    install(torch.nn.ModuleList([mod]), verbose=False)
    x, nw, w8 = rows(3, 256), rows(256), weights(33, 256, 8, 32)
    calls = [lambda: quantized_matmul(x, w, s, b), lambda: quantized_matmul(x, *w8, group_size=32, bits=8),
             lambda: mod(x), lambda: gate_up_silu(x, w, s, b), lambda: add_rms_norm_(x, x, nw, 1e-6),
             lambda: add_rms_norm_qmm_(x, x, nw, 1e-6, w, s, b)]
    for call in calls:
        def inside(t):
            with pytest.raises(RuntimeError, match="storage"):
                call()
            return (t * t).sum()
        torch.func.grad(inside)(torch.ones(2, device=DEV))
        assert all(torch.isfinite(t.float()).all() for t in torch.utils._pytree.tree_leaves(call()))
