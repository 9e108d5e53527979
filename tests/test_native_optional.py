"""The package without its native call path (CPU only): where the extension is absent or made for another
torch, native() warns once and hands out functions that decline, so every call takes its Python form;
where it cannot be built, build() still leaves the kernel library and warns."""

import os
import sys
import types
import warnings

import pytest

from mlx_tree_spec_amd import _lib, build

NAMES = ("qmm", "linear", "gate_up", "norm", "norm_qmm")


def _bind(*args):
    raise AssertionError("an extension of another torch must not be called")


@pytest.mark.parametrize("found", [None, types.SimpleNamespace(TORCH_VERSION="1.0", bind=_bind),
                                   types.SimpleNamespace(bind=_bind)])
def test_native_declines_where_it_cannot_be_loaded(monkeypatch, found):
    if not os.path.exists(_lib.LIB_PATH):
        pytest.skip("libqmm4.so is not built (run __graft_entry__.build())")
    monkeypatch.setattr(_lib, "_native", None)
    monkeypatch.setitem(sys.modules, "mlx_tree_spec_amd._native", found)  # None: not there
    with pytest.warns(RuntimeWarning, match="native call path"):
        native = _lib.native()
    assert all(getattr(native, name)("any", "arguments", 3) is None for name in NAMES)
    with warnings.catch_warnings():
        warnings.simplefilter("error")  # the second call does not warn again
        assert _lib.native() is native


def test_build_without_the_extension_keeps_the_library(monkeypatch, tmp_path):
    stale = tmp_path / "_native.so"
    stale.write_bytes(b"of earlier sources")
    linked = []

    def no_headers(out):
        raise RuntimeError("Python.h: No such file or directory")

    monkeypatch.setattr(build, "NATIVE_PATH", str(stale))
    monkeypatch.setattr(build, "_build_native", no_headers)
    monkeypatch.setattr(build, "_link", lambda srcs, out: linked.append(out))
    with pytest.warns(RuntimeWarning, match="could not be built"):
        assert build.build() == build.LIB_PATH
    assert linked == [build.LIB_PATH, build.FLOOR_PATH] and not stale.exists()
