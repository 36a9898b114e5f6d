"""Host side of the native binding, without a GPU: what the module hands to it, and what happens where it is
missing, cannot be built, or was built for another torch."""

import importlib.util
import os
import sys
import types
import warnings

import pytest
import torch

from helpers import ROOT
from dynconv import _capi
from dynconv.modules import GroupedLowRankDynamicShortConvolution


@pytest.mark.parametrize("head_dim", [None, 32, 32.0])
def test_module_head_dim(head_dim, monkeypatch):
    """A head dim that is a whole float reaches the binding as the int that the Python path makes of it."""
    seen = []
    fake = types.SimpleNamespace(grouped_module=lambda *a: seen.append(a[-1]) or "ys")
    monkeypatch.setattr(_capi, "binding", fake)
    m = GroupedLowRankDynamicShortConvolution(64, 7, 4, groups=2, head_dim=head_dim)
    assert m(torch.zeros(1, 3, 128), torch.zeros(1, 3, 64)) == "ys"
    assert seen == [None if head_dim is None else 32] and not isinstance(seen[0], float)


def _build_module():
    spec = importlib.util.spec_from_file_location("dynconv_build", os.path.join(ROOT, "dynamic-conv1d_amd", "build.py"))
    mod = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(mod)
    return mod


def test_build_goes_on_without_a_host_compiler(tmp_path, monkeypatch, capsys):
    b = _build_module()
    old = tmp_path / "_binding.so"
    old.write_bytes(b"")
    monkeypatch.setattr(b, "BINDING_OUT", str(old))
    monkeypatch.setenv("CXX", str(tmp_path / "no-such-compiler"))
    assert b.build_binding() is None
    assert not old.exists(), "a binding of an earlier build stays behind"
    assert "skipped (no C++ compiler" in capsys.readouterr().out
    monkeypatch.delenv("CXX")
    monkeypatch.setenv("ROCM_PATH", str(tmp_path))
    assert b.build_binding() is None


def test_a_source_that_does_not_compile_fails_the_build(tmp_path, monkeypatch):
    b = _build_module()
    src = tmp_path / "torch_binding.cpp"
    src.write_text("int f( {\n")
    monkeypatch.setattr(b, "BINDING_SRC", str(src))
    monkeypatch.setattr(b, "BINDING_OUT", str(tmp_path / "_binding.so"))
    with pytest.raises(RuntimeError, match="torch_binding.cpp failed"):
        b.build_binding(verbose=False)


def _load_with(monkeypatch, module):
    import dynconv

    monkeypatch.setitem(sys.modules, "dynconv._binding", module)
    monkeypatch.setattr(dynconv, "_binding", module, raising=False)
    return _capi._load_binding(_capi.LIB_PATH)


def test_binding_for_another_torch_warns(monkeypatch):
    calls = []
    fake = types.ModuleType("dynconv._binding")
    fake.torch_version, fake.init = "0.0.0", calls.append
    with pytest.warns(UserWarning, match="built for torch 0.0.0"):
        assert _load_with(monkeypatch, fake) is None
    fake.torch_version = torch.__version__
    with warnings.catch_warnings():
        warnings.simplefilter("error")
        assert _load_with(monkeypatch, fake) is fake
    assert calls == [_capi.LIB_PATH]
