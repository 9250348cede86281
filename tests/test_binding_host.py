"""Without the native host path -- not built, or built for another torch -- the linears take the general
path, with one warning; a build without it keeps the kernel library. No device is needed."""

from __future__ import annotations

import shutil
import warnings

import pytest
import torch

from llmopt.kernels import _lib, build, ops
from llmopt.quantization import QuantLinear, QuantLinearConfig


@pytest.fixture
def fresh(monkeypatch):
    monkeypatch.setattr(_lib, "_binding", None)
    monkeypatch.setattr(_lib, "_binding_tried", False)
    return monkeypatch


def _falls_back():
    module = QuantLinear(128, 64, QuantLinearConfig(4, 128, True, torch.bfloat16), bias=False)
    x = torch.zeros(1, 128, dtype=torch.bfloat16)
    with pytest.warns(RuntimeWarning, match="native host path"):
        assert _lib.load_binding() is None
    with warnings.catch_warnings():
        warnings.simplefilter("error")  # told once
        assert ops.module_linear(x, module, 64) is None


def test_missing(fresh, tmp_path):
    fresh.setattr(_lib, "binding_path", lambda: tmp_path / "_llmopt_torch.so")
    _falls_back()


def test_not_loadable(fresh, tmp_path):
    path = tmp_path / "_llmopt_torch.so"
    path.write_bytes(b"\x7fELF not a library")
    fresh.setattr(_lib, "binding_path", lambda: path)
    _falls_back()


def test_built_for_another_torch(fresh, tmp_path):
    # A copy under a path of its own: the module state of the loaded one stays as it is.
    path = tmp_path / "_llmopt_torch.so"
    shutil.copy(_lib.binding_path(), path)
    fresh.setattr(_lib, "binding_path", lambda: path)
    fresh.setattr(torch, "__version__", "0.1.0")
    _falls_back()


def test_loads_where_it_is_built(fresh):
    module = _lib.load_binding()
    assert module is not None and module.torch_version == torch.__version__.split("+")[0]
    assert _lib.load_binding() is module


def test_build_goes_on_without_it(monkeypatch, tmp_path, capsys):
    def fails(verbose=False):
        raise RuntimeError("g++ failed")

    old = tmp_path / "_llmopt_torch.so"
    old.write_bytes(b"an earlier build's")
    monkeypatch.setattr(build, "BINDING", old)
    monkeypatch.setattr(build, "build_binding", fails)
    assert build.build_binding_if_possible() is None
    assert not old.exists() and "left out" in capsys.readouterr().err
