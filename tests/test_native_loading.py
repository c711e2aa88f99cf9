"""Loading of the native bridge: what a call does while it is not loaded, what compiling
on demand builds, and the errors of a missing or unloadable module."""

from __future__ import annotations

import shutil

import pytest
import torch

from deformops_amd import _build
from deformops_amd.backends.eager.msda import forward as eager_forward
from deformops_amd.backends.hip import _lib, _native
from deformops_amd.backends.hip import msda as adapter
from deformops_amd.core.errors import (
    KernelBuildError,
    KernelNotProvidedError,
    KernelUnavailableError,
    NoBackendError,
)
from deformops_amd.registry import Backend, MSDAContext, msda
from deformops_amd.registry._dispatch import _Entry

BUILT = _native._PATH


@pytest.fixture
def absent(monkeypatch, tmp_path):
    """The path of a bridge that is not built, of a process that has loaded none."""
    monkeypatch.delenv("DEFORMOPS_COMPILE", raising=False)
    monkeypatch.setattr(_native, "_loaded", None)
    monkeypatch.setattr(_native, "_PATH", tmp_path / "_native.so")
    return tmp_path / "_native.so"


@pytest.fixture
def registered(monkeypatch):
    """The HIP adapter in the registry, as its module files it where there is a GPU."""
    msda.available()  # the adapters are imported
    entry = _Entry(adapter.msda_hip, lambda context: True, adapter.load, adapter.direct)
    monkeypatch.setitem(msda._entries, Backend.HIP, entry)
    monkeypatch.setattr(msda, "_chosen", {})


def operands():
    shapes, starts = torch.tensor([[4, 4], [2, 2]]), torch.tensor([0, 16])
    return torch.randn(1, 20, 2, 8), shapes, starts, torch.rand(1, 3, 2, 2, 4, 2), torch.rand(1, 3, 2, 8)


def test_cpu_calls_do_not_need_the_bridge(absent, registered):
    args = operands()
    for _ in range(2):
        torch.testing.assert_close(msda(*args), eager_forward(*args), rtol=0, atol=0)
    with pytest.raises(ValueError, match="value"):
        msda(args[0][0], *args[1:])


def test_a_gpu_call_without_the_bridge_is_the_policys_refusal(absent, registered):
    context = MSDAContext(torch.device("cuda"), 2, 2, 4, torch.float32, (9, 5), False, 3, head_dim=8)
    for _ in range(2):
        with pytest.raises(NoBackendError, match="not built"):
            msda._choose(context)
    assert adapter.direct(*operands(), softmax=False) is None
    with pytest.raises(KernelNotProvidedError, match="not built"):
        adapter.load()


@pytest.mark.parametrize("how", ["argument", "environment"])
def test_compiling_on_demand_builds_a_missing_bridge(absent, monkeypatch, how):
    assert _lib.library_path().exists()
    built = []

    def build_bridge(*, verbose=False):
        shutil.copy(BUILT, absent)
        built.append(absent)

    monkeypatch.setattr(_build, "build_bridge", build_bridge)
    with pytest.raises(KernelNotProvidedError):
        adapter.load(compile=False)
    if how == "environment":
        monkeypatch.setenv("DEFORMOPS_COMPILE", "1")
    assert adapter.load(compile=True if how == "argument" else None) == str(_lib.library_path())
    assert built == [absent] and _native.loaded() is _native.load()


def test_a_bridge_that_does_not_build_or_load_raises_the_documented_errors(absent, monkeypatch):
    def build_bridge(*, verbose=False):
        raise OSError("no compiler")

    monkeypatch.setattr(_build, "build_bridge", build_bridge)
    with pytest.raises(KernelBuildError, match="no compiler"):
        _native.load(compile=True)
    absent.write_bytes(b"not a shared object")
    with pytest.raises(KernelUnavailableError, match="cannot be loaded"):
        _native.load()
    assert _native.loaded() is None
