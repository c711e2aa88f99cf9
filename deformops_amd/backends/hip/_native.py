"""The native bridge of plain eager calls (csrc/bridge.cpp), loaded on first use.

``deformops_amd/lib/_native.so`` is a Python extension module built with the HIP
library (``python -m deformops_amd._build``); it calls that library's entry points at
the addresses the ctypes binding resolved. A missing module raises
:class:`~deformops_amd.core.errors.KernelNotProvidedError`; there is no fallback path.
"""

from __future__ import annotations

import ctypes
import importlib.machinery
import importlib.util
import threading
from pathlib import Path
from types import ModuleType

from ...core.errors import KernelNotProvidedError
from . import _lib

__all__ = ["load"]

_PATH = Path(__file__).resolve().parents[2] / "lib" / "_native.so"
_lock = threading.Lock()
_loaded: ModuleType | None = None


def load() -> ModuleType:
    """The extension module, bound to the loaded HIP library."""
    global _loaded  # noqa: PLW0603
    if _loaded is not None:
        return _loaded
    with _lock:
        if _loaded is not None:
            return _loaded
        library = _lib.load()
        if not _PATH.exists():
            msg = f"the native bridge {_PATH} is not built; run `python -m deformops_amd._build`"
            raise KernelNotProvidedError(msg)
        loader = importlib.machinery.ExtensionFileLoader("_native", str(_PATH))
        module = importlib.util.module_from_spec(importlib.util.spec_from_loader("_native", loader))
        loader.exec_module(module)
        entry_points = (library.cdll.msda_forward, library.cdll.msda_backward_workspace,
                        library.cdll.msda_backward_workspace_size, library.cdll.msda_last_error)
        module.init(*(ctypes.cast(f, ctypes.c_void_p).value for f in entry_points))
        _loaded = module
        return module
