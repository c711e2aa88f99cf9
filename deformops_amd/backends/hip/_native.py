"""The native bridge of plain eager calls (csrc/bridge.cpp), loaded on first use.

``deformops_amd/lib/_native.so`` is a Python extension module built with the HIP
library (``python -m deformops_amd._build``); it calls that library's entry points at
the addresses the ctypes binding resolved. A missing module raises
:class:`~deformops_amd.core.errors.KernelNotProvidedError` (or is built first when the
caller allows compiling); there is no fallback path.
"""

from __future__ import annotations

import ctypes
import importlib.machinery
import importlib.util
import threading
from pathlib import Path
from types import ModuleType

from ...core.errors import KernelBuildError, KernelNotProvidedError, KernelUnavailableError
from . import _lib

__all__ = ["load", "loaded"]

_PATH = Path(__file__).resolve().parents[2] / "lib" / "_native.so"
_lock = threading.Lock()
_loaded: ModuleType | None = None


def loaded() -> ModuleType | None:
    """The extension module if :func:`load` has loaded it already."""
    return _loaded


def load(*, download: bool | None = None, compile: bool | str | None = None) -> ModuleType:  # noqa: A002
    """The extension module, bound to the loaded HIP library. With ``compile`` truthy
    (``None``: with ``DEFORMOPS_COMPILE`` set) whichever of the two is missing is built.

    Raises
    ------
    KernelNotProvidedError
        If the module or the library is missing and compiling was not allowed.
    KernelBuildError
        If compiling was allowed and failed.
    KernelUnavailableError
        If the module is there and cannot be loaded.
    """
    global _loaded  # noqa: PLW0603
    if _loaded is not None:
        return _loaded
    with _lock:
        if _loaded is not None:
            return _loaded
        library = _lib.load(download=download, compile=compile)
        if not _PATH.exists():
            if not _lib.compile_allowed(compile):
                msg = (
                    f"the native bridge {_PATH} is not built; run "
                    f"`python -m deformops_amd._build` (or set DEFORMOPS_COMPILE=1)"
                )
                raise KernelNotProvidedError(msg)
            from ... import _build  # noqa: PLC0415

            try:
                _build.build_bridge()
            except Exception as error:
                msg = f"building {_PATH.name} failed: {error}"
                raise KernelBuildError(msg) from error
        loader = importlib.machinery.ExtensionFileLoader("_native", str(_PATH))
        try:
            module = importlib.util.module_from_spec(importlib.util.spec_from_loader("_native", loader))
            loader.exec_module(module)
        except ImportError as error:
            msg = f"the native bridge {_PATH} cannot be loaded: {error}"
            raise KernelUnavailableError(msg) from error
        entry_points = (library.cdll.msda_forward, library.cdll.msda_backward_workspace,
                        library.cdll.msda_backward_workspace_size, library.cdll.msda_last_error)
        module.init(*(ctypes.cast(f, ctypes.c_void_p).value for f in entry_points))
        _loaded = module
        return module
