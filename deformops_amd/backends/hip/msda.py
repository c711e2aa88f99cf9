r"""Registry adapter of the HIP MSDA kernels (reference: backends/cuda/msda.py:14-51)."""

from __future__ import annotations

from typing import Any

import torch

from ...core.runtime import Method, resolve_method
from ...registry import Backend, msda
from . import _lib, _native
from ._bridge import forward, supports_context


def msda_hip(
    value: Any,
    spatial_shapes: Any,
    level_start_index: Any,
    sampling_locations: Any,
    attention_weights: Any,
    *,
    chunk_step: int = 128,
    num_points: int | None = None,
    channels_per_thread: int = 0,
    threads_per_block: int = 0,
    method: Any = None,
    softmax: bool = False,
    **kwargs: Any,  # noqa: ARG001 - backend options of other builds (fp32acc)
) -> Any:
    """Run MSDA on the gfx950 HIP kernels."""
    use_softmax = resolve_method(method, softmax=softmax) is Method.SOFTMAX
    return forward(
        value,
        spatial_shapes,
        level_start_index,
        sampling_locations,
        attention_weights,
        chunk_step,
        num_points=num_points,
        channels_per_thread=channels_per_thread,
        threads_per_block=threads_per_block,
        softmax=use_softmax,
    )


def load(*, download: bool | None = None, compile: bool | str | None = None) -> str:  # noqa: A002
    """Load libdeformops_amd.so and its native bridge; return the library's path."""
    path = str(_lib.load(download=download, compile=compile).path)
    _native.load(download=download, compile=compile)
    return path


def direct(*tensors: Any, softmax: bool) -> Any:
    """A plain eager GPU call that needs no check the native bridge cannot make, or
    ``None`` (see ``try_forward`` in csrc/bridge.cpp). Also ``None`` until ``load`` has
    loaded the bridge: which backend a call runs on, and the error of a call that none
    can run, stay the policy's."""
    native = _native.loaded()
    return None if native is None else native.try_forward(*tensors, softmax)


if torch.cuda.is_available() and torch.version.hip is not None:
    msda.register(Backend.HIP, msda_hip, supports=supports_context, load=load, direct=direct)
else:
    msda.mark_unavailable(Backend.HIP, "no ROCm GPU is available to this process")
