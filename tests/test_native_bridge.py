"""The native bridge of plain eager calls (csrc/bridge.cpp): what it takes, what it
leaves to the registry's own path, and that its autograd node behaves as a Python
autograd.Function over the same two library calls would (saved-tensor hooks, a second
backward, forward-mode differentiation, views and strides, another stream).

Results are compared bit for bit with the registered operators, which make the same
library calls (grad_value to 1e-5 in float32: its summation order may vary), so no
numeric bar beyond that is needed.
"""

from __future__ import annotations

import pytest
import torch

from deformops_amd.backends.hip import _native
from deformops_amd.registry import Backend, msda
from tests.workloads import make_workload

F32, BF16 = torch.float32, torch.bfloat16


def operands(device, dtype=F32, **kwargs):  # noqa: ANN001, ANN003, ANN201
    w = make_workload(2, batch=1, queries=300, heads=2, channels=16, seed=5, **kwargs).to(device, dtype)
    return list(w.operands()), w.grad_output


class Subclass(torch.Tensor):
    pass


def test_calls_that_are_not_plain_gpu_tensors_are_left_alone():
    (value, shapes, starts, loc, attn), _ = operands("cpu")
    take = _native.load().try_forward
    assert take(value, shapes, starts, loc, attn, False) is None  # CPU tensors
    assert take(value.as_subclass(Subclass), shapes, starts, loc, attn, False) is None
    assert take(None, shapes, starts, loc, attn, False) is None
    assert take(value.tolist(), shapes, starts, loc, attn, False) is None


@pytest.mark.gpu
@pytest.mark.parametrize("change", [
    "heads", "levels", "dtype", "float-table", "rank", "points", "device", "subclass", "function-mode", "vmap",
])
def test_unusual_calls_are_left_to_the_registry(device, change):
    args, _ = operands(device)
    take = _native.load().try_forward
    assert take(*args, False) is not None
    value, shapes, starts, loc, attn = args
    if change == "heads":
        value = value[:, :, :1]
    elif change == "levels":
        shapes = shapes[:2]
    elif change == "dtype":
        attn = attn.to(BF16)
    elif change == "float-table":
        starts = starts.float()
    elif change == "rank":
        value = value[0]
    elif change == "points":
        attn = attn[..., :-1]
    elif change == "device":
        shapes = shapes.cpu()
    elif change == "subclass":
        value = value.as_subclass(Subclass)
    elif change == "function-mode":
        with torch.overrides.BaseTorchFunctionMode():
            assert take(value, shapes, starts, loc, attn, False) is None
        return
    elif change == "vmap":
        def inner(v):  # noqa: ANN001, ANN202
            assert take(v, shapes, starts, loc, attn, False) is None
            return v
        torch.vmap(inner)(value[None])
        return
    assert take(value, shapes, starts, loc, attn, False) is None


@pytest.mark.gpu
def test_level_table_checks_still_run_when_asked_for(device, monkeypatch):
    args, _ = operands(device)
    args[2] = args[2] + 1
    msda(*args)  # treated as empty levels, no read out of bounds
    monkeypatch.setenv("DEFORMOPS_VALIDATE", "1")
    with pytest.raises(ValueError, match="level_start_index"):
        msda(*args)


@pytest.mark.gpu
@pytest.mark.parametrize("method", ["linear", "softmax"])
@pytest.mark.parametrize("layout", ["contiguous", "strided", "split", "int32", "half-locations"])
def test_native_node_matches_the_registered_operators(device, layout, method):
    (value, shapes, starts, loc, attn), grad = operands(device, BF16)
    if layout == "strided":
        value = value.transpose(1, 2).contiguous().transpose(1, 2)
        loc = loc.flip(1).flip(1)[..., [0, 1]]
        attn = torch.cat([attn, attn], -1)[..., : attn.shape[-1]]
    elif layout == "split":
        attn = attn.view(*loc.shape[:-1])
    elif layout == "int32":
        shapes, starts = shapes.int(), starts.int()
    elif layout == "half-locations":
        loc = loc.half()  # neither float32 nor the value dtype: widened
    op = torch.ops.deformops_hip.msda_softmax_forward if method == "softmax" else torch.ops.deformops_hip.msda_forward
    results = []
    for native in (True, False):
        leaves = [t.detach().clone(memory_format=torch.preserve_format).requires_grad_(True) for t in (value, loc, attn)]
        if native:
            out = msda(leaves[0], shapes, starts, leaves[1], leaves[2], method=method)
        else:
            out = op(leaves[0], shapes, starts, leaves[1], leaves[2], 128, loc.shape[4], 0, 0)
        out.backward(grad, retain_graph=True)
        out.backward(grad)  # a retained graph runs again
        results.append([out.detach(), *(leaf.grad for leaf in leaves)])
    for i, (a, b) in enumerate(zip(*results)):
        assert a.dtype == b.dtype and a.shape == b.shape
        if i == 1:  # grad_value: two bfloat16 roundings of sums in another order
            torch.testing.assert_close(a, b, rtol=2**-7, atol=2**-7 * b.abs().max().item())
        else:
            torch.testing.assert_close(a, b, rtol=0, atol=0)


@pytest.mark.gpu
def test_saved_tensor_hooks_see_the_five_operands(device):
    (value, shapes, starts, loc, attn), grad = operands(device)
    leaf = value.clone().requires_grad_(True)
    packed, unpacked = [], []

    def pack(t):  # noqa: ANN001, ANN202
        packed.append(t.shape)
        return t.cpu()

    def unpack(t):  # noqa: ANN001, ANN202
        unpacked.append(t.shape)
        return t.to(device)

    with torch.autograd.graph.saved_tensors_hooks(pack, unpack):
        out = msda(leaf, shapes, starts, loc, attn)
    out.backward(grad)
    assert packed == [t.shape for t in (value, shapes, starts, loc, attn)] and unpacked == packed
    with_hooks, leaf.grad = leaf.grad, None
    msda(leaf, shapes, starts, loc, attn).backward(grad)
    torch.testing.assert_close(leaf.grad, with_hooks, rtol=1e-5, atol=1e-5)


@pytest.mark.gpu
@pytest.mark.parametrize("name", ["value", "loc", "attn"])
@pytest.mark.parametrize("change", ["host", "sizes", "strided"])
def test_unpacked_operands_of_another_kind(device, change, name):
    """A saved-tensor hook that hands back host memory or other sizes is an error before the
    launch; other strides are read as what they hold."""
    (value, shapes, starts, loc, attn), grad = operands(device)
    leaves = [t.clone().requires_grad_(True) for t in (value, loc, attn)]
    target = {"value": value, "loc": loc, "attn": attn}[name]

    def unpack(t):  # noqa: ANN001, ANN202
        if t.shape != target.shape:
            return t
        if change == "host":
            return t.cpu()
        return t[:, :, :1] if change == "sizes" else t.transpose(1, 2).contiguous().transpose(1, 2)

    with torch.autograd.graph.saved_tensors_hooks(lambda t: t, unpack):
        out = msda(leaves[0], shapes, starts, *leaves[1:])
    if change != "strided":
        with pytest.raises(RuntimeError, match="unpacked for the backward"):
            out.backward(grad)
        return
    got = torch.autograd.grad(out, leaves, grad)
    want = torch.autograd.grad(msda(leaves[0], shapes, starts, *leaves[1:]), leaves, grad)
    torch.testing.assert_close(got[0], want[0], rtol=1e-5, atol=1e-5)
    for a, b in zip(got[1:], want[1:]):
        torch.testing.assert_close(a, b, rtol=0, atol=0)


@pytest.mark.gpu
@pytest.mark.parametrize("backend", [None, Backend.HIP], ids=["registry", "explicit"])
@pytest.mark.parametrize("no_grad", [False, True], ids=["grad", "no-grad"])
@pytest.mark.parametrize("requires_grad", [False, True], ids=["constant", "leaf"])
@pytest.mark.parametrize("operand", [0, 3, 4], ids=["value", "loc", "weights"])
def test_a_tangent_is_refused_in_every_grad_mode(device, operand, requires_grad, no_grad, backend):
    args, _ = operands(device)
    msda.load(Backend.HIP)  # from here on a registry call tries the bridge first
    with torch.autograd.forward_ad.dual_level():
        primal = args[operand].requires_grad_(requires_grad)
        args[operand] = torch.autograd.forward_ad.make_dual(primal, torch.ones_like(primal))
        with torch.set_grad_enabled(not no_grad), pytest.raises(NotImplementedError, match="forward-mode"):
            msda(*args, backend=backend)
    args[operand] = primal
    msda(*args, backend=backend)  # outside the level it is an ordinary operand again


@pytest.mark.gpu
def test_no_grad_and_inference_mode_record_nothing(device):
    args, _ = operands(device)
    args[0].requires_grad_(True)
    with torch.no_grad():
        assert not msda(*args).requires_grad
    with torch.inference_mode():
        assert not msda(*args).requires_grad
    assert msda(*args).requires_grad


@pytest.mark.gpu
def test_a_call_runs_on_the_current_stream(device):
    args, grad = operands(device)
    want = msda(*args)
    leaf = args[0].clone().requires_grad_(True)
    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(stream):
        out = msda(leaf, *args[1:])
        out.backward(grad)
    torch.cuda.current_stream().wait_stream(stream)
    torch.testing.assert_close(out, want, rtol=0, atol=0)
    assert torch.isfinite(leaf.grad).all() and leaf.grad.abs().sum() > 0


@pytest.mark.gpu
def test_traced_calls_record_the_operator(device):
    args, _ = operands(device)
    assert msda.get(Backend.HIP) is not None
    traced = torch.jit.trace(lambda v: msda(v, *args[1:]), (args[0],), check_trace=False)
    other = torch.randn_like(args[0])
    torch.testing.assert_close(traced(other), msda(other, *args[1:]), rtol=0, atol=0)
