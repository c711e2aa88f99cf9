"""Samples staged in chunks (the forward beyond 8 KB of records a wave and 24 MB a grid,
grad_sample beyond 4 KB), at the sizes where it can go wrong: a last chunk of one sample,
chunks that end inside a level, samples that are no multiple of a unit's lanes, one or
several chunks (with and without the barrier that keeps a workgroup's waves in step),
every dtype. And grad_sample's 8-byte location gradient stores against its 4-byte ones.

Tolerances are the parity suite's (float32 1e-5 forward, 1e-4 backward; 16-bit 2e-2 of the
largest element; float64 1e-10); the stores must agree bit for bit.
"""

from __future__ import annotations

import pytest
import torch

from deformops_amd.backends.hip import _lib
from deformops_amd.registry import msda
from tests.test_hip_msda import check_against_oracle
from tests.workloads import make_workload

pytestmark = pytest.mark.gpu

F32, BF16, F16, F64 = torch.float32, torch.bfloat16, torch.float16, torch.float64
LEVELS = ((17, 13), (9, 7), (5, 4), (3, 2), (1, 1))


@pytest.mark.parametrize("softmax", [False, True], ids=["linear", "softmax"])
@pytest.mark.parametrize(("dtype", "loc_dtype"), [(F32, F32), (BF16, BF16), (F16, F16), (BF16, F32), (F64, F64)],
                         ids=["f32", "bf16", "f16", "bf16-f32loc", "f64"])
@pytest.mark.parametrize(("levels", "points", "channels"), [
    (3, 3, 32), (3, 4, 32), (1, 17, 32), (3, 7, 32), (5, 8, 32), (1, 33, 32), (5, 5, 64), (5, 8, 64), (2, 33, 16),
    (5, 13, 8), (4, 16, 128),
])
def test_chunked_staging_matches_the_oracle(device, levels, points, channels, dtype, loc_dtype, softmax):
    w = make_workload(2, batch=2, queries=203, heads=3, channels=channels, points=points, levels=LEVELS[:levels],
                      locations="uniform", seed=3).to(device, dtype, loc_dtype)
    check_against_oracle(*w.operands(softmax=softmax), w.grad_output, softmax=softmax, dtype=dtype,
                         label=f"L={levels} P={points} D={channels}")


@pytest.mark.parametrize("softmax", [False, True], ids=["linear", "softmax"])
@pytest.mark.parametrize(("dtype", "loc_dtype"), [(F32, F32), (BF16, F32), (F16, F16), (F64, F64)],
                         ids=["f32", "bf16-f32loc", "f16", "f64"])
@pytest.mark.parametrize(("levels", "points", "channels"), [
    (1, 33, 32), (3, 7, 16), (5, 8, 32), (5, 5, 64), (2, 33, 16), (5, 13, 8), (4, 16, 128), (5, 4, 24),
])
def test_forward_in_chunks_equals_the_forward_staged_whole(device, levels, points, channels, dtype, loc_dtype, softmax):
    """A grid of up to 24 MB of records is staged whole, a larger one in chunks: the same call
    repeated over the batch gives the same bits."""
    w = make_workload(2, batch=2, queries=203, heads=3, channels=channels, points=points, levels=LEVELS[:levels],
                      locations="uniform", seed=6).to(device, dtype, loc_dtype)
    value, shapes, starts, loc, attn = w.operands(softmax=softmax)
    samples = levels * points
    per_call = 2 * 203 * 3 * samples * (dtype.itemsize + 2 * loc_dtype.itemsize + (48 if dtype is F64 else 32))
    whole, many = (24 << 20) // per_call // 2, (24 << 20) // per_call + 2
    assert whole >= 1

    def forward(times):
        v, x, a = (t.repeat(times, *[1] * (t.dim() - 1)) for t in (value, loc, attn))
        return msda(v, shapes, starts, x, a, softmax=softmax)

    want = forward(1)
    for times in (whole, many):
        got = forward(times).view(times, *want.shape)
        torch.testing.assert_close(got, want.expand_as(got), rtol=0, atol=0)


@pytest.mark.parametrize("dtype", [F32, BF16], ids=["f32", "bf16-f32loc"])
def test_location_gradients_at_a_four_byte_offset(device, dtype):
    """grad_sampling_locations need only be 4-byte aligned: float pairs then take two stores."""
    lib = _lib.load()
    w = make_workload(2, batch=1, queries=301, heads=4, seed=9).to(device, dtype, F32)
    value, shapes, starts, loc, attn = w.operands()
    grads = [torch.empty_like(value), torch.empty_like(attn)]
    buffer = torch.empty(loc.numel() + 1, dtype=F32, device=device)
    results = []
    for offset in (0, 1):
        out = buffer[offset : offset + loc.numel()]
        out.fill_(float("nan"))
        lib.check(lib.backward(
            value.data_ptr(), _lib.DTYPE_CODES[dtype], shapes.data_ptr(), starts.data_ptr(), 0, loc.data_ptr(), 0,
            attn.data_ptr(), w.grad_output.data_ptr(), grads[0].data_ptr(), out.data_ptr(), grads[1].data_ptr(),
            *w.sizes, 0, torch.cuda.current_stream().cuda_stream))
        torch.cuda.synchronize()
        results.append(out.clone())
    torch.testing.assert_close(results[0], results[1], rtol=0, atol=0)
