"""The record sort and the owners over its streams (the workspace backward of calls
with P a multiple of 4), against the float64 oracle and against the counting sort's
path, at the sizes where they can go wrong: chunks that are exactly full, one sample
short or a single query; more chunks than one wave holds ranges of; more buckets than
the LDS counters; tables whose bucket offsets need coarse buckets; tile and level
edges; heads of 16 to 64 channels; levels long and short enough for split and for
per-wave tasks; units of more samples than share a softmax, in chunks of one and of four
groups a thread. tests/test_abi_host.py checks that every row takes the path it stands
for.

Tolerances are the parity suite's: float32 1e-4 (grad_value's products of split 16-bit
parts have relative error at most 3 * 2^-16 = 4.6e-5 each), 16-bit 2e-2 of the largest
element (two roundings to bfloat16 are 2 * 2^-9 = 4e-3 of an element).
"""

from __future__ import annotations

import pytest
import torch

from deformops_amd.backends.hip import _lib
from tests.test_hip_msda import BWD_TOL, check_against_oracle, rel_err, run_hip
from tests.workloads import make_workload

pytestmark = pytest.mark.gpu

F32, BF16, F16, F64 = torch.float32, torch.bfloat16, torch.float16, torch.float64

#: levels, batch, queries, heads, channels, points
SHAPES = {
    "one-query": (((1, 1),), 1, 1, 1, 16, 4),
    "chunk-full": (((16, 16),), 1, 256, 2, 32, 4),
    "chunk-and-one": (((16, 16),), 1, 257, 2, 32, 4),
    "many-chunks": (((33, 31),), 1, 90001, 1, 16, 4),
    "many-buckets": (((400, 400), (9, 9)), 1, 3000, 1, 16, 4),
    "line": (((1, 20000),), 1, 20000, 1, 16, 4),
    "lines": (((3, 7000), (9000, 1)), 1, 20000, 1, 16, 4),
    "tile-edges": (((7, 9), (8, 8), (9, 17), (1, 1), (24, 16)), 2, 1003, 3, 48, 4),
    "wide-heads": (((19, 25), (10, 13)), 1, 4001, 2, 64, 8),
    "decoder": (((100, 134), (50, 67), (25, 34), (13, 17)), 2, 301, 4, 32, 4),
    "coarse-and-fine": (((64, 64), (4, 4)), 2, 5000, 4, 32, 4),
    "long-units": (((40, 50), (20, 25), (10, 13), (5, 7), (3, 4)), 1, 5000, 2, 32, 4),
}
DTYPES = [(F32, F32), (BF16, BF16), (F16, F16), (BF16, F32), (F16, F32)]


def record_chunks(levels, sizes, dtype, loc_dtype, *, softmax=False):
    """``(queries per chunk, chunks per (image, head), log2 of the tiles per bucket)`` of a
    call's record sort, the last -1 where a tile has four buckets of its own; 0 chunks
    where the counting sort takes the call (host only)."""
    B, _, H, _, Q, L, P = sizes
    chunk, chunks, offsets = _lib.load().record_plan(dtype, loc_dtype, sizes, _lib.FLAG_SOFTMAX if softmax else 0)
    tiles = 0
    for h, w in levels:
        t8 = -(-h // 8) * -(-w // 8)
        side = 4 if B * H * t8 < 384 and 13 * Q * P >= 24 * 640 * t8 else 8
        tiles += -(-h // side) * -(-w // side)
    if B * H * chunks * (4 * tiles + 1) <= offsets:
        return chunk, chunks, -1
    shift = 0
    while B * H * chunks * ((tiles >> shift) + L + 1) > offsets:
        shift += 1
    return chunk, chunks, shift


@pytest.mark.parametrize("softmax", [False, True], ids=["linear", "softmax"])
@pytest.mark.parametrize(("dtype", "loc_dtype"), DTYPES, ids=["f32", "bf16", "f16", "bf16-f32loc", "f16-f32loc"])
@pytest.mark.parametrize("shape", sorted(SHAPES))
def test_record_path_matches_the_oracle_and_the_counting_sort(device, shape, dtype, loc_dtype, softmax):
    levels, B, Q, H, D, P = SHAPES[shape]
    # A location gradient is a W (G01 - G00), of order W: at W = 20,000 it leaves f16's
    # range (65,504), so the long levels take float32 locations there.
    if max(max(side) for side in levels) > 4096 and loc_dtype is F16:
        loc_dtype = F32
    w = make_workload(2, batch=B, queries=Q, heads=H, channels=D, points=P, levels=levels, locations="uniform",
                      seed=11).to(device, dtype, loc_dtype)
    check_against_oracle(*w.operands(softmax=softmax), w.grad_output, softmax=softmax, dtype=dtype, label=shape)
    got = run_hip(*w.operands(softmax=softmax), w.grad_output, softmax=softmax)
    with _lib.path_override(_lib.PATH_ATOMIC_SORT):  # the counting sort
        want = run_hip(*w.operands(softmax=softmax), w.grad_output, softmax=softmax)
    assert rel_err(got[1], want[1].double().cpu()) <= BWD_TOL[dtype]
    for g, r in zip(got[2:], want[2:]):  # the same kernel on the same inputs
        torch.testing.assert_close(g, r, rtol=0, atol=0)


#: levels (all from position 0), batch, queries, heads, positions: one bucket per tile of a
#: level far from square, one per tile of levels that share positions, one per four tiles
COARSE = {
    "line": (((1, 20000),), 1, 20000, 1, 20000),
    "shared": (((64, 64),) * 8, 48, 640, 8, 4096),
    "stacked-lines": (((1, 20000),) * 16, 6, 320, 8, 20000),
}


def coarse_operands(shape, dtype, device):
    """Calls whose owners read coarse buckets: more tiles than the offsets' memory holds."""
    g = torch.Generator(device).manual_seed(5)
    levels, B, Q, H, S = COARSE[shape]
    L, starts = len(levels), (0,) * len(levels)
    value = torch.randn(B, S, H, 16, generator=g, device=device).to(dtype)
    loc = torch.rand(B, Q, H, L, 4, 2, generator=g, device=device)
    attn = torch.rand(B, Q, H, L * 4, generator=g, device=device).to(dtype)
    grad = torch.randn(B, Q, H * 16, generator=g, device=device).to(dtype)
    return (value, torch.tensor(levels, device=device), torch.tensor(starts, device=device), loc, attn), grad


@pytest.mark.parametrize("bad", [float("inf"), float("nan")], ids=["inf", "nan"])
@pytest.mark.parametrize(("shape", "dtype"), [("line", F32), ("line", BF16), ("shared", BF16), ("stacked-lines", F16)])
def test_a_nonfinite_channel_reaches_only_the_tiles_its_query_samples(device, shape, dtype, bad):
    """A product of a zero weight and an infinity is NaN, so a non-finite grad_output channel
    spoils the whole tile of each of its query's samples, and nothing else: where owners read
    coarse buckets, the candidates that have no corner in the tile stay out of it."""
    args, grad = coarse_operands(shape, dtype, device)
    grad[-1, 7, 3] = bad
    got = run_hip(*args, grad, softmax=False)[1]
    with _lib.path_override(_lib.PATH_ATOMIC_SORT):  # the counting sort: a tile's own samples
        want = run_hip(*args, grad, softmax=False)[1]
    spoilt = ~torch.isfinite(got)
    assert spoilt.any() and not (spoilt & torch.isfinite(want)).any()
    spoilt[-1, :, 0, 3] = False
    assert not spoilt.any()  # nor any other image, head or channel
    ok = torch.isfinite(want)
    assert rel_err(got[ok], want[ok].double().cpu()) <= BWD_TOL[dtype]


@pytest.mark.parametrize(("dtype", "offset"), [
    (F32, -3.4e38), (F32, -1e9), (F32, 1e5), (BF16, -3.38e38), (BF16, -1e9), (F16, -65000.0), (F16, 3e4),
    (F64, -1e9),  # the counting sort and the owner kernel on vector units
])
@pytest.mark.parametrize(("levels", "points", "queries"), [
    (((24, 24), (12, 12), (6, 6)), 4, 700),  # statistics formed by every group of a unit
    (((24, 24), (12, 12), (6, 6), (3, 3), (2, 2)), 8, 300),  # by one thread per unit
    (((24, 24), (12, 12), (6, 6)), 3, 700),  # the counting sort's, where they fit their range
], ids=["per-group", "per-unit", "counting-sort"])
def test_softmax_of_logits_far_from_zero(device, levels, points, queries, dtype, offset):
    """Masks of the type's lowest value, or any offset that swallows the logits: a fully masked
    unit's weights are 1 / (L P) each, as in the forward. max + log(sum) in one float drops the
    logarithm beyond about 1e7, and rounds it to 0.008 at 1e5."""
    w = make_workload(2, batch=2, queries=queries, heads=3, channels=32, points=points, levels=levels,
                      locations="uniform", seed=4).to(device, dtype, F64 if dtype is F64 else F32)
    value, shapes, starts, loc, logits = w.operands(softmax=True)
    logits = logits.clone()
    logits[:, ::3] = (logits[:, ::3].double() + offset).clamp(torch.finfo(dtype).min, torch.finfo(dtype).max).to(dtype)
    check_against_oracle(value, shapes, starts, loc, logits, w.grad_output, softmax=True, dtype=dtype,
                         label=f"offset {offset}")
