"""RMSNorm rows that start off a 16-byte boundary, in every kernel: the
packets are the aligned ones at another address, so each result must be bit
for bit that of the same rows laid out on 16-byte boundaries."""

from __future__ import annotations

import pytest
import torch

from ako_amd import _native
from ako_amd.ops.rmsnorm_hip import rmsnorm_hip, rmsnorm_residual_hip
from ako_amd.ops.rmsnorm_tp import rmsnorm_shard_apply_hip, rmsnorm_shard_partial_hip

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a GPU")]
DEV = "cuda"
# (rows, hidden): short rows, register rows with and without a partial packet
# (early and late weights, one and several packets per lane, the shapes whose
# aligned rows store write-through), the pipelined launches, the two-pass kernel.
SHAPES = [(5, 3), (33, 80), (3, 515), (40, 4096), (257, 4099), (300, 4096), (10300, 4096), (270, 8191), (300, 16384),
          (2051, 16384), (2, 70001)]


def _rows(rows: int, hidden: int, dtype: torch.dtype, seed: int, start: int, pad: int) -> torch.Tensor:
    """The seed's rows with ``pad`` elements between them, from element ``start`` of an allocation."""
    gen = torch.Generator(device=DEV).manual_seed(seed)
    values = torch.randn(rows, hidden, generator=gen, device=DEV).to(dtype)
    step = hidden + pad
    buf = torch.zeros(rows * step + start, dtype=dtype, device=DEV)
    view = buf[start:].view(rows, step)[:, :hidden]
    view.copy_(values)
    return view


def _aligned_pad(hidden: int) -> int:
    return -hidden % 8


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("start,pad", [(1, 0), (2, 0), (7, 1), (0, 3)])
def test_unaligned_rows_match_aligned_rows(start: int, pad: int, dtype) -> None:
    for rows, hidden in SHAPES:
        case = f"{rows}x{hidden} {dtype}"
        w = torch.randn(hidden + 1, device=DEV).to(dtype)
        x, r = (_rows(rows, hidden, dtype, seed, start, pad) for seed in (1, 2))
        xa, ra = (_rows(rows, hidden, dtype, seed, 0, _aligned_pad(hidden)) for seed in (1, 2))
        for weight in (w[:-1], w[1:]):
            same = weight.clone()
            assert torch.equal(rmsnorm_hip(x, weight), rmsnorm_hip(xa, same)), case
            got, expected = rmsnorm_residual_hip(x, r, weight), rmsnorm_residual_hip(xa, ra, same)
            assert torch.equal(got[0], expected[0]) and torch.equal(got[1], expected[1]), case
        (s, sums), (sa, sums_a) = rmsnorm_shard_partial_hip(x, r), rmsnorm_shard_partial_hip(xa, ra)
        assert torch.equal(s, sa) and torch.equal(sums, sums_a), case
        y = rmsnorm_shard_apply_hip(x, w[1:], sums, hidden)
        assert torch.equal(y, rmsnorm_shard_apply_hip(xa, w[1:].clone(), sums, hidden)), case


def test_forced_kernels_take_unaligned_rows() -> None:
    """The two-pass kernel, the pipelined kernel and write-through stores when
    asked for (the last keep to aligned rows by themselves)."""
    x, r = (_rows(300, 4096, torch.float16, seed, 1, 1) for seed in (1, 2))
    xa, ra = (_rows(300, 4096, torch.float16, seed, 0, 0) for seed in (1, 2))
    w = torch.randn(4096, device=DEV).to(torch.float16)
    for settings in ({3: 1}, {9: 2}, {1: 16, 2: 1, 12: 2}):
        try:
            for key, value in settings.items():
                _native.set_tuning(0, key, value)
            got, expected = rmsnorm_residual_hip(x, r, w), rmsnorm_residual_hip(xa, ra, w)
            assert torch.equal(got[0], expected[0]) and torch.equal(got[1], expected[1]), settings
            assert torch.equal(rmsnorm_hip(x, w), rmsnorm_hip(xa, w)), settings
        finally:
            for key in settings:
                _native.set_tuning(0, key, 0)
