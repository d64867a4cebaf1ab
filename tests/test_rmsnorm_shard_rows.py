"""The apply half of the sharded RMSNorm at the row counts where a workgroup
takes two rows (4096 up), 8 apart: whole and partial groups of 16 rows, each
row the same as in a launch of one row per workgroup; and both halves at the
widest slice."""

from __future__ import annotations

import pytest
import torch

from ako_amd.ops.rmsnorm_tp import rmsnorm_shard_apply_hip, rmsnorm_shard_partial_hip

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a GPU")]


@pytest.mark.parametrize("rows", [4095, 4096, 4097, 4103, 4104, 8191])
@pytest.mark.parametrize("width", [8, 264, 515])
def test_two_rows_per_workgroup(rows: int, width: int) -> None:
    gen = torch.Generator(device="cuda").manual_seed(rows + width)
    x, r = (torch.randn(rows, width, generator=gen, device="cuda").to(torch.bfloat16) for _ in range(2))
    w = torch.randn(width, generator=gen, device="cuda").to(torch.bfloat16)
    s, sums = rmsnorm_shard_partial_hip(x, r)
    assert torch.equal(s, x + r)
    y = rmsnorm_shard_apply_hip(s, w, sums, 4 * width)
    parts = [rmsnorm_shard_apply_hip(s[i:i + 1000], w, sums[i:i + 1000], 4 * width) for i in range(0, rows, 1000)]
    assert torch.equal(y, torch.cat(parts))


def test_widest_slice() -> None:
    """2^31 - 1 columns, the most that the entry points take: the index past the
    last whole packet stays below 2^31 (7 columns of bfloat16 are there)."""
    width = 2**31 - 1
    x = torch.ones(1, width, dtype=torch.bfloat16, device="cuda")
    x[0, -7:] = 2.0
    s, sums = rmsnorm_shard_partial_hip(x)
    # 256 lanes add about 2^23 exact ones each in fp32 (exact), then 256 sums (2^-24 each).
    assert abs(float(sums[0]) - (width + 7 * 3)) <= width * 256 * 2.0**-24
    y = rmsnorm_shard_apply_hip(s, x[0], sums, width)
    assert bool((y[0, :-7] == 1.0).all()) and bool((y[0, -7:] == 4.0).all())
