"""RMSNorm rows of at most 64 packets (``rmsnorm_short``, several rows to a
wavefront): at the widths where the lanes per row change, with partial
packets and with idle lanes, and at row counts that leave partial workgroups.

The kernel adds in the order of one wavefront per row (the register kernel's
one-packet shape, forced through the tuning keys), so whole outputs must be
bit-identical to it; the small launches also go against the oracle.
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

from ako_amd import _native
from ako_amd.ops.rmsnorm_hip import rmsnorm_hip, rmsnorm_residual_hip
from oracle import ops as oracle
from tests._util import NAMES, to_np

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a GPU")]
DEV = "cuda"
MAX_ULPS = {torch.float16: 2.0, torch.bfloat16: 2.0, torch.float32: 4.0}
# Packets per row: the edges of each lane count, and idle lanes inside one.
PACKETS = [0, 1, 3, 4, 5, 8, 10, 16, 17, 24, 32, 33, 64]


def _inputs(rows: int, hidden: int, dtype: torch.dtype):
    """x and residual with rows a multiple of 16 bytes apart (the packet path at any width), and a weight."""
    gen = torch.Generator(device=DEV).manual_seed(rows * 1000 + hidden)
    step = -(-hidden // 8) * 8
    x, r = (torch.randn(rows, step, generator=gen, device=DEV).to(dtype)[:, :hidden] for _ in range(2))
    w = (torch.randn(hidden, generator=gen, device=DEV) * 0.1 + 1.0).to(dtype)
    return x, r, w


def _one_wavefront_per_row(fn):
    """fn with the register kernel's (1 wavefront, 1 packet) shape forced."""
    try:
        _native.set_tuning(0, 1, 1)
        _native.set_tuning(0, 2, 1)
        return fn()
    finally:
        _native.set_tuning(0, 1, 0)
        _native.set_tuning(0, 2, 0)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("extra", [0, 1, 3])
def test_short_rows(dtype, extra: int) -> None:
    per_packet = 16 // dtype.itemsize
    for packets in PACKETS:
        hidden = packets * per_packet + extra
        if hidden == 0:
            continue
        for rows in (1, 3, 33, 259):
            case = f"{rows}x{hidden} {dtype}"
            x, r, w = _inputs(rows, hidden, dtype)
            y = rmsnorm_hip(x, w, 1e-6)
            yr, s = rmsnorm_residual_hip(x, r, w, 1e-6)
            rep = oracle.gate(oracle.rmsnorm(to_np(x), to_np(w), 1e-6, dtype=NAMES[dtype]), to_np(y), NAMES[dtype])
            assert rep["passed"] and rep["err_ulps"] <= MAX_ULPS[dtype], (case, rep)
            ey, es = oracle.rmsnorm_residual(to_np(x), to_np(r), to_np(w), 1e-6, dtype=NAMES[dtype])
            np.testing.assert_array_equal(to_np(s), es, err_msg=case)
            rep = oracle.gate(ey, to_np(yr), NAMES[dtype])
            assert rep["passed"] and rep["err_ulps"] <= MAX_ULPS[dtype], (case, rep)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("hidden,rows", [(40, 131_075), (80, 65_540), (128, 65_541), (192, 32_771), (384, 16_387),
                                         (67, 131_073)])
def test_short_rows_of_many_row_launches(hidden: int, rows: int, dtype) -> None:
    """Launches past the row count where plain rows with idle lanes take two
    row groups per workgroup, the last of them partial."""
    if dtype == torch.float32 and hidden > 256:
        pytest.skip("more than 64 packets")
    x, r, w = _inputs(rows, hidden, dtype)
    y = rmsnorm_hip(x, w, 1e-6)
    yr, s = rmsnorm_residual_hip(x, r, w, 1e-6)
    assert torch.equal(s, x + r)
    assert torch.equal(y, _one_wavefront_per_row(lambda: rmsnorm_hip(x, w, 1e-6)))
    assert torch.equal(yr, _one_wavefront_per_row(lambda: rmsnorm_residual_hip(x, r, w, 1e-6)[0]))
    pick = torch.tensor([0, 1, rows // 2, rows - 2, rows - 1], device=DEV)
    rep = oracle.gate(oracle.rmsnorm(to_np(x[pick]), to_np(w), 1e-6, dtype=NAMES[dtype]), to_np(y[pick]), NAMES[dtype])
    assert rep["passed"] and rep["err_ulps"] <= MAX_ULPS[dtype], rep
