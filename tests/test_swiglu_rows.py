"""SwiGLU on strided rows of any width and start (``swiglu_rows``, packets of
all rows laid end to end) against the dense kernel on contiguous copies: the
same arithmetic on the same elements, so bit-identical outputs."""

from __future__ import annotations

import pytest
import torch

from ako_amd.ops.swiglu_hip import swiglu_hip
from oracle import ops as oracle
from tests._util import NAMES, to_np

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a GPU")]
DEV = "cuda"


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("rows,width", [(2, 1), (3, 7), (5, 8), (33, 31), (7, 513), (64, 2048), (3, 4099),
                                        (1200, 4101), (3001, 1408)])
def test_halves_match_contiguous_copies(rows: int, width: int, dtype) -> None:
    """The two halves of one tensor: rows without a whole packet, with a partial
    one, on and off 16-byte boundaries, and launches that go to the XCDs in runs."""
    gen = torch.Generator(device=DEV).manual_seed(rows + width)
    for start in (0, 1):
        buf = (torch.randn(rows * 2 * width + start, generator=gen, device=DEV) * 3).to(dtype)
        both = buf[start:].view(rows, 2 * width)
        gate, up = both[:, :width], both[:, width:]
        y = swiglu_hip(gate, up)
        assert torch.equal(y, swiglu_hip(gate.contiguous(), up.contiguous()))
        assert torch.equal(y, swiglu_hip(gate, up.contiguous()))
    if rows * width < 100_000:
        rep = oracle.gate(oracle.swiglu(to_np(gate), to_np(up), dtype=NAMES[dtype]), to_np(y), NAMES[dtype])
        assert rep["passed"] and rep["err_ulps"] <= (4.0 if dtype == torch.float32 else 2.0), rep


@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
def test_dense_blocks_off_a_boundary(dtype) -> None:
    gen = torch.Generator(device=DEV).manual_seed(3)
    gate, up = ((torch.randn(4099 * 3 + 1, generator=gen, device=DEV) * 3).to(dtype)[1:].view(3, 4099) for _ in range(2))
    assert torch.equal(swiglu_hip(gate, up), swiglu_hip(gate.clone(), up.clone()))
