"""RMSNorm launches on both sides of every row count at which the register
kernel's shape changes: rows are independent and a row's sums are the same in
any launch of its shape, so every launch must agree with the oracle, and with
the same rows computed in a decode-sized launch within the order of the sums."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from ako_amd.ops.rmsnorm_hip import rmsnorm_hip, rmsnorm_residual_hip
from oracle import ops as oracle
from tests._util import NAMES, to_np

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a GPU")]
DEV = "cuda"
MAX_ULPS = {torch.float16: 2.0, torch.bfloat16: 2.0, torch.float32: 4.0}
# Row counts around 256 (decode) and where 5120, 5632, 6144 and 8192
# wavefronts of 1-16 per row are used up, with odd ones between.
ROWS = [255, 257, 320, 321, 513, 704, 769, 1025, 1409, 1537, 2049, 3073, 4096, 4097, 6145, 8193]


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("packets", [65, 128, 200, 256, 384, 512, 640, 1024, 1500, 2048])
def test_launch_shapes(packets: int, dtype) -> None:
    per_packet = 16 // dtype.itemsize
    for rows in ROWS:
        hidden = packets * per_packet + (3 if rows % 3 == 0 else 0)  # some with a partial packet
        if rows * hidden * dtype.itemsize > 160 << 20:
            continue
        gen = torch.Generator(device=DEV).manual_seed(rows + hidden)
        x, r = (torch.randn(rows, hidden, generator=gen, device=DEV).to(dtype) for _ in range(2))
        w = (torch.randn(hidden, generator=gen, device=DEV) * 0.1 + 1.0).to(dtype)
        y = rmsnorm_hip(x, w, 1e-6)
        yr, s = rmsnorm_residual_hip(x, r, w, 1e-6)
        assert torch.equal(s, x + r), (rows, hidden)
        pick = torch.tensor([0, 1, rows // 3, rows - 2, rows - 1], device=DEV)
        for got, source in ((y, x), (yr, s)):
            expected = oracle.rmsnorm(to_np(source[pick]), to_np(w), 1e-6, dtype=NAMES[dtype])
            rep = oracle.gate(expected, to_np(got[pick]), NAMES[dtype])
            assert rep["passed"] and rep["err_ulps"] <= MAX_ULPS[dtype], (rows, hidden, rep)
            # Every row, against the unfused arithmetic in 64 bits: rounding to
            # the storage type (half an ulp, 2^-11 / 2^-8 / 2^-24 of the value)
            # and a few fp32 roundings (2^-22).
            xs = source.double()
            exact = xs * torch.rsqrt(xs.square().mean(-1, keepdim=True) + 1e-6) * w.double()
            bound = exact.abs() * ({torch.float16: 2.0**-11, torch.bfloat16: 2.0**-8, torch.float32: 2.0**-24}[dtype]
                                   + 2.0**-20) + 2.0**-24  # subnormal half spacing
            assert bool(((got.double() - exact).abs() <= bound).all()), (rows, hidden)
    assert np.isfinite(rep["err_ulps"])
