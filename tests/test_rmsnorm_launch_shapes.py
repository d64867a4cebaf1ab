"""RMSNorm launches on both sides of every row count at which the register
kernel's shape changes. Every launch agrees with the oracle and with 64 bits
within a bound, and adds a row's squares in one order for its width, whatever
shape it takes: bit for bit the result of the one shape that defines the order
(forced through the tuning keys), and of residual rows in decode-sized
launches."""

from __future__ import annotations

import pytest
import torch

from ako_amd import _native
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


def _order(packets: int, one_packet: bool) -> tuple[int, int]:
    """Wavefronts per row and packets per lane of the shape that defines a row's order of sums."""
    for limit, two, one in ((128, (1, 2), (1, 2)), (256, (2, 2), (2, 2)), (512, (4, 2), (8, 1)),
                            (1024, (8, 2), (16, 1)), (2048, (16, 2), (16, 2))):
        if packets <= limit:
            return one if one_packet else two
    return (16, 4)


def _in_shape(shape: tuple[int, int], fn):
    try:
        for key, value in zip((1, 2), shape):
            _native.set_tuning(0, key, value)
        return fn()
    finally:
        for key in (1, 2):
            _native.set_tuning(0, key, 0)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("packets", [65, 128, 129, 200, 256, 257, 384, 512, 640, 1024, 1500, 2048, 2500, 4096])
def test_every_launch_adds_in_the_rows_order(packets: int, dtype) -> None:
    per_packet = 16 // dtype.itemsize
    for rows in [33, *ROWS, 9000]:  # 9000 x 512 packets: between the register and the pipelined launches
        for tail in (0, 3):
            hidden = packets * per_packet + tail
            if rows * hidden * dtype.itemsize > 160 << 20:
                continue
            gen = torch.Generator(device=DEV).manual_seed(rows + hidden)
            x, r = (torch.randn(rows, hidden, generator=gen, device=DEV).to(dtype) for _ in range(2))
            w = (torch.randn(hidden, generator=gen, device=DEV) * 0.1 + 1.0).to(dtype)
            case = (rows, hidden)
            y, (yr, s) = rmsnorm_hip(x, w, 1e-6), rmsnorm_residual_hip(x, r, w, 1e-6)
            want, _ = _in_shape(_order(packets, True), lambda: rmsnorm_residual_hip(x, r, w, 1e-6))
            assert torch.equal(yr, want), case
            few, _ = rmsnorm_residual_hip(x[:100], r[:100], w, 1e-6)
            assert torch.equal(yr[:100], few), case
            # From 16 rows per workgroup of the pipelined kernel (16 wavefronts per CU) plain full rows of 512 or
            # 1024 packets add as it does.
            cus = torch.cuda.get_device_properties(0).multi_processor_count
            pipelined = tail == 0 and packets in (512, 1024) and rows >= 16 * cus * (1024 // packets)
            order = _order(packets, rows <= 256 or pipelined)
            assert torch.equal(y, _in_shape(order, lambda: rmsnorm_hip(x, w, 1e-6))), case
