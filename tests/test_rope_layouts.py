"""RoPE's lane layouts (``rope_packets``): packets of 8, 4, 2 and 1 elements,
halves that are no whole number of packets, halves longer than a wavefront,
rows off 16-byte boundaries, and launches on both sides of every size at
which the layout changes. RoPE rounds like the oracle, so all comparisons are
bit for bit."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from ako_amd.ops.rope_hip import rope_hip, rope_qk_cache_hip, rope_qk_hip
from ako_amd.ops.rope_ref import build_rope_tables
from oracle import ops as oracle
from tests._util import NAMES, to_np

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a GPU")]
DEV = "cuda"
HEAD_DIMS = [2, 4, 6, 8, 10, 14, 16, 18, 26, 40, 72, 80, 100, 112, 128, 160, 1042]


def _tables(rows: int, head_dim: int, dtype: torch.dtype):
    cos, sin = build_rope_tables(rows, head_dim, device=DEV)
    return cos.to(dtype), sin.to(dtype)


def _qkv(batch: int, seq: int, heads: tuple[int, int, int], head_dim: int, dtype, seed: int, start: int = 0):
    """q, k and v cut out of one projection's output that begins ``start`` elements into its buffer."""
    gen = torch.Generator(device=DEV).manual_seed(seed)
    width = sum(heads) * head_dim
    buf = torch.randn(batch * seq * width + start, generator=gen, device=DEV).to(dtype)
    whole = buf[start:].view(batch, seq, width)
    return [p.view(batch, seq, n, head_dim) for p, n in zip(whole.split([n * head_dim for n in heads], -1), heads)]


@pytest.mark.parametrize("style", ["neox", "interleaved"])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("start", [0, 1])
def test_head_dims_match_the_oracle(start: int, dtype, style: str) -> None:
    for head_dim in HEAD_DIMS:
        q, k, _ = _qkv(2, 5, (3, 2, 1), head_dim, dtype, head_dim, start)
        for tdt in (dtype, torch.float32):
            cos, sin = _tables(5, head_dim, tdt)
            for x, got in zip((q, k), rope_qk_hip(q, k, cos, sin, style)):
                expected = oracle.rope(to_np(x), to_np(cos), to_np(sin), style, dtype=NAMES[dtype],
                                       table_dtype=NAMES[tdt])
                np.testing.assert_array_equal(to_np(got), expected, err_msg=f"{head_dim} {tdt}")


# Wavefronts of whole 16-byte packets, 12 heads: either side of 2048 and of
# 8192, against slices below 1024.
@pytest.mark.parametrize("style", ["neox", "interleaved"])
@pytest.mark.parametrize("head_dim,dtype", [(32, torch.float16), (72, torch.bfloat16), (80, torch.float16),
                                            (128, torch.float16), (160, torch.bfloat16), (192, torch.float16),
                                            (72, torch.float32), (1042, torch.float16)])
def test_launch_sizes_match_small_launches(head_dim: int, dtype, style: str) -> None:
    per_token = 12 * head_dim * dtype.itemsize / 1024  # wavefronts
    for waves in (1500, 5000, 12000, 20000):
        seq = int(waves / per_token) + 1
        q, k, _ = _qkv(1, seq, (8, 4, 1), head_dim, dtype, waves)
        cos, sin = _tables(seq, head_dim, torch.float32)
        qr, kr = rope_qk_hip(q, k, cos, sin, style)
        step = max(1, seq // 23)
        for at in range(0, seq, step):
            part = slice(at, at + step)
            for x, y in ((q, qr), (k, kr)):
                small = torch.cat([rope_hip(x[:, part, h:h + 2], cos[part], sin[part], style)
                                   for h in range(0, x.shape[2], 2)], 2)
                assert torch.equal(small, y[:, part]), (waves, at)


@pytest.mark.parametrize("style", ["neox", "interleaved"])
@pytest.mark.parametrize("head_dim,dtype", [(6, torch.float32), (72, torch.float16), (80, torch.bfloat16),
                                            (128, torch.float16), (136, torch.float16), (192, torch.bfloat16)])
@pytest.mark.parametrize("seq", [1, 700, 4000])
def test_cache_writes_match_separate_calls(seq: int, head_dim: int, dtype, style: str) -> None:
    """The rotated keys and the values in their slots, every other slot untouched, at each layout's sizes."""
    q, k, v = _qkv(2, seq, (8, 4, 4), head_dim, dtype, seq + head_dim, start=1)
    cos, sin = _tables(seq + 10, head_dim, torch.float32)
    caches = [torch.full((2, 4, seq + 10, head_dim), 7.0, dtype=dtype, device=DEV) for _ in range(2)]
    pos = torch.tensor([6], device=DEV)
    qr = rope_qk_cache_hip(q, k, v, cos, sin, pos, *caches, style)
    rows = slice(6, 6 + seq)
    eq, ek = rope_qk_hip(q, k, cos[rows], sin[rows], style)
    assert torch.equal(qr, eq)
    for cache, expected in zip(caches, (ek, v)):
        assert torch.equal(cache[:, :, rows], expected.transpose(1, 2))
        assert bool((cache[:, :, :6] == 7).all()) and bool((cache[:, :, 6 + seq:] == 7).all())
