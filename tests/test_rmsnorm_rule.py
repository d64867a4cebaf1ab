"""The rule that picks an RMSNorm launch's kernel, shape and order of sums
(ako_amd/csrc/rmsnorm_rule.h), walked on the CPU: compiled with g++ from the
header itself.

A register shape of ``wpr`` wavefronts, ``vpt`` packets per lane and ``sums``
sums per lane adds packet ``p`` of a row into chain
``(p / 64) % (wpr * sums)`` of lane ``p % 64``, packets of one chain in
ascending order, and then the chains in order. So the chain of every packet
says the whole order, and two launches add alike when all chains are equal.
"""

from __future__ import annotations

import shutil
import subprocess
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parent.parent / "ako_amd" / "csrc"

DRIVER = r"""
#include <cstdio>
#include <vector>
#include "rmsnorm_rule.h"
using namespace ako;

// Without arguments, norm_route of the launches on stdin:
// <nvec> <full> <row bytes> <rows> <residual> <cus> <8 keys>, one launch per input line.
int shards() {  // every row of a launch in one workgroup, and no more workgroups than allowed
  long bad = 0;
  for (int64_t cap : {1, 2, 3, 5, 8, 9, 15, 16, 64, 1000})
    for (int per_block = 1; per_block <= 2; ++per_block) {
      const int64_t most = shard_launch_rows(per_block, cap);
      if (cap >= 8) bad += most <= 0;
      for (int64_t rows = 1; rows <= most; ++rows) {
        const int64_t blocks = shard_blocks(rows, per_block);
        std::vector<int> taken(rows);
        for (int64_t b = 0; b < blocks; ++b)
          for (int64_t k = 0; k < per_block; ++k) {
            const int64_t r = (per_block == 1 ? b : b / 8 * (8 * per_block) + b % 8) + 8 * k;
            if (r < rows) ++taken[r];
            bad += r % 8 != b % 8;  // the XCD that the row was written on
          }
        bad += blocks > cap;
        for (int t : taken) bad += t != 1;
      }
    }
  std::printf("%ld\n", bad);
  return bad != 0;
}

int main(int argc, char**) {
  if (argc > 1) return shards();
  long long nvec, bytes, rows;
  int full, residual, cus, k[8];
  while (std::scanf("%lld %d %lld %lld %d %d", &nvec, &full, &bytes, &rows, &residual, &cus) == 6) {
    for (int& v : k)
      if (std::scanf("%d", &v) != 1) return 2;
    const NormRoute r = norm_route({nvec, full != 0, bytes, rows, residual != 0, cus},
                                   {k[0], k[1], k[2], k[3], k[4], k[5], k[6], k[7]});
    std::printf("%d %d %d %d %d\n", int(r.kernel), r.shape.wpr, r.shape.vpt, r.sums,
                r.shape.wpr > 0 ? reg_sums(r.shape.wpr, r.shape.vpt, residual != 0) : 1);
  }
}
"""
KERNELS = ("short", "reg", "pipe", "stream")
KEYS = ("waves_per_row", "vecs_per_thread", "force_stream", "early_weights", "pipeline", "pipe_blocks_per_cu",
        "load_groups", "write_through")


@pytest.fixture(scope="module")
def route(tmp_path_factory):
    """route(launches) -> [(kernel, wpr, vpt, sums)]; a launch is (rows, hidden, itemsize, residual, {key: value})."""
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("g++ is not available")
    folder = tmp_path_factory.mktemp("rule")
    (folder / "rule.cpp").write_text(DRIVER)
    subprocess.run([gxx, "-O2", "-std=c++17", "-Wall", "-Werror", f"-I{CSRC}", str(folder / "rule.cpp"), "-o",
                    str(folder / "rule")], check=True)

    def ask(launches, cus: int = 256):
        lines = []
        for rows, hidden, itemsize, residual, keys in launches:
            per = 16 // itemsize
            lines.append(" ".join(map(str, [hidden // per, int(hidden % per == 0), hidden * itemsize, rows,
                                            int(residual), cus, *(keys.get(k, 0) for k in KEYS)])))
        out = subprocess.run([str(folder / "rule")], input="\n".join(lines), capture_output=True, text=True,
                             timeout=120, check=True).stdout.split()
        values = [tuple(map(int, out[i:i + 5])) for i in range(0, len(out), 5)]
        assert len(values) == len(launches)
        for launch, (kernel, wpr, vpt, sums, instantiated) in zip(launches, values):
            assert sums in (1, instantiated), launch  # a launch never asks for a variant that is not compiled
        return [(KERNELS[kernel], wpr, vpt, sums) for kernel, wpr, vpt, sums, _ in values]

    ask.exe = folder / "rule"
    return ask


def test_sharded_rows_fill_no_more_workgroups_than_allowed(route) -> None:
    """Two rows a workgroup, 8 apart: each row once, on its XCD, within the cap on workgroups (key 7)."""
    out = subprocess.run([str(route.exe), "shards"], capture_output=True, text=True, timeout=60)
    assert out.returncode == 0, out.stdout


def _expected_order(packets: int, one_packet: bool) -> int:
    """Chains of the order that a row of this many packets has."""
    for limit, two, one in ((64, 1, 1), (128, 1, 1), (256, 2, 2), (512, 4, 8), (1024, 8, 16)):
        if packets <= limit:
            return one if one_packet else two
    return 16


WIDTHS = [65, 100, 127, 128, 129, 200, 255, 256, 257, 300, 384, 511, 512, 513, 640, 1000, 1023, 1024, 1025, 1500, 2047,
          2048, 2049, 3000, 4095, 4096, 4097, 6000, 8192]
ROWS = sorted({1, 2, 255, 256, 257, 100_000} | {limit // waves + off for limit in (4096, 5120, 5632, 6144, 6400, 7168, 8192, 10240)
                                                for waves in range(1, 17) for off in (-1, 0, 1)})


@pytest.mark.parametrize("cus", [256, 64])
@pytest.mark.parametrize("itemsize", [2, 4])
@pytest.mark.parametrize("residual", [False, True])
def test_every_shape_adds_in_the_rows_order(route, residual: bool, itemsize: int, cus: int) -> None:
    launches = [(rows, packets * (16 // itemsize) + tail, itemsize, residual, {})
                for packets in WIDTHS for tail in (0, 1) for rows in ROWS]
    for (rows, hidden, *_), (kernel, wpr, vpt, sums) in zip(launches, route(launches, cus)):
        case = (rows, hidden, kernel, wpr, vpt, sums)
        packets, full = hidden * itemsize // 16, hidden % (16 // itemsize) == 0
        assert kernel in ("reg", "pipe") and wpr * 64 * vpt >= packets, case
        if kernel == "pipe":
            assert full and wpr * 64 * vpt == packets and sums == 1, case
        # Plain rows of 257-1024 packets: one packet per lane in decode-sized
        # launches and from 16 rows per workgroup of the pipelined kernel.
        pipelined = (full and packets in (512, 1024) and hidden * itemsize <= 16384 and rows > 256
                     and rows // (max(1, 16 * 64 // packets) * cus) >= 16)
        order = _expected_order(packets, residual or rows <= 256 or pipelined)
        assert wpr * sums == order, case
        # Each chain's packets ascend lane by lane: chain (p / 64) % order, as in one shape of `order` wavefronts.
        assert vpt % sums == 0 and (sums == 1 or wpr * vpt <= 64), case


def test_resident_shapes_hold_no_more_than_a_row(route) -> None:
    """At most twice the lanes' packets that the row has: no launch takes four packets per lane where two hold it."""
    launches = [(rows, packets * 8, 2, residual, {}) for packets in WIDTHS for rows in ROWS for residual in (False, True)]
    for (rows, hidden, *_), (_, wpr, vpt, _) in zip(launches, route(launches)):
        assert wpr * vpt * 64 < 2 * (hidden // 8) or wpr * vpt <= 2, (rows, hidden, wpr, vpt)


def test_keys_of_a_shape_get_that_shape(route) -> None:
    """A key that names a variant of the large launches' shapes runs on them at every size above decode."""
    for keys in ({"load_groups": 1}, {"load_groups": 2}, {"write_through": 1}, {"write_through": 2}):
        assert route([(300, 16384, 2, res, keys) for res in (False, True)]) == [("reg", 16, 2, 1)] * 2
    full = [(rows, hidden, 2, res) for rows in (257, 1031, 4099) for hidden in (4096, 8192, 16384, 32768)
            for res in (False, True)]
    got = route([(*launch, {"pipeline": 2}) for launch in full])
    assert {kernel for kernel, *_ in got} == {"pipe"}
    assert [shape[1:3] for shape in got] == [
        {4096: (8, 1) if res else (4, 2), 8192: (16, 1) if res else (8, 2), 16384: (16, 2), 32768: (16, 4)}[hidden]
        for _, hidden, _, res in full]


def test_launches_that_the_gpu_tests_name(route) -> None:
    """The sizes at which GPU tests mean a certain kernel reach it (half elements)."""
    def kernels(*launches):
        return route([(rows, hidden, 2, res, {}) for rows, hidden, res in launches])

    # Padded outputs, unaligned rows and captured launches: pipelined, and write-through (16, 2) rows.
    assert {k for k, *_ in kernels((10300, 4096, False), (10300, 4096, True), (5200, 8192, False))} == {"pipe"}
    assert kernels((2051, 16384, False), (2051, 16384, True), (1603, 16384, False), (1603, 16384, True)) == [
        ("reg", 16, 2, 1)] * 4
    # Resident shapes with separate sums beside them.
    assert kernels((300, 16384, False), (300, 16384, True), (1000, 16384, False), (1000, 16384, True)) == [
        ("reg", 8, 4, 2), ("reg", 8, 4, 2), ("reg", 4, 8, 4), ("reg", 8, 4, 2)]
    # Rows that add in the pipelined kernel's order without taking it.
    assert kernels((9000, 4096, False), (4100, 8192, False)) == [("reg", 4, 2, 2), ("reg", 8, 2, 2)]
    assert kernels((9000, 4096, True), (4100, 8192, True)) == [("pipe", 8, 1, 1), ("reg", 16, 1, 1)]
    assert kernels((2, 70001, False), (2, 70001, True)) == [("stream", 0, 0, 1)] * 2
