// Which RMSNorm kernel a launch takes, in which shape, and in which order it
// adds a row's squares. Plain C++ (no HIP), so that a CPU test can walk the
// whole rule.
//
// The order is settled first, from the row's width and the kind of launch,
// and the shape only among those that can add in it: a faster shape never
// changes a result. A residual row adds in one order at every launch size, and
// so does a plain row of at most 256 packets; a plain row of 257-1024 packets
// has one order in launches of at most kFewRows rows and in those of the
// pipelined kernel's size, and another one between.
#pragma once

#include <stdint.h>

namespace ako {

// Launches of at most this many rows leave CUs without a workgroup (256 CUs).
constexpr int64_t kFewRows = 256;

// Widest row (in packets) of rmsnorm_short.
constexpr int64_t kShortPackets = 64;

// Widest row held in registers: 16 wavefronts x 64 lanes x 8 packets (65536
// half-precision elements). Wider rows take the two-pass kernel.
constexpr int64_t kMaxRegPackets = 16 * 64 * 8;

// Wavefronts per row and packets per lane.
struct RegShape {
  int wpr, vpt;
};
// Instantiated shapes, smallest first.
constexpr RegShape kRegShapes[] = {{1, 1}, {1, 2},  {1, 4},  {1, 8},  {2, 1},  {2, 2},  {2, 4},
                                   {2, 8}, {4, 1},  {4, 2},  {4, 4},  {4, 8},  {8, 1},  {8, 2},
                                   {8, 4}, {8, 8},  {16, 1}, {16, 2}, {16, 4}, {16, 8}};

// Separate sums per lane of a register shape that adds in the order of a wider
// one (see rmsnorm_reg); every shape has this one variant beside the one with
// a single sum. The order of `total` = wavefronts x packets: plain rows add as
// 2 x 2, 4 x 2, 8 x 2, 16 x 2 or 16 x 4, residual rows as 2 x 2, 8 x 1, 16 x 1
// or 16 x 2. Plain 4 x 2 and 8 x 2 themselves stand in for 8 x 1 and 16 x 1.
constexpr int reg_sums(int wpr, int vpt, bool residual) {
  const int total = wpr * vpt;
  if (residual && vpt > 4) return 1;  // not among the resident shapes of residual rows
  int order = 0;                      // wavefronts of the order
  if (total == 4) order = 2;
  if (total == 8) order = residual || vpt == 2 ? 8 : 4;
  if (total == 16) order = residual || vpt == 2 ? 16 : 8;
  if (total == 32) order = 16;
  if (total == 64) order = 16;
  return order > wpr ? order / wpr : 1;
}

// Wavefronts and packets of the order in which a launch adds. `one_packet`:
// plain rows of 257-1024 packets take one packet per lane, as residual rows do.
//
// These are also the shapes of large launches (with the plain rows that a
// large launch holds at two packets per lane). Medians of three cold runs per
// shape on MI355X, 16384 rows, fp16 and bf16: plain rows are fastest with two
// packets per lane over 4-16 wavefronts; residual rows, which load two tensors
// per packet, with one packet per lane over 8-16 wavefronts. Launches of at
// most kFewRows (decode) take one packet per lane, a row to a workgroup, since
// one row's latency is the launch's: graph-replayed on MI355X, plain rows of
// 4096 half elements take 1.89 us as (8, 1) against 2.13 us as (4, 2) at 1 row
// (2.04 against 2.28 at 32 rows). Rows of 65-256 packets would gain by it too
// (bf16, cold, (4, 1) against these shapes: 32 rows of 2048, plain 2.52 and 2.89
// us, residual 2.85 and 3.33; 300 rows 2.83 and 3.11, 3.25 and 3.79), as would
// plain rows of 257-512 packets above kFewRows ((8, 1) against (4, 2): 300 x 4096
// 3.27 and 3.43 us), but not in the order of their larger launches.
inline RegShape sum_order(int64_t nvec, bool one_packet) {
  if (nvec <= 64) return {1, 1};
  if (nvec <= 128) return {1, 2};
  if (nvec <= 256) return {2, 2};
  if (nvec <= 512) return one_packet ? RegShape{8, 1} : RegShape{4, 2};
  if (nvec <= 1024) return one_packet ? RegShape{16, 1} : RegShape{8, 2};
  if (nvec <= 2048) return {16, 2};
  return nvec <= 4096 ? RegShape{16, 4} : RegShape{16, 8};
}

// Shape of a launch of kFewRows to some thousand rows: the one whose wavefronts
// are resident all at once, so that every row's loads go out at the start and
// no second round of workgroups waits for the first. Fewer packets per lane
// spread a row's latency over more lanes, so the smallest packet count that
// fits and adds in the row's order is taken, and never 16 wavefronts of more
// than one packet (plain rows of 10240-16384, 279-500 rows: 10-25% behind 8 of
// four). Against the order's own shape, fp16, cold and graph-replayed:
// residual 512 x 4096 5.8 -> 4.6 us, 2048 x 4096 15.2 -> 12.6, 4096 x 4096 29.5 ->
// 25.2, 1024 x 8192 15.2 -> 12.8; plain 4096 x 3072 11.9 -> 10.2, 4096 x 4096
// 14.6 -> 12.8, 1024 x 16384 15.0 -> 13.4.
//
// Wavefronts that fit, from sweeps of every shape over 13 widths x 24 row
// counts (bf16, cold, MI355X). A CU holds 32, 24 at eight packets per lane, but
// the lead ends earlier where a row's wavefronts come in large workgroups or
// use most of their packets: past the counts below the next shape is level or
// up to 15% faster.
inline int64_t resident_waves(RegShape s, int64_t nvec, bool residual) {
  if (residual) {
    // Wavefronts that hold a packet; rows with idle ones last a little longer
    // (512 x 6144 5.9 us against 6.4 as (8, 2), but full 384 x 8192 8.0 and 7.6).
    if (s.vpt == 1) return nvec > 64 * (s.wpr - 1) ? 5632 : 6400;
    // 2400 x 2048 8.9 us against 9.9 as (1, 4), 1200 x 4096 8.9 and 10.1 as (2, 4).
    if (s.vpt == 2) return 5120;
    return s.vpt == 4 ? 8192 : 0;
  }
  if (s.vpt == 1) return 5120;
  if (s.vpt == 2) return 8192;
  // 600 x 14336 10.4 us against 8.5 as (4, 8), but 600 x 10240 6.5 and 7.2.
  if (s.vpt == 4) return s.wpr == 8 && nvec > 1280 ? 4096 : 6144;
  // 2100 x 8192 17.1 us against 15.1 as (8, 2), but 2400 x 7168 14.2 and 15.7.
  return s.wpr == 2 && nvec > 896 ? 4096 : 6144;
}

// A shape whose wavefronts fit and that adds in `order`, or {0, 0}. It holds as
// many packets over fewer wavefronts, with more sums per lane.
inline RegShape resident_shape(RegShape order, int64_t nvec, bool residual, int64_t rows) {
  const int total = order.wpr * order.vpt;
  for (int vpt = 1; vpt <= 8; vpt *= 2) {
    const RegShape s{total / vpt, vpt};
    if (s.wpr < 1 || s.wpr > order.wpr || s.wpr > (vpt == 1 ? 16 : 8)) continue;
    const int64_t waves = residual && vpt == 1 ? (nvec + 63) / 64 : s.wpr;
    if (rows * waves <= resident_waves(s, nvec, residual)) return s;
  }
  return {0, 0};
}

// Widest input row (x, plus the residual) the pipelined kernel takes by
// default, the fewest rows per workgroup, and the fewest at which plain rows
// add in its order.
constexpr int64_t kPipeMaxRowBytes = 16 * 1024;
constexpr int64_t kPipeMinRowsPerBlock = 20;
constexpr int64_t kPipeOrderRowsPerBlock = 16;

// Shapes with a pipelined instantiation (those of launches of many rows up to
// 65536 half-precision elements, and their neighbours).
constexpr RegShape kPipeShapes[] = {{4, 2}, {8, 1}, {8, 2}, {16, 1}, {16, 2}, {16, 4}};

inline bool pipe_shape(const RegShape& s) {
  for (const RegShape& c : kPipeShapes)
    if (c.wpr == s.wpr && c.vpt == s.vpt) return true;
  return false;
}

// What the rule looks at, of the launch and of the tuning keys (see RmsTuning).
struct NormCall {
  int64_t nvec;       // whole packets per row
  bool full;          // no partial packet
  int64_t row_bytes;  // of one tensor
  int64_t rows;
  bool residual;
  int cus;
};
struct NormKeys {
  int waves_per_row, vecs_per_thread, force_stream, early_weights, pipeline, pipe_blocks_per_cu, load_groups,
      write_through;
};

// Workgroups of a pipelined launch (a multiple of 8). Workgroups per CU: 16
// wavefronts per CU for plain rows, 8 for residual rows (two tensors in
// flight per row). Measured at 16384 rows of 4096 half elements: plain 6598
// GB/s with 16 wavefronts per CU against 6029 with 8; residual 6976 with 8
// against 6826 with 16.
inline int64_t pipe_blocks(int wpr, bool residual, int64_t rows, int cus, int forced_per_cu) {
  const int waves = residual ? 8 : 16;
  const int64_t per_cu = forced_per_cu > 0 ? forced_per_cu : wpr < waves ? waves / wpr : 1;
  const int64_t blocks = per_cu * cus < rows ? per_cu * cus : rows;
  return blocks >= 16 ? blocks / 8 * 8 : 8;
}

// Rows of rmsnorm_shard_apply, `per_block` to a workgroup: 8 apart, workgroup b
// of a launch starting at row (b / 8) * 8 * per_block + b % 8. So each runs on
// the XCD whose workgroups of the partial half wrote it (workgroup b runs on XCD
// b % 8), soon after its neighbours, and finds what is left of it in the L2.
// Both halves, bf16, MI355X, cold, 4096 rows of 512 / 1024 / 2048: neighbouring
// rows 9.7 / 11.8 / 17.5 us, half a launch apart 9.1 / 12.2 / 17.9, 8 apart 9.0 /
// 11.9 / 17.7 (4096-16384 rows of 64-2048, 8 apart against half a launch apart:
// 1.3% faster on average, at worst 0.7% slower).
//
// Workgroups of a launch of `rows` rows:
inline int64_t shard_blocks(int64_t rows, int per_block) {
  return per_block == 1 ? rows : (rows + 8 * per_block - 1) / (8 * per_block) * 8;
}
// The most rows of one launch of at most `max_blocks` workgroups (8 or more of
// them where per_block > 1):
inline int64_t shard_launch_rows(int per_block, int64_t max_blocks) {
  return per_block == 1 ? max_blocks : max_blocks / 8 * 8 * per_block;
}

enum class NormKernel { kShort, kReg, kPipe, kStream };
struct NormRoute {
  NormKernel kernel;
  RegShape shape;  // kReg and kPipe
  int sums;        // kReg: sums per lane
};

// Rows of at most kShortPackets take rmsnorm_short unless a shape is forced.
//
// The pipelined kernel takes full rows only (no packet past the row's end)
// and launches of many rows. By default it runs rows of 512 or 1024
// packets whose inputs (x, and the residual) total at most 16 KiB, as one
// packet per lane per tensor over nvec / 64 wavefronts, once a launch is too
// large to be resident at once. Its lead depends on the outputs: 16384
// residual rows of 4096 take 76-78 us written over the buffers of the call
// before, whose lines the 256 MB MALL still holds, but 98-105 us into buffers
// not touched lately, against 86-87 us for rmsnorm_reg either way (plain 4096
// 41 and 53 against 44 us, plain 8192 77 and 97 against 84 us). Below 20
// rows per workgroup it is level at best: residual 4096 x 4096 23.4 and 26.3
// against 22.7 us, plain 4096 x 8192 23.4 and 28.3 against 23.7 us; plain rows
// add in its order from 16 all the same. Rows of 32 KiB of input (residual
// 8192, plain and residual 16384), and two packets per lane at any width, were
// 3-18% slower pipelined.
//
// Resident shapes are for the defaults: a key that names a variant of the
// large launches' shapes (8 = 2, 9 = 2, 11, 12) gets the shape it belongs to.
inline NormRoute norm_route(const NormCall& a, const NormKeys& k) {
  const bool forced_shape = k.waves_per_row > 0 || k.vecs_per_thread > 0;
  if (a.nvec <= kShortPackets && !forced_shape && k.force_stream == 0) return {NormKernel::kShort, {0, 0}, 1};
  if (k.force_stream != 0 || a.nvec > kMaxRegPackets) return {NormKernel::kStream, {0, 0}, 1};

  const bool few = a.rows <= kFewRows;
  const bool pipe_rows = !few && a.rows < (int64_t(1) << 31) && a.full;
  const bool pipe_width = (a.nvec == 512 || a.nvec == 1024) && a.row_bytes * (a.residual ? 2 : 1) <= kPipeMaxRowBytes;
  int64_t rows_per_block = 0;
  if (k.pipeline == 0 && !forced_shape && pipe_rows && pipe_width)
    rows_per_block = a.rows / pipe_blocks(static_cast<int>(a.nvec / 64), a.residual, a.rows, a.cus, k.pipe_blocks_per_cu);
  if (rows_per_block >= kPipeMinRowsPerBlock) return {NormKernel::kPipe, {static_cast<int>(a.nvec / 64), 1}, 1};

  // A plain launch that adds in the pipelined kernel's order without taking it
  // keeps the shape of large launches.
  const bool pipe_order = !a.residual && rows_per_block >= kPipeOrderRowsPerBlock;
  const RegShape order = sum_order(a.nvec, a.residual || few || pipe_order);
  RegShape s = pipe_order ? sum_order(a.nvec, false) : order;
  const bool variant_key = k.early_weights == 2 || k.pipeline == 2 || k.load_groups != 0 || k.write_through != 0;
  if (!few && !pipe_order && !variant_key && !forced_shape) {
    const RegShape r = resident_shape(order, a.nvec, a.residual, a.rows);
    if (r.wpr > 0) s = r;
  }
  int sums = order.wpr / s.wpr;
  if (forced_shape) {
    const RegShape want{k.waves_per_row > 0 ? k.waves_per_row : s.wpr, k.vecs_per_thread > 0 ? k.vecs_per_thread : s.vpt};
    for (const RegShape& c : kRegShapes)
      if (c.wpr == want.wpr && c.vpt == want.vpt && int64_t(c.wpr) * 64 * c.vpt >= a.nvec) s = c;
    sums = 1;
  }
  if (k.pipeline == 2 && pipe_rows && int64_t(s.wpr) * 64 * s.vpt == a.nvec && pipe_shape(s))
    return {NormKernel::kPipe, s, 1};
  return {NormKernel::kReg, s, sums};
}

}  // namespace ako
