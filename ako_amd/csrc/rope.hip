// Rotary position embedding (neox and interleaved pairing) for gfx950.
//
// One kernel, rope_packets: each lane moves one 16-byte packet (or packet
// pair) of one head of one token. Lanes are numbered through the packets of a
// head, the heads of a token (those of a second and third tensor continue the
// first's), then the tokens, so a wavefront covers whole heads back to back
// and no lane waits on a token's last head. Rotating a (q, k) pair is one
// launch (ako_rope_qk_fwd). A lane finds its packet, head, token and batch by
// multiply-shift divisions. It has one of three layouts:
//
//   kInterleaved  a packet holds whole (2i, 2i+1) pairs.
//   kHalves       neox: a lane holds packet j of the lower and packet j of the
//                 upper half, and writes both. Heads do not straddle
//                 wavefronts, so that each half's stores of one head leave
//                 together.
//   kWhole        neox: a lane holds one packet of the head and reads the
//                 partner packet half a head away too, but writes only its
//                 own, so a wavefront's loads and stores run through whole
//                 heads. For small launches, and for halves that are no
//                 whole lines, whose lines kHalves touches in two
//                 instructions (run_packet has the sizes).
//
// Packets need no alignment (common.h), so any strides and table offsets take
// them. Where a half (interleaved: a head) is no whole number of packets, the
// last packet is moved back to end with it: the overlap is computed by two
// lanes from the same inputs and stored twice with the same values. Heads
// shorter than a packet take packets of 4, 2 or 1 elements.
//
// KV-cache mode (CACHE): the position of token s is read on the device (*pos +
// s), the tables are read at that row, q is rotated to its output, k is rotated
// into slot *pos + s of the key cache and v is copied into the same slot of the
// value cache, all in the one launch. A captured decode step can then be
// replayed while *pos advances.
//
// Numerics follow ako/ops/rope_ref.py:73-107: a' = a*c - b*n and
// b' = a*n + b*c in fp32 with each product rounded separately (the library is
// built with -ffp-contract=off), then rounded to the storage dtype.

#include <algorithm>

#include "common.h"
#include "launch.h"

namespace ako {

RopeTuning g_rope_tuning;

struct RopeTensorDev {
  const void* x;
  void* y;
  int64_t heads;
  int64_t sxb, sxs, sxh;
  int64_t syb, sys, syh;
};

struct RopeDev {
  RopeTensorDev t0, t1, t2;  // t2: copied, not rotated (KV-cache mode only)
  const int64_t* pos;        // KV-cache mode: device-side position of token s = 0
  int64_t cache_len;
  const void* cos;
  const void* sin;
  int64_t st;
  unsigned units;        // heads (of all tokens and tensors) in this launch
  unsigned token0;       // the launch starts at head head0 of this token
  unsigned head0;
  unsigned heads;        // heads per token, all tensors
  unsigned seq;
  unsigned per_unit;     // lanes per head
  unsigned per_wave;     // kHalves: whole heads per wavefront
  int half;              // head_dim / 2
  int last;              // element offset of the last packet of a half (interleaved: of a head)
  FastDiv by_unit, by_heads, by_seq;
  XcdRuns runs;          // workgroup order over the XCDs
};

enum RopeLayout { kInterleaved, kHalves, kWhole };

// LNT: non-temporal source loads. kWhole reads every line through two packets
// and mostly wants it kept for the second (run_packet).
template <typename T, typename TT, RopeLayout LAYOUT, int E, bool LNT, bool CACHE, int BLOCK>
__global__ __launch_bounds__(BLOCK) void rope_packets(RopeDev a) {
  constexpr int NT = LAYOUT == kInterleaved ? E / 2 : E;  // table values per lane
  using P = Pack<T, E>;

  // Which packet (32-bit arithmetic: the host bounds a launch's lanes). Spare
  // lanes load what the last head's lanes load and skip only their stores:
  // with no branch ahead of the loads, every kernel argument is fetched at
  // once at the start instead of in a second scalar load round trip.
  const unsigned block = block_order(blockIdx.x, gridDim.x, a.runs);
  unsigned unit, j;
  bool live;
  if constexpr (LAYOUT == kHalves) {
    const unsigned lane = threadIdx.x % kWave;
    const unsigned q = fast_div(lane, a.by_unit);
    j = lane - q * a.per_unit;
    live = q < a.per_wave;
    unit = (block * (BLOCK / kWave) + threadIdx.x / kWave) * a.per_wave + (live ? q : 0);
  } else {
    const unsigned id = block * BLOCK + threadIdx.x;
    unit = fast_div(id, a.by_unit);
    j = id - unit * a.per_unit;
    live = true;
  }
  if (unit >= a.units) {
    live = false;
    unit = a.units - 1;
  }
  const unsigned u = unit + a.head0;
  const unsigned tl = fast_div(u, a.by_heads);
  const unsigned h = u - tl * a.heads;
  const unsigned token = a.token0 + tl;
  const unsigned b = fast_div(token, a.by_seq);
  const unsigned s = token - b * a.seq;

  // The tensor of head h is chosen field by field, by value: the fields then
  // come from scalar kernel-argument loads and a per-lane select. Binding a
  // reference to the per-lane choice makes the compiler fetch the whole
  // descriptor with vector loads, a memory round trip that every wavefront
  // waits for before it can issue its first data load.
  const unsigned n0 = static_cast<unsigned>(a.t0.heads), n01 = n0 + static_cast<unsigned>(a.t1.heads);
  const bool first = h < n0;
  [[maybe_unused]] const bool third = CACHE && h >= n01;
  const auto pick = [&](const auto& f0, const auto& f1, const auto& f2) { return first ? f0 : (third ? f2 : f1); };
  const unsigned hh = first ? h : (third ? h - n01 : h - n0);
  // The packet's element offset in its half (interleaved: its head), in the
  // source row, of its partner there, and in the table row.
  unsigned offset;
  [[maybe_unused]] bool upper = false;
  if constexpr (LAYOUT == kWhole) {
    upper = j >= a.per_unit / 2;
    if (upper) j -= a.per_unit / 2;
  }
  offset = j * E < static_cast<unsigned>(a.last) ? j * E : static_cast<unsigned>(a.last);
  const unsigned own_at = LAYOUT == kWhole && upper ? offset + a.half : offset;
  [[maybe_unused]] const unsigned partner_at = LAYOUT == kWhole && upper ? offset : offset + a.half;
  const unsigned table_at = LAYOUT == kInterleaved ? offset / 2 : offset;

  // Row of the tables and, in KV-cache mode, the cache slot of this token. A
  // token whose slot falls outside the cache writes no cache slot, and its q
  // rows are filled with NaN (table row 0 is read and replaced by NaN, so the
  // rotation yields NaN): the broken contract shows instead of stale memory.
  float c[NT], n[NT];
  int64_t p = s;
  [[maybe_unused]] bool dropped = false;
  const auto load_tables = [&]() {
    if constexpr (CACHE) {
      const int64_t pp = *a.pos + s;
      dropped = pp < 0 || pp >= a.cache_len;
      p = dropped ? 0 : pp;
    }
    load_f32<TT, NT>(static_cast<const TT*>(a.cos) + p * a.st + table_at, c);
    load_f32<TT, NT>(static_cast<const TT*>(a.sin) + p * a.st + table_at, n);
  };
  // In KV-cache mode the source rows do not depend on the position, which is
  // a dependent scalar load: their loads are issued first, so the position's
  // round trip overlaps them instead of preceding them. Otherwise the table
  // row goes first, as the data loads' addresses need no memory read either.
  if constexpr (!CACHE) load_tables();
  const T* src = static_cast<const T*>(pick(a.t0.x, a.t1.x, a.t2.x)) + b * pick(a.t0.sxb, a.t1.sxb, a.t2.sxb) +
                 s * pick(a.t0.sxs, a.t1.sxs, a.t2.sxs) + hh * pick(a.t0.sxh, a.t1.sxh, a.t2.sxh);
  P own;
  [[maybe_unused]] P partner;
  own = load_pack<T, E, LNT>(src + own_at);
  if constexpr (LAYOUT != kInterleaved) partner = load_pack<T, E, LNT>(src + partner_at);
  if constexpr (CACHE) load_tables();
  // The destination's offset is formed while the loads are in flight (all but
  // the cache slot, which the position decides); the empty asm keeps the
  // compiler from forming it after them instead, 0.5-1% at (4, 2048, 40, 128).
  int64_t to = b * pick(a.t0.syb, a.t1.syb, a.t2.syb) + hh * pick(a.t0.syh, a.t1.syh, a.t2.syh) + own_at;
  const int64_t row_stride = pick(a.t0.sys, a.t1.sys, a.t2.sys);
  if constexpr (!CACHE) to += s * row_stride;
  asm volatile("" : "+v"(to));
  // Every load is issued before the first is waited for: left to itself the
  // compiler widens the tables, and waits for them, between the data loads.
  __builtin_amdgcn_sched_barrier(0);
  if (!live) return;
  if constexpr (CACHE) {
    if (dropped) {
      if (!first) return;  // no cache slot for this token
#pragma unroll
      for (int e = 0; e < NT; ++e) c[e] = n[e] = __builtin_nanf("");
    }
  }
  if constexpr (CACHE) to += (first ? static_cast<int64_t>(s) : p) * row_stride;
  T* dst = static_cast<T*>(pick(a.t0.y, a.t1.y, a.t2.y)) + to;
  if constexpr (CACHE) {
    if (third) {
      store_pack<T, E, true>(dst, own);
      if constexpr (LAYOUT == kHalves) store_pack<T, E, true>(dst + a.half, partner);
      return;
    }
  }
  P o;
  if constexpr (LAYOUT == kInterleaved) {
#pragma unroll
    for (int i = 0; i < E / 2; ++i) {
      const float x0 = to_f32(own.e[2 * i]), x1 = to_f32(own.e[2 * i + 1]);
      o.e[2 * i] = from_f32<T>(x0 * c[i] - x1 * n[i]);
      o.e[2 * i + 1] = from_f32<T>(x0 * n[i] + x1 * c[i]);
    }
  } else if constexpr (LAYOUT == kWhole) {
#pragma unroll
    for (int e = 0; e < E; ++e) {
      const float xc = to_f32(own.e[e]) * c[e], pn = to_f32(partner.e[e]) * n[e];
      o.e[e] = from_f32<T>(upper ? pn + xc : xc - pn);
    }
  } else {
    P hi;
#pragma unroll
    for (int e = 0; e < E; ++e) {
      const float x0 = to_f32(own.e[e]), x1 = to_f32(partner.e[e]);
      o.e[e] = from_f32<T>(x0 * c[e] - x1 * n[e]);
      hi.e[e] = from_f32<T>(x0 * n[e] + x1 * c[e]);
    }
    store_pack<T, E, true>(dst + a.half, hi);
  }
  store_pack<T, E, true>(dst, o);
}

namespace {

RopeTensorDev to_dev(const RopeTensorArgs& t) {
  return RopeTensorDev{t.x, t.y, t.heads, t.sxb, t.sxs, t.sxh, t.syb, t.sys, t.syh};
}

constexpr int64_t kLanesPerLaunch = int64_t(1) << 30;  // ids and grid work-items stay well below 2^32

// Launches of at least kRunsMinBlocks workgroups go to the XCDs in runs of
// kRun where that streamed faster than block order: fp32 (3 x 1025 x 64 heads
// of 128, interleaved 35.3 -> 32.6 us, neox 33.4 -> 32.6 us), interleaved (8 x
// 4096 x 64 heads of 128, fp16 171.7 -> 166.5 us), one tensor in halves (4 x
// 2048 x 32 heads of 128 22.6 -> 22.4 us; runs of 128 22.9 us) and halves into
// the caches (4 x 2000 x 48 heads of 128 33.7 -> 32.5 us). Not the rest: fp16 q
// and k in halves 27.7 against 27.9 us, whole heads of 80 18.9 against 19.3 us,
// interleaved into the caches 34.3 against 34.4 us. Below 4096 workgroups runs
// were level or up to 2% slower.
constexpr int64_t kRunsMinBlocks = 4096;
constexpr unsigned kRun = 32;

template <typename T, RopeLayout LAYOUT, bool CACHE>
XcdRuns runs_for(int64_t blocks, bool one_tensor) {
  const int forced = g_rope_tuning.xcd_chunk;
  if (forced > 0) return make_xcd_runs(static_cast<unsigned>(forced));
  const bool runs = CACHE ? LAYOUT == kHalves
                          : sizeof(T) == 4 || LAYOUT == kInterleaved || (LAYOUT == kHalves && one_tensor);
  return make_xcd_runs(runs && blocks >= kRunsMinBlocks ? kRun : 1u);
}

template <typename T, typename TT, RopeLayout LAYOUT, int E, bool LNT, bool CACHE, int BLOCK>
hipError_t run_block(RopeDev d, int64_t units, hipStream_t stream) {
  // kHalves: kWave lanes hold per_wave heads, otherwise per_unit lanes a head.
  const int64_t lanes_per_unit = LAYOUT == kHalves ? ceil_div(kWave, d.per_wave) : d.per_unit;
  const int64_t per_launch = std::max<int64_t>(1, kLanesPerLaunch / lanes_per_unit);
  for (int64_t u0 = 0; u0 < units; u0 += per_launch) {
    const int64_t n = std::min(per_launch, units - u0);
    d.units = static_cast<unsigned>(n);
    d.token0 = static_cast<unsigned>(u0 / d.heads);
    d.head0 = static_cast<unsigned>(u0 % d.heads);
    const int64_t lanes = LAYOUT == kHalves ? ceil_div(n, d.per_wave) * kWave : n * d.per_unit;
    const int64_t blocks = ceil_div(lanes, BLOCK);
    d.runs = runs_for<T, LAYOUT, CACHE>(blocks, d.t1.heads == 0);
    AKO_LAUNCH((rope_packets<T, TT, LAYOUT, E, LNT, CACHE, BLOCK>), dim3(static_cast<unsigned>(blocks)),
               dim3(BLOCK), 0, stream, d);
    const hipError_t err = hipGetLastError();
    if (err != hipSuccess) return err;
  }
  return hipSuccess;
}

// One wavefront per workgroup for launches of at most kSmallWaves wavefronts,
// so that they spread over as many CUs as possible, and for whole heads into
// the caches; four otherwise. MI355X, fp16, 40 heads of 128: 64 tokens 2.14
// against 2.36 us, 512 tokens (2560 wavefronts) 3.21 against 3.35 us, 1024
// tokens (5120) 5.33 against 5.12 us; into the caches, 8000 tokens, 48 heads of
// 80 27.4 against 29.9 us, halves of 128 33.8 us both ways.
constexpr int64_t kSmallWaves = 4096;

template <typename T, typename TT, RopeLayout LAYOUT, int E, bool LNT, bool CACHE>
hipError_t run_layout(RopeDev d, int64_t tokens, hipStream_t stream) {
  const int64_t packets = ceil_div(int64_t(d.last), E) + 1;
  d.per_unit = static_cast<unsigned>(LAYOUT == kWhole ? 2 * packets : packets);
  d.per_wave = LAYOUT == kHalves ? kWave / d.per_unit : 1;
  d.by_unit = make_fastdiv(d.per_unit);
  const int64_t units = tokens * d.heads;
  const int64_t waves = LAYOUT == kHalves ? ceil_div(units, d.per_wave) : ceil_div(units * d.per_unit, kWave);
  const int forced = g_rope_tuning.waves_per_block;
  const bool one_wave = waves <= kSmallWaves || (CACHE && LAYOUT != kHalves);
  return forced == 1 || (forced <= 0 && one_wave)
             ? run_block<T, TT, LAYOUT, E, LNT, CACHE, kWave>(d, units, stream)
             : run_block<T, TT, LAYOUT, E, LNT, CACHE, 4 * kWave>(d, units, stream);
}

// neox layouts, by the wavefronts (1 KiB of source rows each) that whole heads
// would take and the bytes of a half. MI355X, fp16, 40 heads; "in cache": source
// rows that a kernel has just written, as the projection before does, else
// rows from memory.
//
//   up to 1024: whole heads. One wavefront's latency is the launch's, and one
//     packet to store is less of it than two: heads of 128, 64 tokens 2.20
//     against 2.32 us in halves, heads of 80 2.16 against 2.28.
//   halves of a 128-byte line or more above that: kHalves. 4 x 2048 tokens of
//     heads of 128 27.7 against 29.1 us; heads of 192, 1024 tokens 7.9 against 8.6
//     us (in cache 8.6 and 11.0), 8192 tokens 44.7 and 48.5 (35.6 and 38.3); into
//     the caches, 48 heads of 192, 512 / 2048 / 4 x 2048 tokens 6.2 / 15.6 / 52.7
//     against 6.9 / 17.6 / 64.0 us.
//   but whole heads from 16384 to 40960, whose rows stay in the cache between the
//     projection and this launch, where such halves are no whole lines: in cache
//     2048 tokens of heads of 160 / 208 10.7 / 13.4 against 11.7 / 13.7 us (from
//     memory 12.7 / 15.8 and 12.1 / 14.8), and from 16384 on where they are no whole
//     packets either (heads of 136, 2048 / 4096 tokens in cache 10.4 / 17.0 against
//     11.4 / 20.3 us, from memory level). Not into the caches, where it is slower.
//   shorter halves: whole heads, but halves from 2048 to 8192, where the launch
//     is resident at once and the doubled source and table reads of whole heads
//     are not hidden: 512 tokens of heads of 64 / 80 / 96 2.74 / 3.17 / 3.53 against
//     2.88 / 3.24 / 3.72 us; 2048 tokens 6.3 / 7.8 / 8.6 against 5.8 / 6.9 / 7.8 us.
//
// Whole heads read every line twice and load without the non-temporal hint,
// which keeps the lines for the partner reads. In cache, with the hint / without:
// heads of 72 / 80 / 136, 64 tokens 2.48 / 2.16 / 2.68 -> 2.18 / 1.96 / 2.40 us,
// heads of 80 / 96, 2048 tokens 10.4 / 10.9 -> 9.1 / 8.8, heads of 80 into the
// caches, 1536 tokens 10.6 -> 9.9; from memory level (heads of 80 / 96, 2048 tokens
// 7.7 / 8.6 -> 7.9 / 8.7).
// Only launches of more than kHalvesMaxWaves of halves of at most 64 bytes have
// it: there rows from memory lose more (2048 tokens of heads of 64 6.4 -> 6.7 us).
//
// Against one wavefront per (token, group of heads) in halves for every shape:
// heads of 64 / 80 / 96 at 4 x 2048 17.6 / 22.4 / 25.9 -> 15.8 / 18.9 / 22.2 us;
// heads of 72, one lane per rotated pair then, 61 -> 18.6 us; interleaved heads
// of 80 / 192 19.4 / 50 -> 18.2 / 40.4 us; heads of 128 and 192 unchanged.
constexpr int64_t kWholeAlwaysWaves = 1024;
constexpr int64_t kHalvesMinWaves = 2048, kHalvesMaxWaves = 8192;
constexpr int64_t kWholeCachedWaves = 16384, kWholeCachedMaxWaves = 40960;

template <typename T, typename TT, int E, bool CACHE>
hipError_t run_packet(RopeDev d, bool neox, int64_t tokens, hipStream_t stream) {
  if (!neox) {
    d.last = 2 * d.half - E;
    if constexpr (E >= 2) return run_layout<T, TT, kInterleaved, E, true, CACHE>(d, tokens, stream);
    return hipErrorInvalidValue;
  }
  d.last = d.half - E;
  const int64_t packets = ceil_div(d.half, E), half_bytes = d.half * static_cast<int64_t>(sizeof(T));
  const int64_t waves = ceil_div(tokens * d.heads * 2 * packets, kWave);
  const bool whole_lines = half_bytes % 128 == 0 || sizeof(T) == 4 || CACHE;
  const bool whole_cached = !whole_lines && waves > kWholeCachedWaves &&
                            (waves <= kWholeCachedMaxWaves || half_bytes % 16 != 0);
  // kHalves needs a half's packets within one wavefront.
  const bool halves = packets <= kWave && waves > kWholeAlwaysWaves &&
                      (half_bytes >= 128 ? !whole_cached : waves > kHalvesMinWaves && waves <= kHalvesMaxWaves);
  if (halves) return run_layout<T, TT, kHalves, E, true, CACHE>(d, tokens, stream);
  if (waves > kHalvesMaxWaves && half_bytes <= 64)
    return run_layout<T, TT, kWhole, E, true, CACHE>(d, tokens, stream);
  return run_layout<T, TT, kWhole, E, false, CACHE>(d, tokens, stream);
}

// Elements per packet: 16 bytes, or the largest smaller power of two that a
// half (interleaved: a head) has.
template <typename T, typename TT, bool CACHE>
hipError_t run_cache(const RopeArgs& a, const RopeDev& d, hipStream_t stream) {
  constexpr int E = 16 / sizeof(T);
  const int64_t tokens = a.batch * a.seq, elements = a.neox ? a.head_dim / 2 : a.head_dim;
  if (elements >= E) return run_packet<T, TT, E, CACHE>(d, a.neox, tokens, stream);
  if constexpr (E > 4) {
    if (elements >= 4) return run_packet<T, TT, 4, CACHE>(d, a.neox, tokens, stream);
  }
  if (elements >= 2) return run_packet<T, TT, 2, CACHE>(d, a.neox, tokens, stream);
  return run_packet<T, TT, 1, CACHE>(d, a.neox, tokens, stream);
}

template <typename T, typename TT>
hipError_t run_typed(const RopeArgs& a, hipStream_t stream) {
  RopeDev d{};
  d.t0 = to_dev(a.t0);
  d.t1 = to_dev(a.t1);
  d.t2 = to_dev(a.t2);
  d.pos = a.pos;
  d.cache_len = a.cache_len;
  d.cos = a.cos;
  d.sin = a.sin;
  d.st = a.st;
  d.heads = static_cast<unsigned>(a.t0.heads + a.t1.heads + (a.pos != nullptr ? a.t2.heads : 0));
  d.seq = static_cast<unsigned>(a.seq);
  d.half = static_cast<int>(a.head_dim / 2);
  d.by_heads = make_fastdiv(d.heads);
  d.by_seq = make_fastdiv(d.seq);
  return a.pos != nullptr ? run_cache<T, TT, true>(a, d, stream) : run_cache<T, TT, false>(a, d, stream);
}

template <typename T>
hipError_t run_table(const RopeArgs& a, hipStream_t stream) {
  switch (a.table_dtype) {
    case kF32: return run_typed<T, float>(a, stream);
    case kF16: return run_typed<T, _Float16>(a, stream);
    case kBF16: return run_typed<T, __bf16>(a, stream);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace

hipError_t launch_rope(const RopeArgs& a, hipStream_t stream) {
  switch (a.dtype) {
    case kF32: return run_table<float>(a, stream);
    case kF16: return run_table<_Float16>(a, stream);
    case kBF16: return run_table<__bf16>(a, stream);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace ako
