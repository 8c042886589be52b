// Workgroup order of a prefill call: which (query tile and KV chunk, sequence,
// head) a workgroup takes.  The host chooses the order (workgroup_order) and the
// kernel reads its place out of it (workgroup_place); no device code beyond that,
// so that the order can be checked on the CPU.
#pragma once

#include <stdint.h>

#if defined(__HIPCC__)
#define IFA4_HOST_DEVICE __host__ __device__ __forceinline__
#else
#define IFA4_HOST_DEVICE inline
#endif

namespace ifa4 {

// Workgroup i runs on XCD i % 8, and each XCD has its own L2.  Three orders, one
// decoding (x = i % 8 and slot i / 8, or x = 0 and slot i when lanes == 0; a slot
// counts heads fastest, then rounds, then query tiles and chunks):
//   linear  heads, then sequences;
//   pairs   XCD x gets the (sequence, kv head) pairs x, x + 8, ..., whose K/V then
//           stay in that XCD's L2;
//   spread  `unit` query heads of one kv head stay together, and the query tiles
//           of a sequence's unit take turns on the 1 << spread_log XCDs of its heads.
struct WorkgroupOrder {
  int32_t lanes;       // 3: XCD-aware (i & 7, i >> 3); 0: not
  int32_t unit;        // heads side by side in the slots of one round
  int32_t rounds;      // rounds per query tile and chunk
  int32_t pair_heads;  // pairs: kv heads of a sequence, else 0
  int32_t spread_log;  // spread: log2 of the XCDs a unit's query tiles go round
  int32_t turn;        // 1: the rounds of a query tile begin one later than the last tile's
};

struct WorkgroupPlace {
  int32_t qc;  // index of the query tile and chunk, 0 the first in the order
  int32_t seq, head;
};

// Place of workgroup i; false: a slot past the last sequence.  Every workgroup of a
// call goes through this before its first load: two divisions, one more for pairs
// or turned rounds.  (One decoding per order, six divisions on the way: calls that
// fit the chip at once ran 1 to 6% longer, 64 x 32 queries over 100 keys 10.5 -> 11.1 us.)
IFA4_HOST_DEVICE bool workgroup_place(const WorkgroupOrder& o, uint32_t i, int32_t batch,
                                      WorkgroupPlace* at) {
  const uint32_t x = o.lanes ? i & 7u : 0u, slot = i >> o.lanes;
  const uint32_t group = slot / (uint32_t)o.unit, m = slot - group * (uint32_t)o.unit;
  const uint32_t qc = group / (uint32_t)o.rounds;
  uint32_t r = group - qc * (uint32_t)o.rounds;
  at->qc = (int32_t)qc;
  if (o.pair_heads) {
    const uint32_t pair = x + 8u * r, seq = pair / (uint32_t)o.pair_heads;
    at->seq = (int32_t)seq;
    at->head = (int32_t)((pair - seq * (uint32_t)o.pair_heads) * (uint32_t)o.unit + m);
    return true;
  }
  if (o.turn) r = (r + qc) % (uint32_t)o.rounds;
  at->seq = (int32_t)((r << o.spread_log) + ((x + 7u * qc) & ((1u << o.spread_log) - 1u)));
  at->head = (int32_t)((x >> o.spread_log) * (uint32_t)o.unit + m);
  return at->seq < batch;
}

// Orders of `heads` tiles side by side (`group` of them per kv head) of `batch`
// sequences, and the workgroups of one query tile and chunk in them.
inline WorkgroupOrder linear_order(int32_t heads, int32_t batch, bool turn) {
  return WorkgroupOrder{0, heads, batch, 0, 0, turn ? 1 : 0};
}
inline WorkgroupOrder pairs_order(int32_t heads, int32_t group, int32_t batch) {
  return WorkgroupOrder{3, group, batch * (heads / group) / 8, heads / group, 0, 0};
}
inline WorkgroupOrder spread_order(int32_t heads, int32_t unit, int32_t batch) {
  const int32_t units = heads / unit;  // per sequence: 1, 2, 4 or a multiple of 8
  int32_t log = 0;
  while (units << log < 8) ++log;
  return WorkgroupOrder{3, log > 0 ? unit : units / 8 * unit, (batch + (1 << log) - 1) >> log, 0,
                        log, 1};
}
inline int64_t order_blocks(const WorkgroupOrder& o) {
  return (int64_t)o.unit * o.rounds << o.lanes;
}

// A call as the order sees it.
struct OrderShape {
  int32_t heads, group;  // query tiles side by side, of them per kv head
  int32_t batch;
  int32_t ragged;        // rows a sixteenth (1) or a quarter (2) below batch * longest, or 0
  int32_t qtiles;        // query tiles of the longest sequence
  int32_t chunks;        // KV chunks of a split call, or 1
  int64_t live;          // workgroups with work, estimated from the rows
  int64_t slots;         // resident workgroups
  bool windowed;         // a window bounds every query tile's keys
  bool proj;             // fused projection
};

// The order of a call.  Pairs suit equal lengths: every pair is the same work.  In a
// ragged batch of more work than the chip holds at once the busiest XCD sets the time,
// and work differs by sequence but not by head: heads go to XCDs then.  Units of four
// heads of one kv head (their K/V tiles come from HBM once) in the spread order; smaller
// groups in the linear order with its sequences turned, in the place of pairs.  Under a
// window all query tiles are alike, what is left is the K/V a unit shares, and units of
// three and four spread from about one workgroup per CU on.  (One box, us, before ->
// after; per-token bf16 bias of extent 1024 unless said; `proj`: the fused projection.)
//   spread  16 x 17..1900 tokens, Hq 8 / Hkv 2 134 -> 95, shared table 93.9 -> 61.8,
//           Hq 16 / Hkv 4 201 -> 186, Hq 8 / Hkv 1 171 -> 95; 12 x 500..1500, 8 / 2 74.8 ->
//           61.0; 8 x 100..1500 not causal 95.0 -> 65.6, causal 58.2 -> 57.4; proj 16 x
//           17..1900 122.8 -> 94.2, 24 x 50..800 60.1 -> 52.4; window 511 over 100..4000
//           keys 9 x 100..1000, 8 / 2 (448 live) 44.2 -> 38.8, 13 x 100..400 (240)
//           37.1 -> 36.2, 16 / 2 (480) 44.8 -> 39.1
//   turned  16 x 17..1900, Hq = Hkv = 4 93.3 -> 73.5, 6 / 3 97.5 -> 82.3, 8 / 4 134.7 ->
//           104.7 (spread in units of two: 118.9); proj 8 / 4 8 x 500..3000 144 -> 115
// What keeps the order of equal lengths, with what it would measure otherwise:
// workgroups all resident at once (spread 6 x 300..2000, 8 / 2, 456 live 61.9 -> 62.2,
// 9 x 50..1200, 392 40.5 -> 43.2; turned 16 x 100..700, 6 / 3, 395 28.4 -> 31.4; proj 10 x
// 100..600, 16 / 4, 256 of 256 40.6 -> 43.2, hence a quarter more there; window 511 6 x
// 150..600, 8 / 2, 184 29.7 -> 33.8; units of two, 7 x 200..1500, 8 / 4 without a cache 37.5 ->
// 49.6, 11 x 100..900 over 1000 44.2 -> 60.0); sequences of one query tile, which has no turn to
// take (64 x 45..90 queries over 1K..2K keys, 16 / 2 136.2 -> 139.4); groups above two in
// the turned order, whose heads then meet their K/V in several L2s (the same, 24 / 4 208
// -> 233; 200 x over 150..300, 6 / 2 58.1 -> 60.6); the turned order, and the projection,
// of lengths less than a quarter apart (32 x 400..520, 4 / 4 30.4 -> 31.5); the linear
// order, taken where pairs do not divide evenly, is not turned (12 x 500..1500, 6 / 3 61.0
// -> 63.8); split calls (chunks > 1: 3 x 333..512 tokens over 3K..9K keys 65.3 -> 69.0).
// A multiple of eight kv heads of one query head each is on the same XCD in the linear
// order as in pairs, so there turning is free and taken whatever the work (6 x 700..2048,
// d 64, 464 live 32.5 -> 31.4; 8 x 1000..2000, d 128 94.1 -> 80.5).
inline WorkgroupOrder workgroup_order(const OrderShape& c) {
  const bool pairs = (int64_t)c.batch * (c.heads / c.group) % 8 == 0;
  if (c.ragged > 0 && c.batch >= 6 && c.qtiles > 1 && c.chunks == 1) {
    const bool full = c.live >= (c.proj ? c.slots + c.slots / 4 : c.slots);
    const bool apart = c.ragged > 1;
    int32_t unit = c.group < 4 ? c.group : 4;
    while (c.group % unit != 0) --unit;
    const int32_t units = c.heads / unit;
    const int32_t xcds = units % 8 == 0 ? 1 : 8 % units == 0 ? 8 / units : 0;
    if (unit > 1 && xcds > 0 && c.batch >= xcds) {
      if (unit == 4 && full && (apart || !c.proj)) return spread_order(c.heads, unit, c.batch);
      if (c.windowed && unit > 2 && !c.proj && 16 * c.live >= 7 * c.slots)
        return spread_order(c.heads, unit, c.batch);
    }
    if (pairs && c.group <= 2 && full && apart) return linear_order(c.heads, c.batch, true);
    if (c.group == 1 && c.heads % 8 == 0 && !c.proj) return linear_order(c.heads, c.batch, true);
  }
  return pairs ? pairs_order(c.heads, c.group, c.batch) : linear_order(c.heads, c.batch, false);
}

}  // namespace ifa4
