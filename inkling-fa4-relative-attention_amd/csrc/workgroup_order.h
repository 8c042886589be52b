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

// The order of a call.  Pairs in fixed XCDs suit equal lengths
// (every pair the same work).  In a ragged batch the work differs by sequence
// but not by head, so heads go to XCDs instead, and a sequence's query tiles
// take turns on the XCDs of its heads: units of up to four heads of one kv head
// stay together (their K/V tiles come from HBM once), unit v of a sequence on
// XCDs v * spread .. + spread - 1.  Against pairs in fixed XCDs (one box, us;
// per-token bf16 bias of extent 1024 unless said): 16 x 17..1900 tokens,
// Hq 8 / Hkv 2 133.5 -> 93, shared table 93.9 -> 61.8, Hq 16 / Hkv 4 197 -> 183,
// Hq 8 / Hkv 1 171 -> 92; 12 x 1000..4096, shared table 249 -> 206.  Units of one
// head 136 and of two 100 on the first; one head of every kv head per XCD (the
// linear order) 100.  With one head per kv head there is no K/V to share, and
// the linear order, its sequences turned by one per query tile, is as fast or
// faster (Hq = Hkv = 4: 92.6 -> 72.2 against 75.7; 5 x 500..4000 over 4 heads 83
// against 88), as with fewer sequences than XCDs to take turns on, and for the
// KV chunks of a split call (3 x 333..512 tokens over 3K..9K keys: 65.3 against 69.0).
// Few sequences leave the equal-length order as it was: which of them meets which
// XCD is then a draw either way (3 x 126..1864 over Hq 16 / Hkv 4 38.2 in it, 42.9
// in this one; 5 x 409..768 over 4 heads 23.3 against 24.6).
inline WorkgroupOrder workgroup_order(int32_t heads, int32_t group, int32_t batch, bool ragged,
                                      int32_t chunks) {
  const bool pairs = (int64_t)batch * (heads / group) % 8 == 0;
  const bool turn = ragged && batch >= 6;
  if (turn && chunks == 1) {
    int32_t unit = group < 4 ? group : 4;
    while (group % unit != 0) --unit;
    const int32_t units = heads / unit;
    const int32_t xcds = units % 8 == 0 ? 1 : 8 % units == 0 ? 8 / units : 0;
    if (unit > 1 && xcds > 0 && batch >= xcds) return spread_order(heads, unit, batch);
    return linear_order(heads, batch, true);
  }
  return pairs ? pairs_order(heads, group, batch) : linear_order(heads, batch, turn);
}

}  // namespace ifa4
