// gfx950 tile table.  Replaces the per-arch Triton presets of
// src/inkling_fa4/autotune_configs.py:17-50 (seq-length buckets of
// BLOCK_Q/BLOCK_K/num_warps/num_stages for sm86/sm90/sm100).
//
// Prefill: one shape for every sequence length, and a sequence-length (grid)
// dependent split of the KV range (prefill_split_for, below).  The kernel is
// written for 4 waves x 32 query rows (BLOCK_Q 128) and 64-key KV tiles in two
// LDS stages (64 KiB of LDS at head_dim 128, so two workgroups fit in the 160
// KiB of a CU; 236 VGPRs, two waves per SIMD); the shape is a compile-time
// property of the kernel, listed here so the host reports what runs.  Swept on
// causal batch 8, Hq 8 / Hkv 2, d 128 at S 1024 / 2048 / 4096 / 8192
// (profiles/sweep_prefill_shapes_b8.md): BLOCK_K 64 x 4 waves 0.0314 / 0.0771 /
// 0.2646 / 0.9865 ms; 256-row workgroups of 8 waves +13 / +4.5 / +1.4 / +1.5%;
// 32-key tiles +9 / +6 / +6 / +6%; 64 rows per wave at one wave per SIMD
// (PREFILL_NQB 2) +79% at S 4096 (profiles/sweep_prefill_knobs_b8_s4096.md).
// SQ_VALU_MFMA_BUSY_CYCLES is the same for every variant and GRBM_GUI_ACTIVE
// follows the time: the shape sets how much of the MFMA work overlaps the
// softmax, not how much MFMA work there is.
//
// Decode: persistent waves of the stream-K pass (at most one per 32-key step).
#pragma once

#include <stdint.h>

namespace ifa4 {

struct PrefillTileEntry {
  int32_t head_dim;
  int32_t block_q;
  int32_t block_k;
  int32_t waves;
  int32_t stages;
};

constexpr PrefillTileEntry kPrefillTiles[] = {
    {64, 128, 64, 4, 2},
    {128, 128, 64, 4, 2},
};

// Persistent waves of the decode stream pass (at most; never more than the
// steps), from the sweep on the 64-sequence batch (KV 1K-16K, non-causal;
// profiles/sweep_decode_waves_b64.md, before the K/V loads were non-temporal;
// with them, profiles/sweep_decode_nt_b64.md: contiguous 896 waves 0.097 ms,
// 1536 0.103; paged 0.105 either way):
//   contiguous bf16: 896 waves 0.112 ms, 1024 0.112, 768 0.113, 2048 0.116,
//                    512 0.151 (too few bytes in flight);
//   paged (blocks of 16): 2048 0.120, 1024 0.121, 896 0.133, 768 0.149 -- a
//                    table-window refill stalls the wave, more waves hide it;
//   fp8 K/V: 2048 0.065, 3072 0.074, 1536 0.078, 1024 0.084 (half the bytes
//                    per step: more waves for the same bytes in flight).
#ifndef IFA4_DECODE_WAVES
#define IFA4_DECODE_WAVES 896
#endif
#ifndef IFA4_DECODE_WAVES_PAGED
#define IFA4_DECODE_WAVES_PAGED 2048
#endif
#ifndef IFA4_DECODE_WAVES_FP8
#define IFA4_DECODE_WAVES_FP8 2048
#endif
constexpr int64_t kDecodeWaves = IFA4_DECODE_WAVES;
constexpr int64_t kDecodeWavesPaged = IFA4_DECODE_WAVES_PAGED;
constexpr int64_t kDecodeWavesFp8 = IFA4_DECODE_WAVES_FP8;
constexpr int32_t kDecodeStep = 32;  // keys per step of a decode wave

// Upper bound of the 32-key steps of a decode call: every (sequence, kv head)
// at max_seqlen_k keys (one key when causal: top-left alignment, Lq = 1).
// key0_only: top-left causal decode, which sees key 0 only.
inline int64_t decode_max_steps(int64_t batch, int64_t kv_heads, int64_t max_seqlen_k,
                                bool key0_only) {
  const int64_t keys = key0_only ? (max_seqlen_k > 0 ? 1 : 0) : max_seqlen_k;
  return batch * kv_heads * ((keys + kDecodeStep - 1) / kDecodeStep);
}

// Small calls (few caches, or few steps): at least kDecodeMinSteps 32-key
// steps per wave, and at most kDecodeMaxParts waves per (sequence, kv head)
// cache -- or, for caches longer than kDecodeMaxParts * kDecodePartSteps
// steps, one wave per kDecodePartSteps steps.  With the combine split over
// several workgroups for many-part segments, a part of 2 steps (the same as the
// floor per wave, which then is the binding cap) measured fastest: one
// sequence of 16K / 32K / 64K keys 14.8 / 21.2 / 23.6 -> 12.9 / 15.8 / 21.3 us
// (8 steps per part before), fp8 cache 32K 21.9 -> 15.0, paged 32K 30.0 -> 18.6;
// 8K, 128K and the 64-sequence batch unchanged.  Same-session sweeps, Hq 8 /
// Hkv 2, d 128, non-causal (profiles/sweep_decode_small.md).
#ifndef IFA4_DECODE_MIN_STEPS
#define IFA4_DECODE_MIN_STEPS 2
#endif
#ifndef IFA4_DECODE_MAX_PARTS
#define IFA4_DECODE_MAX_PARTS 128
#endif
#ifndef IFA4_DECODE_PART_STEPS
#define IFA4_DECODE_PART_STEPS 2
#endif
constexpr int64_t kDecodeMinSteps = IFA4_DECODE_MIN_STEPS;
constexpr int64_t kDecodeMaxParts = IFA4_DECODE_MAX_PARTS;
constexpr int64_t kDecodePartSteps = IFA4_DECODE_PART_STEPS;

// fp8 caches of d 128 (contiguous or paged) whose kv heads sit side by side in
// every row (head stride = head_dim) stream their kv heads in pairs, one wave
// over whole rows of both (a pair holds at most 8 query heads); the kernel
// then sees half the kv heads, twice the group and 32-key steps of twice the
// bytes.
#ifndef IFA4_DECODE_FP8_PAIRS
#define IFA4_DECODE_FP8_PAIRS 1
#endif
#ifndef IFA4_DECODE_WAVES_FP8_PAIR
#define IFA4_DECODE_WAVES_FP8_PAIR 1024
#endif
constexpr int64_t kDecodeWavesFp8Pair = IFA4_DECODE_WAVES_FP8_PAIR;
// (paged: 1536, as for one kv head per wave more waves hide the block-table
// window refills; batch 64 at blocks of 16, one box: 64.5 us at 1024, 59.6 at
// 1536, 60.4-60.9 at 2048, against 66.0 streaming one kv head per wave)
#ifndef IFA4_DECODE_WAVES_FP8_PAIR_PAGED
#define IFA4_DECODE_WAVES_FP8_PAIR_PAGED 1536
#endif
constexpr int64_t kDecodeWavesFp8PairPaged = IFA4_DECODE_WAVES_FP8_PAIR_PAGED;
inline bool decode_pairs(bool fp8, int64_t head_dim, int64_t kv_heads, int64_t group,
                         int64_t k_stride_h, int64_t v_stride_h) {
  return IFA4_DECODE_FP8_PAIRS && fp8 && head_dim == 128 && kv_heads % 2 == 0 &&
         2 * group <= 8 && k_stride_h == head_dim && v_stride_h == head_dim;
}

// Short caches: one launch with a workgroup of 8 waves per (sequence, kv head)
// (4 for groups above 8) instead of the stream and combine passes.  A wave's
// steps wait for one another's loads (about 2 us each), so it pays up to three
// steps a wave (a window of 512 keys is 17 steps), and up to four where the
// segments alone fill the chip.  Two passes -> one launch (one box, us, Hq 8 /
// Hkv 2, d 128; sequences x keys):
//   bf16 1 x 300..600 14.2 -> 9.0, 64 x 300..600 18.3 -> 12.6, 128 x 100..200 16.5 -> 8.8,
//   128 x 512 26.5 -> 15.3, 64 x 500..1000 22.3 -> 18.8, 128 x 1024 39.6 -> 25.4, but 16 x
//   1024 14.1 -> 16.2, 16 x 2048 16.2 -> 27.0;
//   paged 64 x 250..500 18.1 -> 13.4, fp8 18.0 -> 13.9, window 511 over 200..6000 paged
//   keys 24 sequences 15.8 -> 14.2, 64 20.8 -> 15.2; window 1023 (33 steps) 16.9 -> 21.1.
// With 4 waves a segment everything but 64 x 256 is slower (64 x 512 13.4, windows 18.5).
// Groups above 8 take half the waves: their Q rows and tiles fill the LDS.
constexpr int64_t decode_whole_waves(int64_t group) { return group > 8 ? 4 : 8; }
inline bool decode_whole(int64_t segments, int64_t group, int64_t max_steps) {
  const int64_t waves = decode_whole_waves(group);
  if (2 * max_steps <= 5 * waves) return true;
  return max_steps <= 4 * waves && segments >= 128;
}

// kv_heads: as the kernel sees them (pairs when pair is set).
inline int32_t decode_waves_for(int64_t batch, int64_t kv_heads, int64_t max_seqlen_k,
                                bool key0_only, bool fp8, bool paged, bool pair = false) {
  const int64_t t = decode_max_steps(batch, kv_heads, max_seqlen_k, key0_only);
  int64_t w = kDecodeWaves;
  if (paged && kDecodeWavesPaged > w) w = kDecodeWavesPaged;
  if (fp8 && kDecodeWavesFp8 > w) w = kDecodeWavesFp8;
  if (pair) w = paged ? kDecodeWavesFp8PairPaged : kDecodeWavesFp8Pair;
  const int64_t by_steps = (t + kDecodeMinSteps - 1) / kDecodeMinSteps;
  const int64_t seg_steps = batch * kv_heads > 0 ? t / (batch * kv_heads) : 0;
  const int64_t long_parts = (seg_steps + kDecodePartSteps - 1) / kDecodePartSteps;
  const int64_t by_parts =
      batch * kv_heads * (long_parts > kDecodeMaxParts ? long_parts : kDecodeMaxParts);
  if (by_steps < w) w = by_steps;
  if (by_parts < w) w = by_parts;
  return (int32_t)w;
}

// Split KV for prefill calls whose grid leaves the chip underfilled (few
// sequences or heads, short sequences): the longest query tile's KV range is
// the critical path, so when it exceeds the work one slot would get with
// perfect balance, every query tile's range is cut into chunks of that many
// tiles (at least kPrefillMinChunk), one workgroup per chunk, and a second pass
// merges the chunks' partials by log-sum-exp.  The chunk is then lengthened
// until the chunks with work fit the resident slots at once: with the balanced
// share, a query tile's last chunk is short and the count overshoots the slots
// a little (528 for one sequence of 4096 over 4 heads), and the few left over
// ran as a second round.  Fitted, against the balanced share (same session):
// one sequence over 4 heads, S 4096 / 8192: 61.6 -> 48.6, 141.6 -> 109.5 us;
// 8 x 1024: 39.5 -> 36.2; 4 x 2048: 59.5 -> 50.0; 2 x 4096 over 4 heads and
// 1 x 4096 over 8: 90.7 -> 74.2 (S 1024 / 2048 fit already: unchanged).
// Where splitting pays (same-session sweeps with the balanced share, per-token
// bf16 bias of extent 1024, Hq = Hkv, causal):
//   * grids of at most a quarter of the resident slots always: one sequence
//     over 4 heads, S 1024 / 2048 / 4096: 45.4 -> 22.2, 71.9 -> 31.3,
//     104.9 -> 65.8 us;
//   * grids of up to half of them when the longest range is at least
//     kPrefillSplitWideMinTiles: batch 8 x 1024 over 4 heads (256 workgroups,
//     16 tiles) 53.4 -> 43.3 us, 4 x 2048 73.1 -> 63.7, 1 x 8192 172.5 -> 147.7;
//     with 8-tile ranges the merge costs more than it saves (16 x 512: 30.6 ->
//     31.9 us; the shared-table 8 x 512 over 8 heads: 18.0 -> 28.8);
//   * with fitted chunks, grids below the slots too, when the chunk is at most
//     half of the longest range or shortens it by kPrefillSplitMinSaved tiles
//     (against no split, same session): 3 x 4096 over 4 heads (384 workgroups,
//     chunk 44 of 64 tiles) 112.3 -> 104.8 us, 5 x 2048 (16 of 32) 71.4 ->
//     61.5, 1 x 8192 over 6 (86 of 128) 185.5 -> 170.3, 5 x 1024 over 8 (8 of
//     16) 48.2 -> 41.5; at 22 of 32 (6 x 2048, 3 x 2048 over 8) equal, at 12 of
//     16 (12 x 1024) 1% slower, at 14 of 16 (7 x 1024 over 8) 12% slower;
//   * never at the slots and above: every grid of 512 workgroups measured lost
//     (8 x 1024 over 8 heads 32.0 -> 45.6 us, 1 x 16384 over 4 heads 373 -> 447,
//     2 x 8192 206 -> 225), and no chunk fits the slots there.
// The estimate assumes every sequence holds max_seqlen_q queries over
// max_seqlen_k keys (top-left); it only steers performance, any chunk size
// gives the same results up to rounding.  kPrefillSlots: resident workgroups
// of the prefill kernel on MI355X (256 CUs x 2).
constexpr int64_t kPrefillSlots = 512;
// Shortest chunk: 2 tiles (against 4, one sequence over 4 heads, same session:
// S 384 / 512 / 1024 18.6 -> 14.3, 18.5 -> 14.7, 20.4 -> 18.8 us; 3 tiles in
// between).
#ifndef IFA4_PREFILL_MIN_CHUNK
#define IFA4_PREFILL_MIN_CHUNK 2
#endif
constexpr int32_t kPrefillMinChunk = IFA4_PREFILL_MIN_CHUNK;
#ifndef IFA4_PREFILL_SPLIT_MAX_GRID
#define IFA4_PREFILL_SPLIT_MAX_GRID 511
#endif
constexpr int64_t kPrefillSplitMaxGrid = IFA4_PREFILL_SPLIT_MAX_GRID;  // below kPrefillSlots
// A split is taken when its chunk is at most half of the longest KV range, or
// shortens that range by at least this many tiles.
#ifndef IFA4_PREFILL_SPLIT_MIN_SAVED
#define IFA4_PREFILL_SPLIT_MIN_SAVED 16
#endif
constexpr int64_t kPrefillSplitMinSaved = IFA4_PREFILL_SPLIT_MIN_SAVED;
constexpr int64_t kPrefillSplitSmallGrid = 128;                        // kPrefillSlots / 4
// Chunk length as a percentage of the balanced share (sweep knob).
#ifndef IFA4_PREFILL_CHUNK_PCT
#define IFA4_PREFILL_CHUNK_PCT 100
#endif
constexpr int64_t kPrefillChunkPct = IFA4_PREFILL_CHUNK_PCT;
// Lengthen the chunk until every chunk with work is resident at once (1), or
// keep the balanced share (0; sweep knob).
#ifndef IFA4_PREFILL_CHUNK_FIT
#define IFA4_PREFILL_CHUNK_FIT 1
#endif
constexpr int64_t kPrefillSplitWideMinTiles = 16;

struct PrefillSplit {
  int32_t chunk_tiles;  // 0: no split
  int32_t n_chunks;     // chunk slots per query tile in the grid
  int32_t seen_chunks;  // of them, those a query tile with pruned tiles can need
};

// Masks of a call: a sequence's query 0 sits at key position qpos.
struct PrefillMasks {
  bool causal;
  int64_t window_left;  // -1: none
  int64_t qpos;
};
// The masks a plan goes by.  It takes the longest cache for every sequence and,
// bottom-right without a window, every key for every query (the causal mask takes max_q
// keys at most).
inline PrefillMasks plan_masks(bool causal, int64_t window_left, bool bottom_right, int64_t max_q,
                               int64_t max_k) {
  return PrefillMasks{causal && !(bottom_right && window_left < 0), window_left,
                      bottom_right && max_k > max_q ? max_k - max_q : int64_t(0)};
}
// Keys [kbeg, kend) that queries [q0, q_hi) of a sequence over lk keys see.
inline void prefill_keys(int64_t q0, int64_t q_hi, int64_t lk, const PrefillMasks& m,
                         int64_t* kbeg, int64_t* kend) {
  *kend = m.causal && q_hi + m.qpos < lk ? q_hi + m.qpos : lk;
  *kbeg = m.window_left >= 0 && q0 + m.qpos > m.window_left ? q0 + m.qpos - m.window_left : 0;
}

// Packed rows: the query heads of a kv head share query tiles (block_q / group
// queries x group heads) when every sequence fits one tile of block_q queries and
// packing leaves at most three quarters of the tiles.  A sequence of a few
// queries otherwise takes one workgroup per head with one or two of its four
// waves at work, each streaming the same K/V.
inline bool prefill_can_pack(int64_t group, int64_t max_q, int64_t block_q) {
  if (group <= 1 || group > block_q || max_q <= 0 || max_q > block_q) return false;
  const int64_t step = block_q / group;
  return 4 * ((max_q + step - 1) / step) <= 3 * group;
}

// It pays where the call has more work than it has room for (grid: workgroups without
// it, key_tiles: of the longest range): a call whose workgroups are all resident at
// once and short is one range long either way, and packed rows fill that range's
// waves or cut it into chunks and a merge pass.  So it packs
//   - more workgroups than fit at once: 200 x 8 queries 20.8 -> 7.4 us, x 64 26.0 -> 21.3,
//     64 x 17..96 over Hq 16 / Hkv 2 21.2 -> 19.7;
//   - ranges of 16 tiles on, where half of the 32-row waves go (12 x 2..5 queries over
//     1K..8K keys 42.4 -> 22.9, 4 x 16 over 14K 31.6 -> 22.6), or the ranges together
//     are 6000 tiles of up to 32 queries, or of any if they are 64 on, or 3000 if 128 on (16
//     x 32 over 8K 64.3 -> 46.1, 64 x 24 over 2K 57.3 -> 43.1, 4 x 64 over 14K 41.6 -> 34.8, 3 x
//     20..40 over 3K..9K 26.7 -> 22.3, x 50..96 30.9 -> 28.9);
//   - where three quarters of the waves go and the bias is per token: 64 x 2 over 500
//     keys 17.5 -> 14.3 (shared table, whose tiles are cheap, x 8 14.3 -> 15.9).
// Without one of these it measured (packed against not): 64 x 32 over 500 keys 20.4 ->
// 25.9, 64 x 96 28.9 -> 32.4, 64 x 64 over 2K 71.1 -> 73.5, 16 x 24 without a cache 6.6 ->
// 7.1, 64 x 17..96 12.4 -> 13.5 (shared table 10.9 -> 13.3), 4 x 64 over 4K 23.2 -> 26.2.
// (One box, Hq 8 / Hkv 2, d 128, per-token bf16 bias unless said.)
inline bool prefill_packs(int64_t grid, int64_t key_tiles, int64_t group, int64_t max_q,
                          bool table) {
  const int64_t waves = group * ((max_q + 31) / 32), packed = (max_q * group + 31) / 32;
  if (grid > kPrefillSlots) return true;
  const int64_t enough = key_tiles >= 128 ? 3000 : 6000;
  if (key_tiles >= 16 &&
      (2 * packed <= waves || (grid * key_tiles >= enough && (max_q <= 32 || key_tiles >= 64))))
    return true;
  return !table && 4 * packed <= waves && grid * key_tiles >= 512;
}

// Tiles of the longest query tile and of all query tiles of one (sequence,
// head), for a sequence of lq queries over lk keys.
inline void prefill_tile_work(int64_t lq, int64_t lk, const PrefillMasks& m, int32_t block_q,
                              int32_t block_k, int64_t* tmax, int64_t* total) {
  *tmax = 0;
  *total = 0;
  for (int64_t q0 = 0; q0 < lq; q0 += block_q) {
    int64_t kbeg, kend;
    prefill_keys(q0, q0 + block_q < lq ? q0 + block_q : lq, lk, m, &kbeg, &kend);
    const int64_t t = kend > kbeg ? (kend + block_k - 1) / block_k - kbeg / block_k : 0;
    if (t > *tmax) *tmax = t;
    *total += t;
  }
}

// Chunks with work of one (sequence, head) when the KV range of every query
// tile is cut at multiples of `chunk` key tiles (the kernel's alignment).
inline int64_t prefill_chunk_count(int64_t lq, int64_t lk, const PrefillMasks& m,
                                   int32_t block_q, int32_t block_k, int64_t chunk) {
  int64_t n = 0;
  for (int64_t q0 = 0; q0 < lq; q0 += block_q) {
    int64_t kbeg, kend;
    prefill_keys(q0, q0 + block_q < lq ? q0 + block_q : lq, lk, m, &kbeg, &kend);
    if (kend <= kbeg) continue;
    n += ((kend + block_k - 1) / block_k - 1) / chunk - (kbeg / block_k) / chunk + 1;
  }
  return n;
}

// The slots a split may fill and when it pays, per kernel.
struct SplitRule {
  int64_t slots;       // resident workgroups
  int64_t small_grid;  // grids up to here split whatever the range
  int64_t min_saved;   // else a chunk of at most half of it, or this many tiles saved
  int64_t min_tiles;   // shorter ranges do not split
};
constexpr SplitRule kPrefillSplitRule = {kPrefillSlots, kPrefillSplitSmallGrid,
                                         kPrefillSplitMinSaved, 0};
// Fused projection: one 256-row workgroup per CU, and a tile in the bias band costs
// it about 3 us, so any underfilled grid splits when that saves four tiles of a range of
// eight.  Whole calls without and with the split (one box, us, Hq 8 / Hkv 2, d 128, extent
// 1024, bf16 r): 2 x 900..2100 tokens 86.0 -> 51.1, 1 x 1000 66.5 -> 32.8, 1 x 3000 117 ->
// 78, 3 x 100..600 over 300..2000 keys bottom-right 102.5 -> 61.8, window 255 6 x 300..400
// (nine tiles) 41.5 -> 38.0, 3 x 2000 98.7 -> 93.0 (98.0 when 16 tiles had to be saved), 6 x
// 1200 (240 workgroups, no split) 76.  Shorter ranges, split: 6 x 50..300 (five tiles) 24.0 ->
// 25.9, 10 x 200 (four) 23.7 -> 29.7, 6 x 300..400 (six or seven) 28.4 -> 31.7, Hq 16 / Hkv 4
// 28.4 -> 35.8.
constexpr SplitRule kProjSplitRule = {256, 256, 4, 8};

// Tiles of the longest range from which a windowed bottom-right call splits: the merge
// pass costs about as much as four tiles of a per-token bias (2 us each) or six of a shared
// table, and the more the more workgroups there are.  Split against not, by workgroups
// without the split and tiles (one box, us, bf16 bias; t: shared table):
//     4..12   4 tiles 12.3 / 11.6   5 13.5 / 15.0   7 13.4 / 17.3   t 5 12.7 / 12.1   t 6 11.9 / 12.7
//    16..24   4 14.0 / 12.2         5 14.7 / 15.0   7 15.0 / 17.8   t 6 13.9 / 12.9   t 7 14.6 / 15.0
//    32..48   4 14.6 / 12.1         5 14.7 / 14.2   6 14.7 / 15.9   t 6 12.2 / 12.5   t 8 12.6 / 15.0
//    64..128  4 18.2 / 12.8         7 22.2 / 19.1   9 24.9 / 23.4   t 9 24.3 / 18.0   t 11 26.0 / 20.6
//   144..288                                                       t 18 37.7 / 29.5  t 19 32.5 / 31.0
inline int64_t window_split_tiles(int64_t grid, bool table) {
  if (table) return grid < 16 ? 6 : grid < 32 ? 7 : grid < 64 ? 8 : grid <= 128 ? 12 : 32;
  return grid < 32 ? 5 : grid < 64 ? 6 : 10;
}
// Shortest chunk of such a call from 64 workgroups on (chunks of two tiles against four:
// window 511 8 x 128 queries over 1.5K keys 25.8 -> 23.6, window 700 4 x 256 with a
// shared table 28.0 -> 22.4, window 1023 1 x 1000 over 200 keys 24.7 -> 26.8).
constexpr int64_t kWindowMinChunk = 4;

// bottom_right: the queries are the last of their sequence's keys.  The estimate
// takes the longest cache for every sequence and, without a window, every key for
// every query (the causal mask takes max_q keys at most).  With a window the
// ranges are short wherever the queries sit: counting them so (instead of the
// whole cache, us on one box): 3 x 300..500 queries, window 511, over 100..4000
// keys 37.7 -> 27.3, 1 x 1000 32.9 -> 23.1, 6 x 20..40 21.9 -> 15.3.
// no_prune: masked tiles are visited too (debug).  forced_chunk > 0: split every query
// tile into chunks of that many tiles.  table: the bias is a shared table.
inline PrefillSplit prefill_split_for(int64_t batch, int64_t n_heads, int64_t max_q,
                                      int64_t max_k, bool causal, int64_t window_left,
                                      bool bottom_right, bool no_prune, int32_t block_q,
                                      int32_t block_k, int32_t forced_chunk, bool table,
                                      const SplitRule& rule = kPrefillSplitRule) {
  PrefillSplit s{0, 1, 1};
  if (batch <= 0 || max_q <= 0 || max_k <= 0) return s;
  PrefillMasks masks = plan_masks(causal, window_left, bottom_right, max_q, max_k);
  int64_t tmax = 0, total = 0;
  prefill_tile_work(max_q, max_k, masks, block_q, block_k, &tmax, &total);
  int64_t chunk = forced_chunk;
  if (chunk <= 0) {
    const int64_t grid = (max_q + block_q - 1) / block_q * n_heads * batch;
    if (grid >= rule.slots || grid > kPrefillSplitMaxGrid) return s;
    if (tmax < rule.min_tiles) return s;
    bool windowed = bottom_right && window_left >= 0 && rule.min_tiles == 0;
    if (windowed && tmax < window_split_tiles(grid, table)) return s;
    if (grid > rule.small_grid && tmax < kPrefillSplitWideMinTiles) return s;
    if (windowed && 3 * (block_q + window_left) > 2 * max_k) {
      // The window covers most of the cache: planned over all of it, in longer chunks
      // (ranges of the window against it: window 1500, 2 x 2000 queries over 200 keys, Hq =
      // Hkv = 4 40.0 -> 35.8; window 1023, 3 x 1000 over 200 43.7 -> 40.0, 30 x 128 over 1.5K,
      // 4 heads 49.7 -> 45.1).
      windowed = false;
      masks = PrefillMasks{false, -1, 0};
      prefill_tile_work(max_q, max_k, masks, block_q, block_k, &tmax, &total);
    }
    const int64_t balanced =
        ((total * batch * n_heads + rule.slots - 1) / rule.slots * kPrefillChunkPct + 99) / 100;
    const int64_t least = windowed && grid >= 64 ? kWindowMinChunk : kPrefillMinChunk;
    chunk = balanced > least ? balanced : least;
    if (IFA4_PREFILL_CHUNK_FIT && chunk < tmax) {
      // Chunks of the balanced share can number a little more than the slots
      // (each query tile's last chunk is short): the few left over then run as
      // a second round.  Take the shortest chunk whose workgroups all fit
      // (binary search; the count falls as the chunk grows).
      auto fits = [&](int64_t c) {
        return prefill_chunk_count(max_q, max_k, masks, block_q, block_k, c) * batch * n_heads <=
               rule.slots;
      };
      if (!fits(chunk)) {
        // hi = tmax: one chunk per query tile whose range starts at key 0, which
        // the grid (below the slots) fits; otherwise the search ends there and
        // the call is not split
        int64_t lo = chunk, hi = tmax;
        while (hi - lo > 1) {
          const int64_t mid = lo + (hi - lo) / 2;
          if (fits(mid)) hi = mid; else lo = mid;
        }
        chunk = hi;
      }
    }
    // A split that shortens the longest range by little does not repay the
    // chunks' partials and the merge pass.
    if (tmax <= chunk || (2 * chunk > tmax && tmax - chunk < rule.min_saved)) return s;
  }
  // chunk slots: enough for a query tile that meets every key tile (chunks are
  // aligned to multiples of `chunk` tiles on the key axis), so the grid and the
  // workspace cover whatever the masks, lengths and alignment of a sequence; a
  // window and the causal mask together leave a query tile block_q + window_left
  // keys wherever it sits, which any alignment cuts into one chunk more
  const int64_t key_tiles = (max_k + block_k - 1) / block_k;
  s.chunk_tiles = (int32_t)chunk;
  s.n_chunks = (int32_t)((key_tiles + chunk - 1) / chunk);
  if (s.n_chunks < 1) s.n_chunks = 1;
  s.seen_chunks = s.n_chunks;
  if (causal && window_left >= 0) {
    const int64_t span = (block_q + window_left + block_k - 1) / block_k + 1;  // tiles
    const int64_t slots = (span + chunk - 1) / chunk + 1;
    if (slots < s.n_chunks) s.seen_chunks = (int32_t)slots;
    if (!no_prune) s.n_chunks = s.seen_chunks;
  }
  return s;
}

}  // namespace ifa4
