// Which kernel a call takes, from its sizes alone.  Plain host code without HIP
// types, so that the rules can be checked on a machine without a GPU
// (tests/test_dispatch_rules.py).
#pragma once

#include <cstddef>

namespace qd {

constexpr int kPfQ = 16;   // queries per workgroup of prefill_exact_kernel

inline long long rounds_of(long long workgroups, int cus) { return (workgroups + cus - 1) / cus; }

// Blocks of 16 lengths that `tokens` queries over seqlen rows on touch.
inline int prefill_blocks(int seqlen, int tokens) {
  return (seqlen - 1 + tokens - 1) / kPfQ - (seqlen - 1) / kPfQ + 1;
}

// Whether the fused plans of `tokens` queries over seqlen rows on share their rows
// in blocks of 16 queries (prefill_exact_kernel) or are scanned one by one.  Both
// put one workgroup on a CU at a time, so what decides is how many rounds of the
// device each takes: a round of the shared form lasts as long as about four of the
// scan's, and a little longer from 129 rows on.  Whole calls on 256 CUs, scan /
// shared us: 16 heads 48 queries (3 rounds) 7.3 / 7.6, 56 (4) 8.8 / 7.7, 128 (8)
// 16.3 / 9.3; 8 heads 64 (2) 5.7 / 7.7, 128 (4) 9.3 / 9.2; 4 heads 128 (2) 6.0 /
// 9.2; 64 heads 12 (3) 7.2 / 7.1; 12 heads 60 after 164 rows (3) 9.8 / 13.0, 100
// after 124 (5) 13.9 / 13.0.
inline bool prefill_shares_fused(int heads, int seqlen, int tokens, int cus) {
  const long long scan = rounds_of((long long)heads * tokens, cus);
  const long long shared = rounds_of((long long)heads * prefill_blocks(seqlen, tokens), cus);
  return scan >= (seqlen + tokens - 1 > 128 ? 5 : 4) * shared;
}

// The same for split plans.  The shared form's time is that of a block of 16
// however few they are, and the two cross where heads x rows x queries is about
// 90000.  Scan / shared us, each with the same merge: 16 heads after 300 rows 10.2 /
// 10.3 at 12 queries, 11.8 / 10.5 at 16; after 1000 7.7 / 9.2 at 4, 9.8 / 9.3 at 8,
// 14.0 / 11.3 at 16; 4 heads after 1000 10.7 / 12.0 at 12, 15.5 / 12.4 at 24; after
// 4000 10.0 / 9.8 at 4, 12.9 / 10.0 at 8; 1 head after 1000 11.9 / 13.7 at 48, after
// 4000 16.4 / 17.3 at 8, 21.0 / 19.8 at 16.  Three kinds of calls cross later:
//   * 6 and 7 queries (20 heads after 1000 rows 11.5 / 12.7, 16 heads 8.8 / 9.2);
//   * few queries on both sides of a block's edge, which pay for two blocks (64
//     heads, 8 queries after 300 rows 12.3 / 14.8);
//   * more than 64 heads: a plan then holds for fewer than 16 lengths, and the runs
//     of one plan in a block go one after another (128 heads, 16 queries after 128
//     rows 20.2 / 24.1).
inline bool prefill_shares_split(int heads, int seqlen, int tokens, int cus) {
  if (tokens < 6) return false;
  long long need = tokens < 8 ? 150000 : 90000;
  if (tokens < 5 * prefill_blocks(seqlen, tokens)) need = 300000;
  if (cus / heads < 4) need = 350000;
  return (long long)heads * seqlen * tokens >= need;
}

// Whether the partials of `tokens` queries are folded by a wave per (query, head)
// (prefill_merge_kernel) or by a workgroup (decode_attention_merge_kernel).  The wave
// adds its splits one after another, so it needs enough waves to read for all of them;
// the workgroup has each slice's sums in its own threads and is the faster one until
// the workgroups queue.  Whole calls, workgroup / wave us: 16 splits (16 heads) 1 query
// after 1000 rows 6.2 / 6.5, 64 queries 32.8 / 34.8, 128 52.0 / 53.6, 256 89.7 / 88.4;
// 8 splits (32 heads, 300 rows) 16 queries 11.9 / 12.1, 128 37.6 / 35.6, 256 80.7 / 74.5;
// 4 splits (64 heads, 600 rows) 32 queries 31.6 / 29.7.  Over 17 and more splits the
// wave's registers for all loads cost more than they gain: 32 splits (8 heads) 1 query
// after 1000 rows 6.0 / 7.2; 64 (4 heads) 6.3 / 8.7, 256 queries 48.5 / 52.3.
constexpr int kWaveMergeSplits = 16;
inline bool prefill_merges_by_wave(int heads, int tokens, int splits) {
  return splits <= kWaveMergeSplits && (long long)heads * tokens >= 192LL * splits;
}

// Whether an exact product of `tokens` rows with n weight rows of K goes to the two-row
// FMA kernel (gemv_batched_kernel), which reads each weight row once and little else, or
// to the fp32 matrix instructions.  Up to 4 tokens the first: two-row / matrix us at 4 /
// 6 / 16 tokens, cold weights, 9.1 / 10.1 / 16.0 against 10.3 / 10.3 / 10.4 (6144 x
// 2048), 5.8 / 6.5 / 10.4 against 6.1 / 6.0 / 6.2 (2048 x 2048), 10.6 / 12.7 / 22.0
// against 11.3 / 11.2 / 11.4 (2048 x 5504).  From K = 7169 its workgroups have four waves,
// no prefetch and a CU to themselves, so it stays the faster one only while they all run
// at once: 1 / 4 tokens, K = 7176, 1024 rows 8.2 / 11.9 against 13.0 / 12.9, 2048 rows
// 9.7 / 13.4 against 14.3 / 14.1, 4096 rows 17.7 / 24.6 against 17.1 / 15.6.
// With a few tokens more it is still ahead on both sides of the usual widths.  Up to 128
// weight rows, K = 256 to 5632, the matrix kernel's few workgroups only wait: 5 tokens 98 x
// 1928 5.4 against 6.0, 6 tokens 3 x 1416 4.1 and 4.8, but 5 tokens 176 x 3176 8.9 and 7.0.
// Past one 32 x 32 tile per CU the matrix kernel's next round is not paid for where K is
// short: 6 tokens 9997 x 240 5.6 and 6.8, 10219 x 936 8.9 and 10.0, but 6931 x 624 6.8 and
// 6.0; 8 tokens 11530 x 440 7.0 and 8.0, but 11773 x 552 8.6 and 8.0.
constexpr int kWideTwoRowWg = 8;   // weight rows per workgroup of the two-row kernel from K = 7169
inline bool exact_two_rows(int tokens, int n, int k, int cus) {
  if (tokens > 8) return false;
  if (tokens > 4 && n > 32 * cus) return tokens <= 6 ? k > 128 && k <= 1024 : k > 256 && k <= 512;
  if (tokens > 4) return tokens <= 6 && n <= 128 && k > 256 && k <= 5632;
  return k <= 7168 || (n + kWideTwoRowWg - 1) / kWideTwoRowWg <= cus;
}

// The matrix-core tile of a product that takes neither ring tile, over `rows` weight
// rows (both weights' in the gate/up form, `paired`) and `tokens` of K: the one whose
// rounds of workgroups, one per CU, cost least.  A round costs a start and an end,
// whatever K, and a time per K tile of 64 (us, fitted to 1600 products of 16-40000 rows,
// 1-400 tokens and K = 64-5504, cold weights, every tile timed on each):
//   64 x 64                              1.7 + 0.33 per K tile
//   32 x 32 and 32 x 16, K over eight waves  1.9 + 0.10 in a single round, 0.16 in more
//   32 x 64, K over two groups           1.9 + 0.23
//   64 x 128, K over two groups          1.9 + 0.42
// With a residual the 64-row tiles end later the more tokens they hold, as each lane
// reads it row by row: 0.03 us per token of 32, and 0.014 of 64 (20000 x 512, 32 tokens
// 9.7 us without, 14.6 with; on 32 x 32 tiles 10.6 and 11.0).  The tiles so chosen are
// 0.15% (with a residual 0.6%) slower than the best of the five on average; by the times
// per K tile alone they were 1.3% and up to 71% (the start decides where K is short and
// rows are many: 40000 x 64, 1 token 7.9 us on 64 x 64 tiles, 12.4 on 32 x 16).  Where a
// lane's four outputs cannot be stored together (`scalar`: y or its rows off 8 bytes), the
// 64 x 128 tile ends later still, as its lanes hold tokens and the 64 x 64 tile's hold
// adjacent outputs: 0.022 us per token of 128, 0.012 with a residual, nothing measurable
// for a pair's half as many (1367 tokens 2010 x 64 13.8 us, 10.2 on 64 x 64 tiles; 403
// 5123 x 448 17.2 and 14.8).  Over 360 such products of 6 us and more the choice is
// then 0.5% (residual 0.7%) slower than the best tile on average, 4.1% (1.4%) without.
// Between equals the smaller tile, which has more of the device at work.
enum class ShortTile { k64, kWave32x16, kWave32x32, kGroup32x64, kGroup64x128 };

inline ShortTile short_tile(long long rows, int tokens, int k, bool paired, bool residual, bool scalar, int cus) {
  const long long kt = k / 64;
  const long long end64 = residual ? 30 * (tokens < 32 ? tokens : 32) : 0;
  const long long per_token = paired || !scalar ? 0 : residual ? 12 : 22;
  const long long end128 = (residual ? 14 * (tokens < 64 ? tokens : 64) : 0) + per_token * (tokens < 128 ? tokens : 128);
  auto rounds = [&](int tn, int tt) { return rounds_of((rows + tn - 1) / tn * ((tokens + tt - 1) / tt), cus); };
  auto wave = [&](int tn, int tt) { return rounds(tn, tt) * (1900 + (rounds(tn, tt) == 1 ? 100 : 160) * kt); };
  ShortTile best = ShortTile::kWave32x16;
  long long cost = wave(32, 16);
  auto take = [&](ShortTile t, long long c) {
    if (c < cost) {
      best = t;
      cost = c;
    }
  };
  take(ShortTile::kWave32x32, wave(32, 32));
  if (!paired) take(ShortTile::kGroup32x64, rounds(32, 64) * (1900 + 230 * kt));
  take(ShortTile::k64, rounds(64, 64) * (1700 + end64 + 330 * kt));
  take(ShortTile::kGroup64x128, rounds(64, 128) * (1900 + end128 + 420 * kt));
  return best;
}

// Whether a product on `tiles` 128 x 128 tiles, one workgroup and CU each, shares K out over
// two slices, folded by a second launch: where both slices of every tile run at once.  That
// tile is taken from half of the CUs on (pick_tile), so this is exactly half of them: 897-1024
// tokens of 2048 rows, 385-512 of 4096, 1921-2048 of 1024.  Engine prompts, us a layer, one
// slice / two: 128 tiles on 256 CUs 237.6 / 221.7 (hidden 2048, FFN 5504, 1022 tokens), 337.0
// / 304.5 (4096, 8192, 510), 160.5 / 158.3 (2048, 2048); 144 tiles, where two slices take a
// second round, 258.7 / 275.4 (1100 tokens); 120 tiles, by then on the short tiles, 237.0 /
// 239.4 (1024, 8192, 1918), 231.3 / 237.4 (2560, 6912, 668).
inline bool ring_two_slices(long long tiles, int cus) { return 2 * tiles <= cus; }
// Bytes of the fp32 partials of two slices under that rule (16 MiB on 256 CUs).
inline size_t ring_two_slice_bytes(int outputs_per_tile, int cus) {
  return (size_t)(cus / 2) * 2 * outputs_per_tile * sizeof(float);
}

}  // namespace qd
