// Which kernel a call takes, from its sizes alone.  Plain host code without HIP
// types, so that the rules can be checked on a machine without a GPU
// (tests/test_dispatch_rules.py).
#pragma once

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
constexpr int kWideTwoRowWg = 8;   // weight rows per workgroup of the two-row kernel from K = 7169
inline bool exact_two_rows(int tokens, int n, int k, int cus) {
  if (tokens > 4) return false;
  return k <= 7168 || (n + kWideTwoRowWg - 1) / kWideTwoRowWg <= cus;
}

}  // namespace qd
