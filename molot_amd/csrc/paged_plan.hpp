// Chunks of a paged batch on the matrix-core kernel (attn_mfma_kernel): the
// rule every wave evaluates over the sequences' lengths, and the host's bounds
// of what it can give.  Plain C++ besides the device attribute.
#ifndef MOLOT_AMD_CSRC_PAGED_PLAN_HPP_
#define MOLOT_AMD_CSRC_PAGED_PLAN_HPP_

#include <cstdint>

#ifdef __HIPCC__
#define MOLOT_PLAN_HD __host__ __device__
#else
#define MOLOT_PLAN_HD
#endif

// The host knows only a bound of the longest sequence; a chunk sized from that
// left a batch of uneven lengths with either a second round of workgroups (two
// fit a CU) or a few long chunks.  Each wave instead sums the lengths (a load a
// lane, with the one it needs anyway) and takes the chunk that gives the
// launch's `target` workgroups, two a CU, in whole rounds of the 4 waves' 32-row
// tiles.  Batches with more than kDynLong rows a chunk then need several rounds
// and take dyn_round's rows (or, of short sequences, one chunk each).
// us a step, 32q/8kv/d128, chunks from the longest sequence against these: Q8
// 13 sequences of 1 .. 2999 rows 27.9 against 19.4; 2 of 3000 and 8000 31.4
// against 16.1; 20 of 31 .. 447 18.7 against 14.1; 64 of 100 .. 1000 32.9
// against 23.3; bf16 7 of 136 .. 2731 26.1 against 19.0; 2 of 3000 and 8000
// 49.3 against 19.2; 64 of 100 .. 1000 51.1 against 37.0; 32 of 512 .. 4096
// 76.0 against 72.3.
constexpr int kDynUnit = 128, kDynLong = 1024, kDynMax = 2048;

// a >= 0, b > 0 (an unsigned division: fewer instructions on the device)
MOLOT_PLAN_HD constexpr int dyn_ceil(int a, int b) {
  return (int)(((unsigned)a + (unsigned)b - 1u) / (unsigned)b);
}

// Rows a chunk of such batches: kDynRound; of Q8 rows, whose steps gain from
// longer chunks, 1024 and 1536 where the sequences have over 2 and over 4 times
// kDynLong rows on average.  us a step at 768, 1024 and 1536 rows, then with chunks
// from the longest sequence, 32q/8kv/d128 Q8: 48 sequences of 100 .. 3000 rows 46.6,
// 49.5, 47.6; 46.8.  32 of 4000 62.8, 55.1, 63.8; 59.3.  63 of 4000 130.0, 114.8,
// 117.2; 118.7.  24 of 12000 135.6, 131.9, 123.9; 130.9.  32 of 1000 .. 9000 84.9,
// 80.5, 77.3; 81.4.  d64, 48 of 12000 137.6, 135.5, 132.7; 129.6.  bf16: 32 of
// 512 .. 4096 63.6, 70.8, 62.4; 69.5.  32 of 1000 .. 9000 132.7, 133.8, 133.6;
// 133.9.  16q/2kv, 100 of 1000 .. 9000 115.7, 117.8, 121.9; 119.5.  64q/8kv, 32 of
// 4000 117.9, 109.9, 125.9; 123.5.
constexpr int kDynRound = 768, kDynLongQ8 = 1536;
MOLOT_PLAN_HD constexpr int dyn_round(int rows, int nseq, bool q8) {
  const unsigned r = (unsigned)rows, n = (unsigned)nseq * kDynLong;  // rows > n: no wrap below
  return !q8 || r <= 2 * n ? kDynRound : r <= 4 * n ? kDynLong : kDynLongQ8;
}

// Rows a chunk: rows = the sequences' attended rows in all.
MOLOT_PLAN_HD constexpr int dyn_chunk(int rows, int nseq, int heads, int target, bool q8) {
  const int den = target - nseq * heads;  // workgroups beyond one a (sequence, head)
  const int c = den > 0 ? dyn_ceil(rows * heads, den) : kDynMax;
  if (den > 0 && c <= kDynLong) return c <= kDynUnit ? kDynUnit : dyn_ceil(c, kDynUnit) * kDynUnit;
  return rows > kDynLong * nseq ? dyn_round(rows, nseq, q8) : kDynMax;
}
// Chunks of a sequence of `rows` attended rows (0: none).
MOLOT_PLAN_HD constexpr int dyn_chunks(int rows, int chunk) { return dyn_ceil(rows, chunk); }

// Bounds over every batch of nseq sequences of at most `span` attended rows
// each, whatever their lengths: chunks round up, so a total just below another's
// may take chunks half as long, and the bound of `span` itself would miss it.
// (The device counts a sequence's rows past span as span: seq_span.)
struct DynPlan {
  int nchunks;    // most chunks of a sequence
  int pairs;      // most (sequence, chunk) pairs, an empty sequence counting one
  int min_chunk;  // least rows a chunk
  int likely;     // several rounds: chunks of a sequence if all have `span` rows, else nchunks
};
// (B * span * heads < 2^30: plan_launch)
constexpr DynPlan dyn_plan(int span, int nseq, int heads, int target, bool q8) {
  const int64_t B = nseq;
  const int den = target - nseq * heads;
  // (in one round the chunks of an uneven batch's long sequences are as many as
  // the bound: 13 of 1 .. 2999 rows, Q8, 19.1 us, 19.5 from the likely ones)
  const int likely = dyn_ceil(span, dyn_chunk((int)(B * span), nseq, heads, target, q8));
  // more than kDynLong rows a chunk (dyn_round's then need a sequence of them)
  const int rounds = span > kDynLong ? dyn_ceil(span, kDynRound) : 1;
  // Q8: the chunks an average sequence's rows fill, and one more for an end
  int each = dyn_ceil(span, kDynLongQ8) < 4 ? 5 : dyn_ceil(span, kDynLongQ8) + 1;
  if (!q8 || each > rounds) each = rounds;
  if (den <= 0) return {rounds, (int)(B * each), span > kDynLong ? kDynRound : kDynMax, likely};
  // chunk >= rows * heads / den, so a sequence has at most den / heads of
  // them, and all together at most that many and one more each
  int n = dyn_ceil(span, kDynUnit);
  if (dyn_ceil(den, heads) < n) n = dyn_ceil(den, heads);
  int64_t pairs = B * n < target / heads ? B * n : target / heads;
  if (pairs < B) pairs = B;
  if (n < 1) n = 1;
  if (B * span * heads <= (int64_t)kDynLong * den) return {n, (int)pairs, kDynUnit, n};
  // dyn_chunk's c may pass kDynLong
  if (n < rounds) n = rounds;
  if (pairs < B * each) pairs = B * each;
  return {n, (int)pairs, kDynUnit, likely};
}

#endif  // MOLOT_AMD_CSRC_PAGED_PLAN_HPP_
