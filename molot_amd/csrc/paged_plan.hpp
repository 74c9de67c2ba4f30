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
// and take kDynRound rows (or, of short sequences, one chunk each).
// us a step, 32q/8kv/d128, chunks from the longest sequence against these: Q8
// 13 sequences of 1 .. 2999 rows 27.9 against 19.4; 2 of 3000 and 8000 31.4
// against 16.1; 20 of 31 .. 447 18.7 against 14.1; 64 of 100 .. 1000 32.9
// against 23.3; bf16 7 of 136 .. 2731 26.1 against 19.0; 2 of 3000 and 8000
// 49.3 against 19.2; 64 of 100 .. 1000 51.1 against 37.0; 32 of 512 .. 4096
// 76.0 against 72.3.
constexpr int kDynUnit = 128, kDynLong = 1024, kDynRound = 768, kDynMax = 2048;

// a >= 0, b > 0 (an unsigned division: fewer instructions on the device)
MOLOT_PLAN_HD constexpr int dyn_ceil(int a, int b) {
  return (int)(((unsigned)a + (unsigned)b - 1u) / (unsigned)b);
}

// Rows a chunk: rows = the sequences' attended rows in all.
MOLOT_PLAN_HD constexpr int dyn_chunk(int rows, int nseq, int heads, int target) {
  const int den = target - nseq * heads;  // workgroups beyond one a (sequence, head)
  const int c = den > 0 ? dyn_ceil(rows * heads, den) : kDynMax;
  if (den > 0 && c <= kDynLong) return c <= kDynUnit ? kDynUnit : dyn_ceil(c, kDynUnit) * kDynUnit;
  return rows > kDynLong * nseq ? kDynRound : kDynMax;
}
// Chunks of a sequence of `rows` attended rows (0: none).
MOLOT_PLAN_HD constexpr int dyn_chunks(int rows, int chunk) { return dyn_ceil(rows, chunk); }

// Bounds over every batch of nseq sequences of at most `span` attended rows
// each, whatever their lengths: chunks round up, so a total just below another's
// may take chunks half as long, and the bound of `span` itself would miss it.
// (The device counts a sequence's rows past span as span: dyn_rows.)
struct DynPlan {
  int nchunks;    // most chunks of a sequence
  int pairs;      // most (sequence, chunk) pairs, an empty sequence counting one
  int min_chunk;  // least rows a chunk
};
constexpr DynPlan dyn_plan(int span, int nseq, int heads, int target) {
  const int64_t B = nseq;
  const int den = target - nseq * heads;
  // more than kDynLong rows a chunk (kDynRound then needs a sequence of them)
  const int rounds = span > kDynLong ? dyn_ceil(span, kDynRound) : 1;
  if (den <= 0) return {rounds, (int)(B * rounds), span > kDynLong ? kDynRound : kDynMax};
  // chunk >= rows * heads / den, so a sequence has at most den / heads of
  // them, and all together at most that many and one more each
  int n = dyn_ceil(span, kDynUnit);
  if (dyn_ceil(den, heads) < n) n = dyn_ceil(den, heads);
  int64_t pairs = B * n < target / heads ? B * n : target / heads;
  if (pairs < B) pairs = B;
  if (B * span * heads > (int64_t)kDynLong * den) {  // dyn_chunk's c may pass kDynLong
    if (n < rounds) n = rounds;
    if (pairs < B * rounds) pairs = B * rounds;
  }
  return {n < 1 ? 1 : n, (int)pairs, kDynUnit};
}

#endif  // MOLOT_AMD_CSRC_PAGED_PLAN_HPP_
