// Host check of molot_amd/csrc/paged_plan.hpp, bf16 and Q8: over every length of
// a lone sequence and over random batches, with the host's bound of the longest
// sequence exact (a fused step attends one row less than it counts) or loose,
// the chunks the device takes stay within the chunks, pairs and least rows that
// the host planned for.  Prints the first failures; exit status 0 if none.
#include <algorithm>
#include <cmath>
#include <cstdio>
#include <random>
#include <vector>

#include "../../molot_amd/csrc/paged_plan.hpp"

namespace {

constexpr int kTarget = 512;  // two workgroups on each of 256 CUs
long g_bad = 0;

void check(const std::vector<int>& lens, int span, int heads, bool q8) {
  const int B = (int)lens.size();
  const DynPlan p = dyn_plan(span, B, heads, kTarget, q8);
  long rows = 0, pairs = 0;
  for (int n : lens) rows += n;
  const int chunk = dyn_chunk((int)rows, B, heads, kTarget, q8);
  int most = 0;
  for (int n : lens) {
    most = std::max(most, dyn_chunks(n, chunk));
    pairs += std::max(1, dyn_chunks(n, chunk));
  }
  if (most <= p.nchunks && pairs <= p.pairs && chunk >= p.min_chunk && chunk <= kDynMax &&
      p.likely >= 1 && p.likely <= p.nchunks)
    return;
  if (g_bad++ < 20)
    std::printf("%s, %d sequences, %d heads, bound %d, %ld rows: chunk %d (planned >= %d), "
                "%d chunks of %d (likely %d), %ld pairs of %d\n",
                q8 ? "Q8" : "bf16", B, heads, span, rows, chunk, p.min_chunk, most, p.nchunks, p.likely, pairs, p.pairs);
}

void check(const std::vector<int>& lens, int span, int heads) {
  check(lens, span, heads, false);
  check(lens, span, heads, true);
}

}  // namespace

int main() {
  std::mt19937 rng(1);
  auto below = [&](int n) { return (int)(rng() % (unsigned)n); };
  for (int heads = 2; heads <= 40; ++heads)
    for (int span = 1; span <= 131072; ++span) {
      check({span}, span, heads);
      check({span - 1}, span, heads);             // a fused step
      if (span % 16 == 0) check({1 + below(span)}, span, heads);  // a table's capacity
    }
  for (int i = 0; i < 400000; ++i) {
    const int B = 1 + below(130), heads = 1 + below(40);
    const int span = 1 + (int)std::exp2(below(1700) / 100.0);
    if ((long)B * span * heads >= 1L << 30) continue;  // plan_launch's own limit
    const int longest = i % 2 ? span - below(2) : below(span) + 1, kind = below(4);
    std::vector<int> lens(B);
    for (int& n : lens)
      n = kind == 0   ? below(longest + 1)
          : kind == 1 ? (below(8) ? 1 : longest)
          : kind == 2 ? longest
                      : std::max(0, longest - below(3));
    lens[0] = longest;
    check(lens, span, heads);
  }
  check({7681, 1, 1, 1}, 7682, 8);
  std::vector<int> lone(13, 1);
  lone[0] = 6529;
  check(lone, 6530, 8);
  std::printf("%ld failures\n", g_bad);
  return g_bad ? 1 : 0;
}
