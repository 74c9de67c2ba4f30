// The prefill attention launch shared by its kernel sources.
#ifndef MOLOT_AMD_CSRC_PREFILL_HPP_
#define MOLOT_AMD_CSRC_PREFILL_HPP_

#include <cstdint>

struct PfArgs {
  const float* q;  // [M][nq][D]
  const void* k;   // token-major cache [N][nkv*D], or pages [block][nkv][page][D]
  const void* v;
  float* o;        // [M][nq][D]
  const int32_t* block_table;  // paged: the sequence's row of block ids
  int nq, nkv, M, N, pos0, window, nqb;  // nqb: blocks of 16 * (waves) query rows per KV head
  int dh;  // head dim as stored (< D: the launch runs padded to D, through the pieces)
  int page_shift;
  float scale;
  // 32-row kernels: a query row's output depends on the keys it attends alone
  // (own_rows below); the cache type then says how to read them
  int own, kv_dtype;
  // the attended keys [T0, T0 + R) of every KV head split into 16-bit pieces
  // once for the launch (pf_split_kernel): [K, V][nkv][3 pieces][R][D]; NULL:
  // the kernel splits each staged tile itself
  const uint16_t* pieces;
  int T0, R;
  int Rsplit;  // pf_split_kernel splits rows [T0, T0 + Rsplit); the appending step wrote the rest
  // split-K over the key tiles (nsplit > 1): split s of a query block takes
  // its share of the tiles and writes unnormalised o and (max, sum) per query
  // row, slot m*nq + head, to part_o [slot][nsplit][D] and part_ml
  // [slot][nsplit][2]; combine_kernel merges them into O
  int nsplit;
  float* part_o;
  float* part_ml;
};

using PfFn = void (*)(PfArgs);
using SplitFn = void (*)(PfArgs, uint16_t*);

#endif  // MOLOT_AMD_CSRC_PREFILL_HPP_
