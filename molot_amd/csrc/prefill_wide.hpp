// Interface of prefill_wide.hip and prefill_narrow.hip.
#ifndef MOLOT_AMD_CSRC_PREFILL_WIDE_HPP_
#define MOLOT_AMD_CSRC_PREFILL_WIDE_HPP_

#include <hip/hip_runtime.h>

#include <cstddef>
#include <cstdint>

#include "prefill.hpp"

constexpr int kWideTile = 32;  // keys a tile
constexpr int kWideTail = 64;  // rows of zeros after a head's pieces (two tiles' overrun)
constexpr int kWideWaves = 8;

// fp16 pieces of a cached value: two for fp32, one for bf16 and Q8 rows.
template <typename T>
constexpr int wide_pieces_v = sizeof(T) == 4 ? 2 : 1;
inline int wide_pieces(bool f32) { return f32 ? 2 : 1; }

// Query rows of a workgroup.
constexpr int wide_rows(int D) { return D <= 128 ? 128 : 64; }

// Workspace of R attended rows, per K and V and KV head: [pieces][Rp][D] fp16,
// then the rows' units [Rp] floats (Rp rows: the tail, and heads stay 16-byte
// aligned).  wide_head_elems counts 16-bit elements.
__host__ __device__ constexpr int64_t wide_padded_rows(int64_t R) {
  return (R + kWideTail + 7) / 8 * 8;
}
__host__ __device__ constexpr int64_t wide_head_elems(int D, int np, int64_t Rp) {
  return np * Rp * D + 2 * Rp;
}
inline size_t wide_bytes(int nkv, int D, int np, int64_t R) {
  return (size_t)2 * nkv * wide_head_elems(D, np, wide_padded_rows(R)) * sizeof(uint16_t);
}

// The split of the cached rows, and the attention kernels over the pieces:
// prefill_narrow.hip (D = 64 and 128), prefill_wide.hip (D = 512).
PfFn prefill_narrow_fn(int D, int kv_dtype, bool own) __attribute__((visibility("hidden")));
SplitFn prefill_wide_split(int D, int kv_dtype, bool paged) __attribute__((visibility("hidden")));
PfFn prefill_wide_fn(int D, int kv_dtype) __attribute__((visibility("hidden")));

#endif  // MOLOT_AMD_CSRC_PREFILL_WIDE_HPP_
