// Device helpers shared by the kernel sources: cache element traits, cross-lane
// reductions, the 16-bit piece splits, LDS barriers and global -> LDS copies.
#ifndef MOLOT_AMD_CSRC_DEVICE_UTIL_HPP_
#define MOLOT_AMD_CSRC_DEVICE_UTIL_HPP_

#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdint>
#include <type_traits>

namespace {


typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));

// ---------------------------------------------------------------------------
// KV element traits: one 16-byte vector = VW elements.
template <typename T>
struct KVT;

template <>
struct KVT<float> {
  static constexpr int VW = 4;
  using vec = f32x4;
  __device__ static __forceinline__ void unpack(const vec& v, float* x) {
    x[0] = v[0];
    x[1] = v[1];
    x[2] = v[2];
    x[3] = v[3];
  }
};

struct bf16_t {
  uint16_t bits;
};

template <>
struct KVT<bf16_t> {
  static constexpr int VW = 8;
  using vec = u32x4;
  __device__ static __forceinline__ void unpack(const vec& v, float* x) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      x[2 * i] = __uint_as_float(v[i] << 16);
      x[2 * i + 1] = __uint_as_float(v[i] & 0xFFFF0000u);
    }
  }
};

// Q8 codes (the row scale is applied by the kernel that reads them).
struct q8_t {
  int8_t code;
};

template <>
struct KVT<q8_t> {
  static constexpr int VW = 16;
  using vec = u32x4;
  __device__ static __forceinline__ void unpack(const vec& v, float* x) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      x[4 * i] = (float)(int8_t)(v[i] & 0xFF);
      x[4 * i + 1] = (float)(int8_t)((v[i] >> 8) & 0xFF);
      x[4 * i + 2] = (float)(int8_t)((v[i] >> 16) & 0xFF);
      x[4 * i + 3] = (float)((int32_t)v[i] >> 24);
    }
  }
};

// K/V rows are read exactly once per step: non-temporal 16-byte loads (the
// streaming hint measurably raises the sustained HBM read rate on gfx950).
// Q8 rows excepted: the KV heads of a token share 128-byte lines (head rows
// of d bytes at t*R + h*d, the token's scales after them), so a line one
// head's workgroup fetched has to stay in the L2 for its neighbour's.
template <typename T>
__device__ __forceinline__ typename KVT<T>::vec load16(const T* p) {
  if constexpr (std::is_same<T, q8_t>::value)
    return *reinterpret_cast<const typename KVT<T>::vec*>(p);
  else
    return __builtin_nontemporal_load(reinterpret_cast<const typename KVT<T>::vec*>(p));
}

// A 16-byte vector of row elements [e, e + VW) of a head row of dh
// elements (dh even, possibly not a multiple of VW), read as VW/2 pieces of
// two elements (Q8: VW/4 pieces of four codes, dh a multiple of 4).  Pieces
// at or past dh read the row's first piece instead: they stay inside the
// row, their K products meet q's zero padding and their V products land in
// output elements that are never stored.
template <typename T>
__device__ __forceinline__ typename KVT<T>::vec load_pad(const T* row, int e, int dh) {
  using V = typename KVT<T>::vec;
  constexpr int PB = 2 * (int)sizeof(T);  // bytes per two-element piece
  V v;
  const char* r = reinterpret_cast<const char*>(row);
  if constexpr (std::is_same<T, q8_t>::value) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int ee = e + 4 * i < dh ? e + 4 * i : 0;
      v[i] = *reinterpret_cast<const uint32_t*>(r + ee);  // plain: heads share lines
    }
  } else if constexpr (PB == 8) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int ee = e + 2 * i < dh ? e + 2 * i : 0;
      const f32x2 x = __builtin_nontemporal_load(reinterpret_cast<const f32x2*>(r + ee * 4));
      v[2 * i] = x[0];
      v[2 * i + 1] = x[1];
    }
  } else {
    static_assert(PB == 4, "fp32 or bf16 rows");
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int ee = e + 2 * i < dh ? e + 2 * i : 0;
      v[i] = __builtin_nontemporal_load(reinterpret_cast<const uint32_t*>(r + ee * 2));
    }
  }
  return v;
}

// Round-to-nearest-even fp32 -> bf16 (include/molot/quant.h:192-198).
__device__ __forceinline__ uint16_t f32_to_bf16(float f) {
  uint32_t u = __float_as_uint(f);
  u += 0x7FFFu + ((u >> 16) & 1u);
  return (uint16_t)(u >> 16);
}

// ---------------------------------------------------------------------------
// Q8 rows (the Q8_0 row quantizer of include/molot/quant.h:34-50, applied
// per KV head row): s = absmax/127 (1 when that is not > 0), codes
// clamp(nearbyint(x/s), -127, 127); a row dequantizes as code * s.  The
// divisions are IEEE-correct (hipcc's default for fp32 / ), so the codes and
// scales are the reference quantizer's bit for bit on the same fp32 input.
__device__ __forceinline__ float q8_scale(float amax) {
  const float s = amax / 127.0f;
  return s > 0.f ? s : 1.0f;
}
__device__ __forceinline__ int q8_code(float x, float s) {
  const int v = (int)__builtin_rintf(x / s);
  return v > 127 ? 127 : (v < -127 ? -127 : v);
}

// ---------------------------------------------------------------------------
// Cross-lane sums.  Lanes are grouped in aligned groups of N; every lane of
// a group receives the group's sum.  Groups up to 16 use DPP within a row
// (quad_perm xor1, quad_perm xor2, row_half_mirror, row_mirror: after the
// quad steps every lane holds its quad's sum, and each mirror pairs a lane
// with one in the other half of its 8/16-lane block).
template <int CTRL>
__device__ __forceinline__ float dpp_f(float x) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), CTRL, 0xF, 0xF, false));
}

// x of lanes l and l ^ 16 (xor16), or l and l ^ 32 (xor32), as the pair
// (lower lane's, upper lane's) in every lane: v_permlane16_swap and
// v_permlane32_swap exchange 16- or 32-lane rows of two registers, so with
// both operands x they leave the lower row's x in the first and the upper
// row's in the second, in both rows (checked lane by lane on the GPU).
// Reducing the pair gives every lane the same operands in the same order,
// where a shuffle would take two LDS round trips.
__device__ __forceinline__ float max_xor16(float x) {
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false,
                                                  false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float max_xor32(float x) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false,
                                                  false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float sum_xor16(float x) {
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false,
                                                  false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
__device__ __forceinline__ float sum_xor32(float x) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false,
                                                  false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// x combined with lane l ^ OFF's x (a sum in the shuffle's operand order)
template <int OFF>
__device__ __forceinline__ float sum_xor(float x) {
  if constexpr (OFF == 16) return sum_xor16(x);
  else if constexpr (OFF == 32) return sum_xor32(x);
  else return x + __shfl_xor(x, OFF);
}
template <int OFF>
__device__ __forceinline__ float max_xor(float x) {
  if constexpr (OFF == 16) return max_xor16(x);
  else if constexpr (OFF == 32) return max_xor32(x);
  else return fmaxf(x, __shfl_xor(x, OFF));
}

template <int N>
__device__ __forceinline__ float group_max(float v) {
  if constexpr (N >= 2) v = fmaxf(v, dpp_f<0xB1>(v));
  if constexpr (N >= 4) v = fmaxf(v, dpp_f<0x4E>(v));
  if constexpr (N >= 8) v = fmaxf(v, dpp_f<0x141>(v));
  if constexpr (N >= 16) v = fmaxf(v, dpp_f<0x140>(v));
  if constexpr (N >= 32) v = max_xor16(v);
  if constexpr (N >= 64) v = max_xor32(v);
  return v;
}

template <int N>
__device__ __forceinline__ float group_sum(float v) {
  if constexpr (N >= 2) v += dpp_f<0xB1>(v);   // quad_perm [1,0,3,2]
  if constexpr (N >= 4) v += dpp_f<0x4E>(v);   // quad_perm [2,3,0,1]
  if constexpr (N >= 8) v += dpp_f<0x141>(v);  // row_half_mirror
  if constexpr (N >= 16) v += dpp_f<0x140>(v); // row_mirror
  if constexpr (N >= 32) v = sum_xor16(v);
  if constexpr (N >= 64) v = sum_xor32(v);
  return v;
}

// Wave-wide max / sum with DPP only (no LDS round trips): the quad and
// mirror steps reduce each row of 16 lanes, row_bcast:15 and row_bcast:31
// carry the partial results up to lane 63, which readlane broadcasts.
template <bool MAX>
__device__ __forceinline__ float wave_reduce(float v) {
  auto op = [](float x, float y) { return MAX ? fmaxf(x, y) : x + y; };
  v = op(v, dpp_f<0xB1>(v));   // quad_perm [1,0,3,2]
  v = op(v, dpp_f<0x4E>(v));   // quad_perm [2,3,0,1]
  v = op(v, dpp_f<0x141>(v));  // row_half_mirror
  v = op(v, dpp_f<0x140>(v));  // row_mirror
  // row_bcast:15 into rows 1 and 3, row_bcast:31 into rows 2 and 3; rows
  // outside the mask keep their value (old = v)
  v = op(v, __int_as_float(__builtin_amdgcn_update_dpp(__float_as_int(MAX ? -INFINITY : 0.f),
                                                       __float_as_int(v), 0x142, 0xA, 0xF,
                                                       false)));
  v = op(v, __int_as_float(__builtin_amdgcn_update_dpp(__float_as_int(MAX ? -INFINITY : 0.f),
                                                       __float_as_int(v), 0x143, 0xC, 0xF,
                                                       false)));
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 63));
}

// exp used by the split-K merges (full-accuracy device expf).
__device__ __forceinline__ float softmax_exp(float x) { return expf(x); }

// The decode kernels' softmax runs in base 2: a score is q.k * scale*log2(e)
// (the matrix-core kernel pre-scales q, the vector-ALU kernel each score), so
// p = 2^(s - m) is one v_exp_f32 (relative error ~|s - m| * 2^-24, within
// the reference's own exp, exp_avx512_ps at 1.5e-6).  The maxima leave the
// kernels in natural units (m * ln 2) for the split-K merges.
constexpr float kLog2e = 1.4426950408889634f;
constexpr float kLn2 = 0.6931471805599453f;
__device__ __forceinline__ float exp2_hw(float x) { return __builtin_amdgcn_exp2f(x); }
// A running max moves only when a score exceeds it by more than kLazyMax
// (p <= 2^8 otherwise): o and l always share the max they were formed with,
// so the result is exact either way, and most blocks skip the rescale.
constexpr float kLazyMax = 8.f;

typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
__device__ __forceinline__ uint32_t bf16_pair_exact(float a, float b) {
  const bf16x2_t p = {(__bf16)a, (__bf16)b};
  return __builtin_bit_cast(uint32_t, p);
}

// split3 of two values at once: each piece of the pair is one
// v_cvt_pk_bf16_f32 (round to nearest even, as split3), element a in the
// low half.  The same pieces as split3 on each value.
__device__ __forceinline__ uint32_t bf16_pair(float a, float b) { return bf16_pair_exact(a, b); }
__device__ __forceinline__ void split3x2(float a, float b, uint32_t& hi, uint32_t& mid,
                                         uint32_t& lo) {
  // The residuals are taken of a and b as rounded to fp32: a product that
  // formed them (a Q8 code times its scale, q times the score scale) must
  // not fuse into the first subtraction, or the pieces would split the
  // unrounded product and differ between the kernels that form a and b
  // differently.
#pragma clang fp contract(off)
  hi = bf16_pair(a, b);
  float ra = a - __uint_as_float(hi << 16), rb = b - __uint_as_float(hi & 0xFFFF0000u);
  mid = bf16_pair(ra, rb);
  ra -= __uint_as_float(mid << 16);
  rb -= __uint_as_float(mid & 0xFFFF0000u);
  lo = bf16_pair(ra, rb);
}

// Two fp16 pieces of a row scaled by a power of two: with the row's largest
// |x| in [2^(ex-1), 2^ex) (frexpf of it), y = x * 2^(14-ex) has |y| < 2^14,
// hi = fp16(y), lo = fp16(y - hi), each rounded to nearest even.  hi + lo
// holds y to 2^-22 of |y| while |y| >= 2^-3 (lo a normal fp16), and to
// 2^-25 absolute below (2^-38 of the row's largest |y|); the scaling is
// exact.  y's unit is 2^(ex-14) (f16_row_unit), the factor that takes a
// dot product of such pieces back: a normal float, so that a masked score's
// -inf stays one over a row of subnormal values (their bits, multiples of
// 2^-149, are whole numbers of y's 2^-24 at the shift of 126 too).
// Non-finite values make NaN pieces.
__device__ __forceinline__ int f16_row_shift(float amax) {
  int ex = 0;
  (void)frexpf(amax, &ex);
  return min(14 - ex, 126);
}
__device__ __forceinline__ float f16_row_unit(int shift) { return ldexpf(1.f, -shift); }
__device__ __forceinline__ uint32_t f16_pair(float a, float b) {
  const _Float16 ha = (_Float16)a, hb = (_Float16)b;
  return (uint32_t)__builtin_bit_cast(uint16_t, ha) |
         ((uint32_t)__builtin_bit_cast(uint16_t, hb) << 16);
}
__device__ __forceinline__ void split2h(float a, float b, int shift, uint32_t& hi, uint32_t& lo) {
#pragma clang fp contract(off)
  const float ya = ldexpf(a, shift), yb = ldexpf(b, shift);
  hi = f16_pair(ya, yb);
  const float ra = ya - (float)__builtin_bit_cast(_Float16, (uint16_t)(hi & 0xFFFFu));
  const float rb = yb - (float)__builtin_bit_cast(_Float16, (uint16_t)(hi >> 16));
  lo = f16_pair(ra, rb);
}
// V rows (the prefill's PV operand): the same split, with the unit kept a
// normal float (shift <= 120: 2^-120 and up; rows below 2^-106 keep fewer
// bits, as fp32 denormals would) and 0 for a row of zeros, which then
// weighs nothing and never sets a tile's largest unit.
__device__ __forceinline__ int f16_vrow_shift(float amax) { return min(f16_row_shift(amax), 120); }
__device__ __forceinline__ float f16_vrow_unit(float amax, int shift) {
  return amax > 0.f ? f16_row_unit(shift) : 0.f;
}

// ---------------------------------------------------------------------------
// Workgroup barrier that orders LDS accesses only.  __syncthreads() also
// waits for every outstanding global load and store of the thread
// (s_waitcnt vmcnt(0)), which would stall the prologue on the K/V blocks
// already in flight.  No global data crosses workgroups inside a launch
// (the combine is a separate kernel).
// s_waitcnt vmcnt(N) alone (expcnt and lgkmcnt at their maxima; gfx9
// encoding: vmcnt bits 3:0 and 15:14, expcnt 6:4, lgkmcnt 11:8).
template <int N>
__device__ __forceinline__ void wait_vmcnt() {
  static_assert(N >= 0 && N < 64, "vmcnt range");
  __builtin_amdgcn_s_waitcnt((N & 15) | (((N >> 4) & 3) << 14) | (7 << 4) | (15 << 8));
}

__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

typedef _Float16 f16x8_t __attribute__((ext_vector_type(8)));

// One 16-byte global -> LDS copy per lane (global_load_lds_dwordx4, scalar
// base + lane offset): lane l's 16 bytes land at LDS address lds + 16*l.
// Written as inline assembly, so the compiler does not see an LDS store in
// flight: with the builtin it put an s_waitcnt vmcnt(0) before the next LDS
// reads it could not tell apart from the copy's destination (the transposed
// V reads of the other tile buffer), which waited for the next tile's copies
// halfway through every tile.  The kernel orders the copies itself
// (wait_vmcnt, then a barrier, before a buffer is read).  m0 takes the LDS
// address as an input operand (the compiler writes it).  The scalar base goes
// through an s_mov_b64 of the same statement: where a vector instruction
// (v_readfirstlane) wrote it, a vector memory instruction may read it only
// five wait states later, a hazard the compiler does not resolve inside inline
// assembly, while a scalar instruction's read is interlocked and its result
// has no such hazard.  It is also the wait state between the write of m0 and
// the copy.
__device__ __forceinline__ void dma16(const void* base, uint32_t off, uint32_t lds) {
  const void* b;
  asm volatile("s_mov_b64 %0, %2\n\tglobal_load_lds_dwordx4 %1, %0"
               : "=&s"(b)
               : "v"(off), "s"(base), "{m0}"(lds)
               : "memory");
}
// A wave-uniform address, in scalar registers whatever formed it.
template <typename P>
__device__ __forceinline__ const P* uniform_ptr(const P* p) {
  const uint64_t u = (uint64_t)p;
  const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)u);
  const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(u >> 32));
  return (const P*)((uint64_t)hi << 32 | lo);
}
// dma16 with 4 bytes a lane (global_load_lds_dword): lane l's 4 bytes
// land at LDS address lds + 4*l.
__device__ __forceinline__ void dma4(const void* base, uint32_t off, uint32_t lds) {
  const void* b;
  asm volatile("s_mov_b64 %0, %2\n\tglobal_load_lds_dword %1, %0"
               : "=&s"(b)
               : "v"(off), "s"(base), "{m0}"(lds)
               : "memory");
}

}  // namespace

#endif  // MOLOT_AMD_CSRC_DEVICE_UTIL_HPP_
