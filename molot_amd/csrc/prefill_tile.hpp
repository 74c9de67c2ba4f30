// Device parts shared by the prefill kernels of 32 query rows a wave
// (prefill_wide.hip, prefill_narrow.hip): the piece workspace's rows, the
// tiles' swizzles, and the softmax of one tile.
#ifndef MOLOT_AMD_CSRC_PREFILL_TILE_HPP_
#define MOLOT_AMD_CSRC_PREFILL_TILE_HPP_

#include <hip/hip_runtime.h>

#include "device_util.hpp"
#include "prefill.hpp"
#include "prefill_wide.hpp"

namespace {

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4_u __attribute__((ext_vector_type(4), aligned(4)));  // dword-aligned
typedef short i16x4_t __attribute__((ext_vector_type(4)));

__device__ __forceinline__ f32x16 mfma32_f16(f16x8_t a, f16x8_t b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
}

// Swizzles of the staged rows (16-byte units; unit ch of row r at ch ^ f(r)).
// K: a 16-byte read takes one unit of 16 consecutive rows.  V: a transposed
// read takes 64 bytes of 4 consecutive rows.  Both then cover 256 bytes
// (D = 64: two rows in 256 bytes, so the row's parity is one bit already).
template <int D>
__device__ __forceinline__ int wk_f(int r) {
  return D == 64 ? (r >> 1) & 7 : r & 15;
}
template <int D>
__device__ __forceinline__ int wv_f(int r) {
  return D == 64 ? ((r >> 1) & 1) << 2 : (r & 3) << 2;
}

// Offset (elements; Q8 bytes) of row t of KV head h in a cache of head dim
// a.dh, and of a Q8 row's scale.
template <typename T, bool PAGED>
__device__ __forceinline__ int64_t wide_row_off(const PfArgs& a, int h, int t, int64_t& soff) {
  constexpr bool Q8 = std::is_same<T, q8_t>::value;
  const int dh = a.dh;
  if constexpr (PAGED) {
    const int pg = 1 << a.page_shift;
    const int64_t blk = a.block_table[t >> a.page_shift];
    const int sl = t & (pg - 1);
    if constexpr (Q8) {
      const int64_t bb = (int64_t)a.nkv * pg * (dh + 4);
      soff = blk * bb + (int64_t)a.nkv * pg * dh + 4 * ((int64_t)h * pg + sl);
      return blk * bb + ((int64_t)h * pg + sl) * dh;
    }
    return ((blk * a.nkv + h) * pg + sl) * (int64_t)dh;
  } else {
    if constexpr (Q8) {
      const int64_t rb = (int64_t)a.nkv * dh + ((4 * a.nkv + 15) & ~15);
      soff = (int64_t)t * rb + (int64_t)a.nkv * dh + 4 * h;
      return (int64_t)t * rb + (int64_t)h * dh;
    }
    return ((int64_t)t * a.nkv + h) * (int64_t)dh;
  }
}

// Elements 8j .. 8j+7 of row t of KV head h (kv: V), 0 past a.dh (even; Q8 a
// multiple of 4), and a Q8 row's scale (1 otherwise): a Q8 element is its code.
template <typename T, bool PAGED>
__device__ __forceinline__ float wide_load8(const PfArgs& a, int kv, int h, int t, int j,
                                            float (&x)[8]) {
  constexpr bool Q8 = std::is_same<T, q8_t>::value;
#pragma unroll
  for (int e = 0; e < 8; ++e) x[e] = 0.f;
  int64_t soff = 0;
  const int64_t off = wide_row_off<T, PAGED>(a, h, t, soff);
  const char* base = reinterpret_cast<const char*>(kv ? a.v : a.k);
  const int e0 = 8 * j, n = min(8, a.dh - e0);  // elements of the row in this unit
  if constexpr (Q8) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      if (4 * i < n) {
        const uint32_t c = *reinterpret_cast<const uint32_t*>(base + off + e0 + 4 * i);
#pragma unroll
        for (int e = 0; e < 4; ++e) x[4 * i + e] = (float)(int8_t)((c >> (8 * e)) & 0xFF);
      }
    }
    return *reinterpret_cast<const float*>(base + soff);
  } else if constexpr (sizeof(T) == 2) {
    const uint16_t* p = reinterpret_cast<const uint16_t*>(base) + off + e0;
    if (n == 8 && (a.dh & 7) == 0) {
      const u32x4 v = *reinterpret_cast<const u32x4*>(p);
      KVT<bf16_t>::unpack(v, x);
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (2 * i < n) {
          const uint32_t v = *reinterpret_cast<const uint32_t*>(p + 2 * i);
          x[2 * i] = __uint_as_float(v << 16);
          x[2 * i + 1] = __uint_as_float(v & 0xFFFF0000u);
        }
    }
  } else {
    const float* p = reinterpret_cast<const float*>(base) + off + e0;
    if (n == 8 && (a.dh & 3) == 0) {
      const f32x4 x0 = *reinterpret_cast<const f32x4*>(p);
      const f32x4 x1 = *reinterpret_cast<const f32x4*>(p + 4);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        x[e] = x0[e];
        x[4 + e] = x1[e];
      }
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (2 * i < n) {
          const f32x2 v = *reinterpret_cast<const f32x2*>(p + 2 * i);
          x[2 * i] = v[0];
          x[2 * i + 1] = v[1];
        }
    }
  }
  return 1.f;
}

// The softmax state of a query row.  o and l are held times 2^-m, and o
// times 2^wsh more; m is an integer, so every rescale is by a power of two.
struct RowState {
  float m = -1e30f;  // no key yet
  float l = 0.f;     // this lane's keys
  int wsh = 1 << 20;
  float sc = 0.f;      // 2^wsh
  float lim = 1e-45f;  // 2^(14-wsh), the bound of z; no V unit yet: any z > 0 needs one
};

// y = z * sc as two fp16 pieces, hi = fp16(y) and lo = fp16(y - hi) of the
// exact product, for a pair of values.
__device__ __forceinline__ void mix_split(float z0, float z1, float sc, uint32_t& hi,
                                          uint32_t& lo) {
  asm("v_fma_mixlo_f16 %0, %1, %2, 0" : "=v"(hi) : "v"(z0), "v"(sc));
  asm("v_fma_mixhi_f16 %0, %1, %2, 0" : "+v"(hi) : "v"(z1), "v"(sc));
  asm("v_fma_mixlo_f16 %0, %1, %2, -%3 op_sel_hi:[0,0,1]" : "=v"(lo) : "v"(z0), "v"(sc), "v"(hi));
  asm("v_fma_mixhi_f16 %0, %1, %2, -%3 op_sel:[0,0,1] op_sel_hi:[0,0,1]"
      : "+v"(lo)
      : "v"(z1), "v"(sc), "v"(hi));
}

// One tile of NK keys a lane: s[e] the scores over the row units (K's ku, the
// q row's qunit: powers of two, Q8 ku times the row's scale), vu the keys' V
// row units.  Leaves y = p * vu * 2^wsh as two fp16 pieces, y < 2^14, and
// returns the factor the row's o takes first.  gmax: the maximum over the
// row's lanes; dead(e): key e is outside the row's range (only asked when the
// tile is not `full`).
//
// A tile whose probabilities and y stay in range (the usual one) takes no row
// maximum: p from the m so far, and two checks.  Otherwise, in any row of the
// wave, m moves where a score passes it by 4, to the integer above; wsh
// follows o down with it, and is lowered where y would pass 2^14, by kRoom
// bits more than needed, so that the next records of 32 rows do not each
// rescale o.
template <int NK, typename GMAX, typename DEAD>
__device__ __forceinline__ float softmax_tile(float (&s)[NK], const float (&ku)[NK],
                                              const float (&vu)[NK], float qunit, RowState& st,
                                              bool full, GMAX&& gmax, DEAD&& dead,
                                              uint32_t (&yh)[NK / 2], uint32_t (&yl)[NK / 2]) {
  constexpr int kRoom = 3;
  constexpr int kNoShift = 1 << 20;
  float ps, zt, z[NK];
#pragma unroll
  for (int e = 0; e < NK; ++e) s[e] *= ku[e];
  if (!full) {
#pragma unroll
    for (int e = 0; e < NK; ++e) s[e] = dead(e) ? -INFINITY : s[e];
  }
  auto probs = [&](float m) {
    ps = 0.f;
    zt = 0.f;
#pragma unroll
    for (int e = 0; e < NK; ++e) {
      const float p = exp2_hw(fmaf(s[e], qunit, -m));
      ps += p;
      z[e] = p * vu[e];
      zt = fmaxf(zt, z[e]);
    }
  };
  probs(st.m);
  float fac = 1.f;
  const bool fine = ps < 512.f && zt < st.lim;
  if (__builtin_amdgcn_ballot_w64(!fine) != 0) {
    float tm = s[0];
#pragma unroll
    for (int e = 1; e < NK; ++e) tm = fmaxf(tm, s[e]);
    tm = gmax(tm) * qunit;
    const float mn = tm > st.m + 4.f ? ceilf(tm) : st.m;
    const int gsh = (int)fminf(mn - st.m, 1e6f);
    probs(mn);
    zt = gmax(zt);
    const int grown = min(st.wsh + gsh, kNoShift);
    const int most = zt > 0.f ? f16_row_shift(zt) : kNoShift;
    int ns = most < grown ? most - kRoom : grown;
    ns = ns == kNoShift ? ns : min(ns, 126);
    fac = ldexpf(1.f, ns - st.wsh - gsh);  // 0 while the row has no key
    st.l *= ldexpf(1.f, -gsh);
    st.m = mn;
    st.wsh = ns;
    st.sc = ns == kNoShift ? 0.f : ldexpf(1.f, ns);
    if (ns != kNoShift) st.lim = ldexpf(1.f, 14 - ns);
  }
  st.l += ps;
#pragma unroll
  for (int e = 0; e < NK; e += 2) mix_split(z[e], z[e + 1], st.sc, yh[e / 2], yl[e / 2]);
  return fac;
}

}  // namespace

#endif  // MOLOT_AMD_CSRC_PREFILL_TILE_HPP_
