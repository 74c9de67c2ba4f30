// Device parts shared by the prefill kernels of 32 query rows a wave
// (prefill_wide.hip, prefill_narrow.hip): the piece workspace's rows, the
// tiles' swizzles, and the softmax of one tile.
#ifndef MOLOT_AMD_CSRC_PREFILL_TILE_HPP_
#define MOLOT_AMD_CSRC_PREFILL_TILE_HPP_

#include <hip/hip_runtime.h>

#include "device_util.hpp"
#include "molot_amd/attn_hip.h"
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

// Rows that the pieces cannot hold for every query row alike.  A product over a
// tile takes each of its keys for all its query rows, a masked one times zero:
// a non-finite V row reaches rows that do not attend it, and a K row's infinity
// leaves no score of its sign.  Where each query row used to read its own keys
// alone (head dims above 256 and those that are not multiples of 8, Q8 at any
// padded one: PfArgs::own) the split marks such rows, and those out of the
// units' range, by a NaN unit, and a workgroup that met one forms its rows'
// results again from the cache (own_rows).
constexpr float kOwnMaxK = 3.0e23f;   // 2^78: past it a raw score times its unit may overflow
constexpr float kOwnMinV = 7.9e-31f;  // 2^-100: below it a V row's unit keeps fewer bits
__device__ __forceinline__ float own_mark(float xmax, float nonfinite, int kv) {
  const bool out = kv ? xmax > 0.f && xmax < kOwnMinV : xmax > kOwnMaxK;
  return out ? NAN : nonfinite;  // 0, or NaN
}

// Element e of the row at off (wide_row_off's unit), not yet times a Q8 scale.
__device__ __forceinline__ float own_elem(const PfArgs& a, const char* base, int64_t off, int e) {
  if (a.kv_dtype == MOLOT_KV_Q8) return (float)reinterpret_cast<const int8_t*>(base)[off + e];
  if (a.kv_dtype == MOLOT_KV_BF16)
    return __uint_as_float((uint32_t)reinterpret_cast<const uint16_t*>(base)[off + e] << 16);
  return reinterpret_cast<const float*>(base)[off + e];
}
__device__ __forceinline__ int64_t own_row_off(const PfArgs& a, int h, int t, int64_t& soff) {
  const bool q8 = a.kv_dtype == MOLOT_KV_Q8;
  if (a.block_table)
    return q8 ? wide_row_off<q8_t, true>(a, h, t, soff) : wide_row_off<float, true>(a, h, t, soff);
  return q8 ? wide_row_off<q8_t, false>(a, h, t, soff) : wide_row_off<float, false>(a, h, t, soff);
}

// The address of the kernel's arguments (a PfArgs, its only parameter), to be
// taken in the kernel itself: a called function has no such pointer (the
// builtin gives null there), so it and own_rows are inlined.
__device__ __forceinline__ uint64_t own_args() {
  uint64_t args = (uint64_t)__builtin_amdgcn_kernarg_segment_ptr();
  asm volatile("" : "+s"(args));
  return args;
}

// Query rows [row0, row0 + n) of KV head h over their own keys of [k_lo, k_hi),
// a row at a time (every lane of the wave takes part), for the launch's split
// sp.  Meant for caches that hold non-finite values; two keys in flight.  The
// arguments are read again from args (own_args), where the compiler cannot move
// the loads ahead: kept in registers through the kernel's loop they would
// spill.
template <int D>
__device__ __forceinline__ void own_rows(uint64_t args, int h, int row0, int n, int k_lo, int k_hi,
                                         int sp) {
  const auto* ka = (const __attribute__((address_space(4))) PfArgs*)args;
  PfArgs a{};
  a.q = ka->q, a.k = ka->k, a.v = ka->v, a.o = ka->o, a.block_table = ka->block_table;
  a.nq = ka->nq, a.nkv = ka->nkv, a.M = ka->M, a.N = ka->N, a.pos0 = ka->pos0;
  a.window = ka->window, a.dh = ka->dh, a.page_shift = ka->page_shift, a.scale = ka->scale;
  a.kv_dtype = ka->kv_dtype, a.nsplit = ka->nsplit, a.part_o = ka->part_o, a.part_ml = ka->part_ml;
  constexpr int EPL = D / 64;  // elements lane + 64*i of a lane
  const int lane = threadIdx.x & 63;
  const int G = a.nq / a.nkv;
  const bool q8 = a.kv_dtype == MOLOT_KV_Q8;
  const char* kb = reinterpret_cast<const char*>(a.k);
  const char* vb = reinterpret_cast<const char*>(a.v);
  for (int row = row0; row < min(row0 + n, a.M * G); ++row) {
    const int m = row / G, pos = a.pos0 + m;
    const int64_t slot = (int64_t)m * a.nq + h * G + (row - m * G);
    int lo = (a.window > 0 && pos - a.window + 1 > 0) ? pos - a.window + 1 : 0;
    lo = max(lo, k_lo);
    const int hi = min(min(pos + 1, a.N), k_hi);
    float q[EPL], o[EPL];
#pragma unroll
    for (int i = 0; i < EPL; ++i) {
      const int e = lane + 64 * i;
      q[i] = e < a.dh ? a.q[slot * a.dh + e] : 0.f;
      o[i] = 0.f;
    }
    const float qsc = a.scale * kLog2e;
    float mx = -INFINITY, l = 0.f;
    for (int t0 = lo; t0 < hi; t0 += 2) {
      float s[2], v[2][EPL];
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        int64_t soff = 0;
        const int64_t off = own_row_off(a, h, min(t0 + u, hi - 1), soff);
        const float ks = q8 ? *reinterpret_cast<const float*>(kb + soff) : 1.f;
        const float vs = q8 ? *reinterpret_cast<const float*>(vb + soff) : 1.f;
        float acc = 0.f;
#pragma unroll
        for (int i = 0; i < EPL; ++i) {
          const int e = lane + 64 * i;
          const bool in = e < a.dh;
          if (in) acc = fmaf(q[i], own_elem(a, kb, off, e), acc);
          v[u][i] = in ? own_elem(a, vb, off, e) * vs : 0.f;
        }
        s[u] = t0 + u < hi ? wave_reduce<false>(acc) * (ks * qsc) : -INFINITY;
      }
      const float mn = fmaxf(mx, fmaxf(s[0], s[1]));
      if (mn > mx) {
        const float f = exp2_hw(mx - mn);
        l *= f;
#pragma unroll
        for (int i = 0; i < EPL; ++i) o[i] *= f;
        mx = mn;
      }
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        if (t0 + u >= hi) break;
        const float p = s[u] == -INFINITY ? 0.f : exp2_hw(s[u] - mx);
        l += p;
#pragma unroll
        for (int i = 0; i < EPL; ++i) o[i] = fmaf(p, v[u][i], o[i]);
      }
    }
    const bool part = a.nsplit > 1;
    const int64_t ps = slot * a.nsplit + sp;
    const float inv = part ? 1.f : l == 0.f ? 0.f : 1.f / l;  // no key: O = 0 (gemm.h:438)
#pragma unroll
    for (int i = 0; i < EPL; ++i) {
      const int e = lane + 64 * i;
      if (part)
        a.part_o[ps * D + e] = o[i];
      else if (e < a.dh)
        a.o[slot * a.dh + e] = o[i] * inv;
    }
    if (part && lane == 0) {
      a.part_ml[2 * ps] = l == 0.f ? -INFINITY : mx * kLn2;
      a.part_ml[2 * ps + 1] = l;
    }
  }
}

// The softmax state of a query row.  o and l are held times 2^-m, and o
// times 2^wsh more; m moves by whole numbers, so every rescale is by a power
// of two.
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

// o / l from o * (1 / l) and its remainder, rounded once but for ties nearby.
__device__ __forceinline__ float div_by(float o, float l, float inv) {
  const float q = o * inv;
  return fmaf(fmaf(-q, l, o), inv, q);
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
// wave, m moves where a score passes it by 4, by a whole number past it; wsh
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
    // a first m within 2^-15 of the maximum (a row of one key then has p = 1 but
    // for that, and loses nothing to the dropped product of the low pieces);
    // multiples of 2^-14, so that steps by whole numbers are exact
    float mn = st.m;
    if (tm > st.m + 4.f)
      mn = st.m != -1e30f       ? st.m + ceilf(tm - st.m)
           : fabsf(tm) < 512.f ? rintf(tm * 16384.f) * (1.f / 16384.f)
                               : ceilf(tm);
    const int gsh = (int)rintf(fminf(mn - st.m, 1e6f));
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
