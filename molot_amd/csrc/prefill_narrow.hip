// Causal prefill attention (include/molot/gemm.h:409-446) for head dims up to
// 128 on the matrix cores: 32 query rows a wave, two waves of opposite phase
// a SIMD.
//
// Query rows of one KV head are r = m*G + g (token m at pos0 + m, q head g of
// the group).  A workgroup of 8 waves owns 128 of them and walks their keys
// in intervals of two tiles of 32: wave (kg, rg) takes the 32 rows of row
// group rg and the tiles 2i + kg.  Per tile it forms S^T = K . Q^T
// (v_mfma_f32_32x32x16_f16, A = K from LDS, B = q pieces in registers), the
// softmax in registers (a lane holds one row and 16 keys, its row's other 16
// in lane ^ 32), and O^T += V^T . P^T with P where the score accumulator left
// it (A = V^T by transposed LDS reads in the same key order).  The two key
// groups' (m, l, o) are merged through LDS at the end.
//
// Why this split: each staged K or V operand of 1 KB serves 32 rows, 85 bytes
// a cycle of LDS reads at the full matrix rate over fp32 values, where 16 rows
// a wave (prefill_mfma16_kernel) ask 170 of an LDS that reads 128.  Waves w
// and w + 4 share a SIMD: key group 0 runs an interval as scores, softmax,
// PV, key group 1 as PV of its last tile, scores, softmax, so that one's
// softmax meets the other's products (its V is copied one interval later).
//
// Products and pieces as prefill_wide.hip: q and p two fp16 pieces, K and V
// NP = 2 for fp32 values, 1 for bf16 and Q8 rows.
//
// Error: the scores take the products with a low piece before the others, and
// the first running maximum of a row is its own (softmax_tile).  Against 64
// bits (2-norm, 32q/8kv/d128 fp32), before, now and prefill_mfma16_kernel: 300
// tokens after 900 3.0e-7, 2.6e-7 and 2.7e-7; 2048 tokens 2.6e-7, 2.2e-7 and
// 2.6e-7; 512 after 16384 7.9e-7, 7.7e-7 and 1.1e-6 (bf16 6.3, 6.3 and 10).
//
// What bounds it (32q/8kv/d128, stamped, cycles an interval; products alone
// take a SIMD 3072 over fp32, 2048 over bf16): 5700 over fp32 and 4100 over
// bf16, the longer key group's PV 1870 / 1280, scores 2600 / 1330 and softmax
// 870 / 900 one after the other; without the copies 5100.  Against
// prefill_mfma16_kernel (16 rows a wave; three bf16 products over bf16 and
// Q8 values): 2048-token prompt fp32 step 154 -> 136 us, 512 tokens after
// 16384 bf16 414 -> 301, Q8 485 -> 298, fp32 497 -> 438 us.
#include <hip/hip_runtime.h>

#include "device_util.hpp"
#include "molot_amd/attn_hip.h"
#include "prefill.hpp"
#include "prefill_tile.hpp"
#include "prefill_wide.hpp"

namespace {

// OWN: PfArgs::own (prefill_tile.hpp).
template <int D, int NP, bool OWN>
__global__ __launch_bounds__(512) void prefill_narrow_kernel(PfArgs a) {
  static_assert(D == 64 || D == 128, "head dims up to 128");
  constexpr int KT = kWideTile;
  constexpr int QB = 128;            // query rows a workgroup
  constexpr int QS = D / 16;         // 16-element steps of the scores
  constexpr int DB = D / 32;         // 32-element blocks of the output
  constexpr int RB = 2 * D;          // bytes of a staged row of one piece
  constexpr int PB = KT * RB;        // bytes of a staged piece of a tile
  constexpr int TB = NP * PB;        // bytes of a staged tile (K or V)
  constexpr int BPT = TB / 1024;     // 1 KB blocks of it
  constexpr int kMergeBytes = QB * D * 4 + QB * 16;
  constexpr int kTiles = 8 * TB;     // K and V, 2 key groups, 2 buffers
  constexpr int LDS = (kTiles > kMergeBytes ? kTiles : kMergeBytes) + 8 * 128;
  __shared__ __attribute__((aligned(16))) char lds[LDS];
  // [K, V][buffer][key group][TB], then the tiles' units [K, V][buffer][key
  // group][32] floats
  auto tile_buf = [&](int kv, int bf, int g) { return lds + ((kv * 2 + bf) * 2 + g) * TB; };
  auto unit_buf = [&](int kv, int bf, int g) {
    return lds + (LDS - 8 * 128) + ((kv * 2 + bf) * 2 + g) * 128;
  };

  const int G = a.nq / a.nkv;
  const int h = blockIdx.x % a.nkv;
  const int rest = (int)(blockIdx.x / a.nkv);
  const int sp = rest % a.nsplit;              // key split
  const int qb = a.nqb - 1 - rest / a.nsplit;  // latest rows (most keys) first
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int kg = w >> 2, rg = w & 3;
  const int c32 = lane & 31, hh = lane >> 5;
  const int rows = a.M * G;
  const int r0 = qb * QB;
  const int rl = min(r0 + QB, rows) - 1;
  auto t0_of = [&](int m) {
    const int pos = a.pos0 + m;
    int t0 = (a.window > 0 && pos - a.window + 1 > 0) ? pos - a.window + 1 : 0;
    return t0 > a.N ? a.N : t0;
  };
  auto nn_of = [&](int m) { return a.pos0 + m + 1 < a.N ? a.pos0 + m + 1 : a.N; };
  const int kt_lo = t0_of(r0 / G);
  const int kt_hi = nn_of(rl / G);
  const int ntile_all = kt_hi > kt_lo ? (kt_hi - kt_lo + KT - 1) / KT : 0;
  const int tb0 = (int)((int64_t)sp * ntile_all / a.nsplit);
  const int ntile = (int)((int64_t)(sp + 1) * ntile_all / a.nsplit) - tb0;
  const int kt_s = kt_lo + tb0 * KT;
  const int nint = (ntile + 1) / 2;

  const int64_t Rp = wide_padded_rows(a.R);
  const uint16_t* khead = a.pieces + (int64_t)h * wide_head_elems(D, NP, Rp);
  const uint16_t* vhead = khead + (int64_t)a.nkv * wide_head_elems(D, NP, Rp);

  // Staging: wave w of key group 0 copies tile w of an interval's four (K of
  // key groups 0 and 1, V of 0 and 1) in blocks of 1 KB (1024/RB rows): lane
  // l's 16 bytes land at block + 16*l, so it loads the unit the swizzle keeps
  // there.  What is the same in every interval is kept in scalars.  A wave
  // waits where the load path is full; key group 0 has the time (it waits for
  // group 1 at the barrier): 141 -> 135 us (2048-token prompt, 32q/8kv/d128
  // fp32) and 305 -> 294 us (512 tokens after 16384, bf16) against both
  // groups copying.
  constexpr int UPR = D / 8, RPB = 64 / UPR, BPP = KT / RPB;
  const int r_in = lane / UPR, jpos = lane % UPR;
  const int stile = w & 3, sg = stile & 1;
  const bool sv = (w & 3) >= 2;
  const char* shead = uniform_ptr(reinterpret_cast<const char*>(sv ? vhead : khead));
  // lane offset in block 0; block t's rows have the swizzle of row r_in with
  // bits 2.. of K's moved by the block (V's repeats every 4 rows, a block's)
  const uint32_t soff = (uint32_t)(r_in * RB + 16 * (jpos ^ (sv ? wv_f<D>(r_in) : wk_f<D>(r_in))));
  const uint32_t smove = sv ? 0u : ~0u;
  auto lds_addr = [](char* p) {
    return (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)p;
  };
  // Part `part` of `parts` of interval it's staging: the next interval's K
  // tiles and key group 0's V, and key group 1's V of this one.
  auto stage = [&](int it, int part, int parts) {
    const int itu = it + 1;  // the units of every tile of the next interval
    if (part == 0 && lane < KT && itu >= 0 && itu < nint)
      dma4(uniform_ptr(shead + NP * Rp * RB + 4 * (int64_t)(kt_s + (2 * itu + sg) * KT - a.T0)),
           (uint32_t)(4 * lane), lds_addr(unit_buf(sv, itu & 1, sg)));
    const int itv = stile == 3 ? it : it + 1;
    if (itv < 0 || itv >= nint) return;
    const int tk = kt_s + (2 * itv + sg) * KT - a.T0;
    char* buf = tile_buf(sv, itv & 1, sg);
    constexpr int PER = BPT;  // blocks a wave
#pragma unroll
    for (int t = 0; t < PER; ++t) {
      if (t * parts / PER != part) continue;
      const int bi = t;
      const int pc = bi / BPP, rb = (bi % BPP) * RPB;
      dma16(uniform_ptr(shead + (pc * Rp + tk + rb) * RB), soff ^ (smove & (16 * wk_f<D>(t * RPB))),
            lds_addr(buf + bi * 1024));
    }
  };
  if (kg == 0) stage(-1, 0, 1);

  // q pieces of this wave's rows (B operand: lane l row c32, elements
  // 16s + 8*hh .. +7), scaled by scale*log2(e) and, with the row's largest
  // |q|, by a power of two
  const int row = r0 + 32 * rg + c32;
  const bool rv = row < rows;
  const int m = rv ? row / G : 0, g = rv ? row - m * G : 0;
  const int64_t slot = (int64_t)m * a.nq + h * G + g;
  const int rt0 = rv ? t0_of(m) : 0;  // a row past the last: any keys (not stored)
  // the keys end at this split's last tile (an odd count leaves key group 1 a
  // tile past it)
  const int rnn = min(rv ? nn_of(m) : 0x7FFFFFFF, kt_s + ntile * KT);
  f16x8_t qh[QS], ql[QS];
  float qunit;
  {
    const float* qr = a.q + slot * a.dh;
    const float qsc = a.scale * kLog2e;
    float x[QS][8];
    const bool v4 = (a.dh & 3) == 0;
    float qm = 0.f;
#pragma unroll
    for (int s = 0; s < QS; ++s) {
      const int e0 = 16 * s + 8 * hh;
      if (v4) {
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          f32x4 y = {0.f, 0.f, 0.f, 0.f};
          if (rv && e0 + 4 * i < a.dh) y = *reinterpret_cast<const f32x4*>(qr + e0 + 4 * i);
#pragma unroll
          for (int e = 0; e < 4; ++e) x[s][4 * i + e] = y[e] * qsc;
        }
      } else {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          f32x2 y = {0.f, 0.f};
          if (rv && e0 + 2 * i < a.dh) y = *reinterpret_cast<const f32x2*>(qr + e0 + 2 * i);
          x[s][2 * i] = y[0] * qsc;
          x[s][2 * i + 1] = y[1] * qsc;
        }
      }
    }
#pragma unroll
    for (int s = 0; s < QS; ++s)
#pragma unroll
      for (int e = 0; e < 8; ++e) qm = fmaxf(qm, fabsf(x[s][e]));
    const int qshift = f16_row_shift(max_xor32(qm));
    qunit = f16_row_unit(qshift);
#pragma unroll
    for (int s = 0; s < QS; ++s) {
      uint32_t h4[4], l4[4];
#pragma unroll
      for (int e = 0; e < 8; e += 2) split2h(x[s][e], x[s][e + 1], qshift, h4[e / 2], l4[e / 2]);
      qh[s] = __builtin_bit_cast(f16x8_t, u32x4{h4[0], h4[1], h4[2], h4[3]});
      ql[s] = __builtin_bit_cast(f16x8_t, u32x4{l4[0], l4[1], l4[2], l4[3]});
    }
  }

  f32x16 o[DB];
#pragma unroll
  for (int b = 0; b < DB; ++b)
#pragma unroll
    for (int i = 0; i < 16; ++i) o[b][i] = 0.f;
  RowState rs;
  f32x16 s;               // a tile's scores: keys 8*(i/4) + 4*hh + i%4
  uint32_t yh[8], yl[8];  // its y pieces, pairs of the same keys
  float fac = 1.f;
  [[maybe_unused]] float mark = 0.f;  // OWN: NaN once this lane's units held one

  // Scores of this wave's tile of interval it; `copies`: a part of the
  // interval's staging between the products.
  auto scores = [&](int it, auto&& copies) {
    const char* kr = tile_buf(0, it & 1, kg) + c32 * RB;
    const int kx = 16 * (hh ^ wk_f<D>(c32));
#pragma unroll
    for (int i = 0; i < 16; ++i) s[i] = 0.f;
    // a step's operands are read while the last step's products run (the
    // compiler would sink the reads to their use).  The products with a low
    // piece first: they are small beside the others, whose sums alone then
    // round at the scores' size.
    f16x8_t kh[QS], kl[2][2];
    auto read_k = [&](int s0) {
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        kh[s0 + j] = *reinterpret_cast<const f16x8_t*>(kr + (kx ^ (32 * (s0 + j))));
        if constexpr (NP == 2)
          kl[(s0 >> 1) & 1][j] =
              *reinterpret_cast<const f16x8_t*>(kr + PB + (kx ^ (32 * (s0 + j))));
      }
    };
    read_k(0);
#pragma unroll
    for (int s0 = 0; s0 < QS; s0 += 2) {
      if (s0 + 2 < QS) read_k(s0 + 2);
      copies(s0 / 2);
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (NP == 2) {
#pragma unroll
        for (int j = 0; j < 2; ++j) s = mfma32_f16(kl[(s0 >> 1) & 1][j], qh[s0 + j], s);
      }
#pragma unroll
      for (int j = 0; j < 2; ++j) s = mfma32_f16(kh[s0 + j], ql[s0 + j], s);
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int i = 0; i < QS; ++i) s = mfma32_f16(kh[i], qh[i], s);
    __builtin_amdgcn_sched_barrier(0);
  };
  auto soft = [&](int it) {
    const int tk = kt_s + (2 * it + kg) * KT;
    const char* ub = unit_buf(0, it & 1, kg) + 16 * hh;
    const char* vb = unit_buf(1, it & 1, kg) + 16 * hh;
    float x[16], ku[16], vu[16];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const f32x4 y = *reinterpret_cast<const f32x4*>(ub + 32 * i);
      const f32x4 z = *reinterpret_cast<const f32x4*>(vb + 32 * i);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        x[4 * i + e] = s[4 * i + e];
        ku[4 * i + e] = y[e];
        vu[4 * i + e] = z[e];
      }
    }
    if constexpr (OWN)
      mark = fmaf(reinterpret_cast<const float*>(unit_buf(0, it & 1, kg))[c32] +
                      reinterpret_cast<const float*>(unit_buf(1, it & 1, kg))[c32],
                  0.f, mark);
    const bool full = __builtin_amdgcn_ballot_w64(tk < rt0 || tk + KT > rnn) == 0;
    fac = softmax_tile<16>(
        x, ku, vu, qunit, rs, full, [](float v) { return max_xor32(v); },
        [&](int e) {
          const int t = tk + 8 * (e >> 2) + 4 * hh + (e & 3);
          return t < rt0 || t >= rnn;
        },
        yh, yl);
  };
  // O^T += V^T . P^T of the tile of interval it.  A transposed read's 16-lane
  // group (2*h + x) takes keys 16j + 8u + 4h .. +3 (lane/4 of it) of the
  // block's 16 columns 16x ..: slots 4u + i of the A operand, P's key order.
  auto pv = [&](int it) {
    if (__builtin_amdgcn_ballot_w64(fac != 1.f) != 0) {
#pragma unroll
      for (int b = 0; b < DB; ++b)
#pragma unroll
        for (int i = 0; i < 16; ++i) o[b][i] *= fac;
    }
    const int l16 = lane & 15;
    const int rr = 4 * hh + (l16 >> 2);
    const char* vr = tile_buf(1, it & 1, kg) + rr * RB + 32 * ((lane >> 4) & 1) +
                     16 * ((l16 & 3) >> 1) + 8 * (l16 & 1);
    const int vx = 16 * wv_f<D>(rr);
    f16x8_t av[2][2][NP];
    auto read_v = [&](int q) {  // step q: key half j, output blocks b0 and b0 + 1
      const int j = q / (DB / 2), b0 = 2 * (q % (DB / 2));
#pragma unroll
      for (int b = 0; b < 2; ++b)
#pragma unroll
        for (int p = 0; p < NP; ++p) {
          i16x4_t t2[2];
#pragma unroll
          for (int u = 0; u < 2; ++u)
            t2[u] = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                (__attribute__((address_space(3))) i16x4_t*)(
                    vr + p * PB + (16 * j + 8 * u) * RB + ((64 * (b0 + b)) ^ vx)));
          av[q & 1][b][p] = __builtin_bit_cast(
              f16x8_t, __builtin_shufflevector(t2[0], t2[1], 0, 1, 2, 3, 4, 5, 6, 7));
        }
    };
    read_v(0);
#pragma unroll
    for (int q = 0; q < DB; ++q) {
      if (q + 1 < DB) read_v(q + 1);
      __builtin_amdgcn_sched_barrier(0);
      const int j = q / (DB / 2), b0 = 2 * (q % (DB / 2));
      const f16x8_t ph = __builtin_bit_cast(
          f16x8_t, u32x4{yh[4 * j], yh[4 * j + 1], yh[4 * j + 2], yh[4 * j + 3]});
      const f16x8_t pl = __builtin_bit_cast(
          f16x8_t, u32x4{yl[4 * j], yl[4 * j + 1], yl[4 * j + 2], yl[4 * j + 3]});
      auto& vc = av[q & 1];
      if constexpr (NP == 2) {
#pragma unroll
        for (int b = 0; b < 2; ++b) o[b0 + b] = mfma32_f16(vc[b][1], ph, o[b0 + b]);
      }
#pragma unroll
      for (int b = 0; b < 2; ++b) o[b0 + b] = mfma32_f16(vc[b][0], pl, o[b0 + b]);
#pragma unroll
      for (int b = 0; b < 2; ++b) o[b0 + b] = mfma32_f16(vc[b][0], ph, o[b0 + b]);
      __builtin_amdgcn_sched_barrier(0);
    }
  };

  wait_vmcnt<0>();
  __syncthreads();
  constexpr int PARTS = QS / 2;  // staging parts of an interval (steps of the scores)
  for (int it = 0; it < nint; ++it) {
    auto copies = [&](int part) {
      if (kg == 0) stage(it, part, PARTS);
    };
    // wave-uniform; past the group's last tile too: its keys are all masked
    if (kg == 1 && it > 0) pv(it - 1);
    scores(it, copies);
    soft(it);
    if (kg == 0) pv(it);
    wait_vmcnt<0>();  // this wave's copies are in LDS
    lds_barrier();
  }
  if (kg == 1 && nint > 0) pv(nint - 1);
  rs.l = sum_xor32(rs.l);
  float redo = 0.f;  // this key group met a marked row
  if constexpr (OWN) redo = __builtin_amdgcn_ballot_w64(mark != 0.f) != 0 ? 1.f : 0.f;

  // merge of the key groups: group 1's o and (l, m, wsh) through LDS
  lds_barrier();  // every wave is past its tiles
  float* mo = reinterpret_cast<float*>(lds) + rg * 32 * D;  // [rg][block][quad][lane] f32x4
  f32x4* ml = reinterpret_cast<f32x4*>(lds + QB * D * 4) + rg * 32;
  if (kg == 1) {
#pragma unroll
    for (int b = 0; b < DB; ++b)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        *reinterpret_cast<f32x4*>(mo + ((b * 4 + i) * 64 + lane) * 4) =
            f32x4{o[b][4 * i], o[b][4 * i + 1], o[b][4 * i + 2], o[b][4 * i + 3]};
    if (hh == 0) ml[c32] = f32x4{rs.l, rs.m, (float)rs.wsh, redo};
  }
  lds_barrier();
  if (kg == 1) return;
  const f32x4 st = ml[c32];
  if constexpr (OWN) {
    if (redo + st[3] != 0.f) {  // wave-uniform
      own_rows<D>(own_args(), h, r0 + 32 * rg, 32, kt_s, kt_s + ntile * KT, sp);
      return;
    }
  }
  if (!rv) return;
  // both in units of the larger max: factors 2^(m_g - M), times 2^-wsh_g for o
  const float M = fmaxf(rs.m, st[1]);
  const float f0 = exp2_hw(rs.m - M), f1 = exp2_hw(st[1] - M);
  const int e0 = -rs.wsh, e1 = -(int)st[2];
  const float l = fmaf(rs.l, f0, st[0] * f1);
  const bool part = a.nsplit > 1;
  const float inv = l > 0.f ? 1.f / l : 0.f;  // no key: O = 0 (gemm.h:438)
  const int64_t ps = slot * a.nsplit + sp;
  float* po = part ? a.part_o + ps * D : a.o + slot * a.dh;
  const int dh = part ? D : a.dh;
  const bool v4 = (dh & 3) == 0;
#pragma unroll
  for (int b = 0; b < DB; ++b)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const f32x4 z = *reinterpret_cast<const f32x4*>(mo + ((b * 4 + i) * 64 + lane) * 4);
      const int e = 32 * b + 8 * i + 4 * hh;
      f32x4 y;
#pragma unroll
      for (int x = 0; x < 4; ++x) {
        y[x] = fmaf(ldexpf(o[b][4 * i + x], e0), f0, ldexpf(z[x], e1) * f1);
        if (!part) y[x] = div_by(y[x], l, inv);
      }
      if (v4) {
        if (e < dh) *reinterpret_cast<f32x4*>(po + e) = y;
      } else {
        if (e < dh) *reinterpret_cast<f32x2*>(po + e) = f32x2{y[0], y[1]};
        if (e + 2 < dh) *reinterpret_cast<f32x2*>(po + e + 2) = f32x2{y[2], y[3]};
      }
    }
  if (part && hh == 0) {
    a.part_ml[2 * ps] = l > 0.f ? M * kLn2 : -INFINITY;
    a.part_ml[2 * ps + 1] = l;
  }
}

}  // namespace

PfFn prefill_narrow_fn(int D, int kv_dtype, bool own) {
  const bool f32 = kv_dtype == MOLOT_KV_F32;
  if (D == 64) {
    if (own) return f32 ? prefill_narrow_kernel<64, 2, true> : prefill_narrow_kernel<64, 1, true>;
    return f32 ? prefill_narrow_kernel<64, 2, false> : prefill_narrow_kernel<64, 1, false>;
  }
  if (own) return f32 ? prefill_narrow_kernel<128, 2, true> : prefill_narrow_kernel<128, 1, true>;
  return f32 ? prefill_narrow_kernel<128, 2, false> : prefill_narrow_kernel<128, 1, false>;
}
