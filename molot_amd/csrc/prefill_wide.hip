// Causal prefill attention (include/molot/gemm.h:409-446) for wide head dims
// on the matrix cores: 32 query rows a wave, the head dim sliced over waves.
//
// Query rows of one KV head are r = m*G + g (token m at pos0 + m, q head g of
// the group), as in prefill_mfma16_kernel.  A workgroup of 8 waves owns
// 64 of them: wave (rg, sl) takes row group rg (of two) and the 128 elements
// sl*128 .. of the head dim, for the scores and for the output.
// Per tile of 32 keys:
//   1. every wave forms its slice's share of S^T = K . Q^T on
//      v_mfma_f32_32x32x16_f16 (A = K from LDS, B = its q pieces in
//      registers) and leaves it in LDS;
//   2. wave sl owns 32/NSL of the row group's rows: it adds the slices'
//      shares, runs the online softmax over whole rows (lanes of a row side
//      by side, DPP reductions) and leaves P's pieces in LDS, and the factor
//      the rows' o must take when the running max or P's unit moved;
//   3. every wave adds its slice of O^T += V^T . P^T (A = V^T by transposed
//      LDS reads).
// Why this split: a wave's registers hold 32 rows x 128 elements of q pieces
// (64) and of o (64), so two waves a SIMD fit at every D, and each staged K
// or V operand of 1 KB serves 32 rows: 16 rows a wave (prefill_mfma16_kernel)
// would ask 170 bytes a cycle of an LDS that reads 128 at the full matrix
// rate, 32 rows ask 85.
//
// Products: q and p enter as two fp16 pieces of a row scaled by a power of
// two (split2h), K and V as NP such pieces: NP = 2 for fp32 values (three
// products a term, 2^-22 of it dropped), NP = 1 for bf16 and Q8 rows, whose
// values (8 bits; codes of 7) one piece holds exactly down to 2^-28 of the
// row's largest (two products).  A Q8 row's fp32 scale goes into its unit.
//
// Error: PV sums a tile on its own and adds it to o once.  With every product
// added to o, whose roundings then are six a tile of o's size, the error
// against 64 bits (2-norm, 8q/2kv/d512 fp32) was larger than the vector-ALU
// kernel's: 1999 tokens 2.2e-7 against 1.9e-7, now 1.8e-7; 300 after 9000
// 4.9e-7 against 3.5e-7, now 2.8e-7 (bf16 4.0, 3.5 and 2.6; Q8 3.9, 3.0 and
// 2.6).  It costs 1.3 % of the step.
//
// What bounds it (D = 512, fp32, 8q/2kv, a fresh 1999-token prompt; cycles a
// tile, stamped before PV's sums were a tile's own): the three phases'
// latencies, 7200 against the 3072 its 192 products of 32 cycles a SIMD take.
// Scores 3000 and PV 2300 (each 1536 of products, then the barrier, the first
// LDS reads and the stores of the shares), the softmax with the next K copies
// 1900.  The copies go out between products and softmax steps: in a row they
// held each wave ~500 cycles.  The step: 1468 us with each query row streamed by
// the vector-ALU kernel (prefill_rows), 196 us here; of the kernel trace's 215
// this kernel 159, the RoPE/append 33, the merge of the key splits 16, the
// split 7.
#include <hip/hip_runtime.h>

#include "device_util.hpp"
#include "molot_amd/attn_hip.h"
#include "prefill.hpp"
#include "prefill_tile.hpp"
#include "prefill_wide.hpp"

namespace {

// The attended keys [T0, T0 + R) of every KV head as fp16 pieces, in the
// layout of prefill_wide.hpp; the kWideTail rows after them are zeros, so
// that the last tile reads finite values.  Thread: 8 elements of a row, a
// row's D/8 units in consecutive lanes; grid (units / 256, nkv, K or V).
template <int D, typename T, bool PAGED>
__global__ __launch_bounds__(256) void wide_split_kernel(PfArgs a, uint16_t* out) {
  constexpr int NP = wide_pieces_v<T>;
  constexpr int UPR = D / 8;
  const int64_t u = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int64_t Rp = wide_padded_rows(a.R);
  // rows [0, Rsplit), and with the last of them the tail
  if (u >= (a.Rsplit == a.R ? Rp : (int64_t)a.Rsplit) * UPR) return;
  const int h = blockIdx.y, kv = blockIdx.z;
  const int64_t r = u / UPR;
  const int j = (int)(u - r * UPR);
  float x[8] = {};
  float s = 1.f;
  if (r < a.R) s = wide_load8<T, PAGED>(a, kv, h, a.T0 + (int)r, j, x);
  float xm = 0.f;
#pragma unroll
  for (int e = 0; e < 8; ++e) xm = fmaxf(xm, fabsf(x[e]));
  xm = group_max<UPR>(xm);
  float mark = 0.f;
  if (a.own) {
#pragma unroll
    for (int e = 0; e < 8; ++e) mark = fmaf(x[e] * s, 0.f, mark);
    mark = own_mark(xm * s, group_sum<UPR>(mark), kv);
  }
  const int shift = kv ? f16_vrow_shift(xm) : f16_row_shift(xm);
  uint32_t pc[2][4];
#pragma unroll
  for (int e = 0; e < 8; e += 2) split2h(x[e], x[e + 1], shift, pc[0][e / 2], pc[1][e / 2]);
  uint16_t* head = out + ((int64_t)kv * a.nkv + h) * wide_head_elems(D, NP, Rp);
#pragma unroll
  for (int p = 0; p < NP; ++p)
    *reinterpret_cast<u32x4*>(head + (p * Rp + r) * D + 8 * j) =
        u32x4{pc[p][0], pc[p][1], pc[p][2], pc[p][3]};
  if (j == 0)
    reinterpret_cast<float*>(head + NP * Rp * D)[r] =
        (kv ? f16_vrow_unit(xm, shift) : f16_row_unit(shift)) * s + mark;
}

template <int D, int NP>
__global__ __launch_bounds__(512) void prefill_wide_kernel(PfArgs a) {
  constexpr int KT = kWideTile;
  constexpr int NSL = D / 128;       // slices of the head dim
  constexpr int RG = 8 / NSL;        // row groups of 32
  constexpr int QB = 32 * RG;        // query rows a workgroup
  constexpr int RPO = 32 / NSL;      // rows of its group a wave owns in the softmax
  constexpr int LPR = 64 / RPO;      // lanes of an owned row
  constexpr int KPL = KT / LPR;      // keys a lane of it holds
  constexpr int RB = 2 * D;          // bytes of a staged row of one piece
  constexpr int TB = NP * KT * RB;   // bytes of a staged tile (K or V)
  constexpr int SXB = 8 * 4096;      // score shares, then P (8 owner regions)
  constexpr bool DB = 4 * TB + SXB <= 160 * 1024;  // two buffers of K and of V
  constexpr int NB = DB ? 2 : 1;
  constexpr int NL = TB / 1024 / 8;  // 1 KB copies a wave issues per K or V tile
  static_assert(NSL == 4 && KPL == 4, "the layout of the shares and of P");
  static_assert(2 * NB * TB + SXB <= 160 * 1024, "LDS");
  __shared__ __attribute__((aligned(16))) char kbuf[NB][TB];
  __shared__ __attribute__((aligned(16))) char vbuf[NB][TB];
  __shared__ __attribute__((aligned(16))) char sx[SXB];

  const int G = a.nq / a.nkv;
  const int h = blockIdx.x % a.nkv;
  const int rest = (int)(blockIdx.x / a.nkv);
  const int sp = rest % a.nsplit;              // key split
  const int qb = a.nqb - 1 - rest / a.nsplit;  // latest rows (most keys) first
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int rg = w / NSL, sl = w % NSL;
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

  const int64_t Rp = wide_padded_rows(a.R);
  const uint16_t* khead = a.pieces + (int64_t)h * wide_head_elems(D, NP, Rp);
  const uint16_t* vhead = khead + (int64_t)a.nkv * wide_head_elems(D, NP, Rp);

  // K or V of the tile at key tk into LDS: 1 KB blocks of 1024/RB rows, wave
  // w blocks w, w + 8, ...; lane l's 16 bytes land at block + 16*l, so it
  // loads the unit the swizzle keeps there
  auto copy1 = [&](int t, int tk, char* buf, const uint16_t* head, bool isv) {
    constexpr int UPR = D / 8, RPB = 64 / UPR, BPP = KT / RPB;
    const int r_in = lane / UPR, jpos = lane % UPR;
    const int bi = w + 8 * t;  // wave-uniform
    const int pc = bi / BPP, rb = (bi % BPP) * RPB;
    const int ch = jpos ^ (isv ? wv_f<D>(rb + r_in) : wk_f<D>(rb + r_in));
    dma16(head + (pc * Rp + (tk - a.T0) + rb) * D, (uint32_t)(r_in * RB + 16 * ch),
          (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)(buf + bi * 1024));
  };
  auto stage = [&](int tk, char* buf, const uint16_t* head, bool isv) {
#pragma unroll
    for (int t = 0; t < NL; ++t) copy1(t, tk, buf, head, isv);
  };

  if (ntile > 0) {
    stage(kt_s, kbuf[0], khead, false);
    if constexpr (DB) stage(kt_s, vbuf[0], vhead, true);
  }

  // q pieces of this wave's rows and slice (B operand: lane l row c32,
  // elements 16s + 8*hh .. +7 of the slice), scaled by scale*log2(e) and,
  // with the row's largest |q| over all slices, by a power of two
  f16x8_t qh[8], ql[8];
  {
    const int row = r0 + 32 * rg + c32;
    const bool rv = row < rows;
    const int m = rv ? row / G : 0, g = rv ? row - m * G : 0;
    const float* qr = a.q + ((int64_t)m * a.nq + h * G + g) * a.dh;
    const float qsc = a.scale * kLog2e;
    float x[8][8];
    const bool v4 = (a.dh & 3) == 0;
#pragma unroll
    for (int s = 0; s < 8; ++s) {
      const int e0 = 128 * sl + 16 * s + 8 * hh;
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
    float qm = 0.f;
#pragma unroll
    for (int s = 0; s < 8; ++s)
#pragma unroll
      for (int e = 0; e < 8; ++e) qm = fmaxf(qm, fabsf(x[s][e]));
    qm = max_xor32(qm);
    float* qmx = reinterpret_cast<float*>(sx);  // [rg][slice][32 rows]
    if (hh == 0) qmx[(rg * NSL + sl) * 32 + c32] = qm;
    lds_barrier();
#pragma unroll
    for (int s = 0; s < NSL; ++s) qm = fmaxf(qm, qmx[(rg * NSL + s) * 32 + c32]);
    const int qshift = f16_row_shift(qm);
#pragma unroll
    for (int s = 0; s < 8; ++s) {
      uint32_t h4[4], l4[4];
#pragma unroll
      for (int e = 0; e < 8; e += 2) split2h(x[s][e], x[s][e + 1], qshift, h4[e / 2], l4[e / 2]);
      qh[s] = __builtin_bit_cast(f16x8_t, u32x4{h4[0], h4[1], h4[2], h4[3]});
      ql[s] = __builtin_bit_cast(f16x8_t, u32x4{l4[0], l4[1], l4[2], l4[3]});
    }
  }
  // the softmax's row of this lane: row orr of the wave's RPO, keys
  // KPL*oc .. +KPL-1 of a tile
  const int orr = lane / LPR, oc = lane % LPR;
  int rt0, rnn;
  float qunit;
  {
    const int row = r0 + 32 * rg + RPO * sl + orr;
    const bool orv = row < rows;
    const int m = orv ? row / G : 0;
    rt0 = orv ? t0_of(m) : 0;  // a row past the last: any keys (not stored)
    rnn = orv ? nn_of(m) : 0x7FFFFFFF;
    const float* qmx = reinterpret_cast<const float*>(sx);
    float qm = 0.f;
#pragma unroll
    for (int s = 0; s < NSL; ++s) qm = fmaxf(qm, qmx[(rg * NSL + s) * 32 + RPO * sl + orr]);
    qunit = f16_row_unit(f16_row_shift(qm));
  }

  f32x16 o[4];
#pragma unroll
  for (int b = 0; b < 4; ++b)
#pragma unroll
    for (int i = 0; i < 16; ++i) o[b][i] = 0.f;
  RowState rs;  // of the owned row

  // Owner region of rows RPO*ow .. of row group g: 4 KB of sx.  First the
  // score shares [slice][RPO rows][32 keys] floats, a row's 16-byte units
  // (key quads) swizzled so that a store of 8 rows and a read of 16 lanes
  // hit distinct units; then, read by its owner alone, overwritten with P:
  // [piece][key octet][row] 16 bytes, and the rows' (alpha, dsh).
  auto region = [&](int ow) { return sx + (rg * NSL + ow) * 4096; };
  auto swz = [](int rr) { return rr & 7; };
  const int my_ow = c32 / RPO, my_rr = c32 % RPO;  // this lane's MFMA column
  char* s_st = region(my_ow) + sl * (RPO * 128) + my_rr * 128;
  const int s_sw = 16 * (hh ^ swz(my_rr));
  const char* s_ld = region(sl) + orr * 128;
  const int o_sw = 16 * swz(orr);
  const char* p_ld = region(my_ow) + (my_ow & 1) * 128 + my_rr * 16;
  char* p_st = region(sl) + (sl & 1) * 128 + orr * 16;

  const float* kun = reinterpret_cast<const float*>(khead + NP * Rp * D) - a.T0 + KPL * oc;
  const float* vun = reinterpret_cast<const float*>(vhead + NP * Rp * D) - a.T0 + KPL * oc;
  float ku[KPL], vu[KPL];
  auto load_units = [&](int tk) {
    const f32x4_u x = *reinterpret_cast<const f32x4_u*>(kun + tk);
    const f32x4_u y = *reinterpret_cast<const f32x4_u*>(vun + tk);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      ku[e] = x[e];
      vu[e] = y[e];
    }
  };
  float mark = 0.f;  // NaN once a tile's units held one (a row's 8 lanes hold all its keys)
  if (ntile > 0) load_units(kt_s);
  wait_vmcnt<0>();
  __syncthreads();

  for (int it = 0; it < ntile; ++it) {
    const int tk = kt_s + it * KT;
    const bool more = it + 1 < ntile;
    const char* kb = kbuf[DB ? (it & 1) : 0];
    const char* vb = vbuf[DB ? (it & 1) : 0];
    {  // 1. this slice's share of the scores
      f32x16 s2[2];
#pragma unroll
      for (int i = 0; i < 16; ++i) s2[0][i] = s2[1][i] = 0.f;
      const char* kr = kb + c32 * RB + 256 * sl;
      const int kx = 16 * (hh ^ wk_f<D>(c32));
#pragma unroll
      for (int s0 = 0; s0 < 8; s0 += 2) {
        f16x8_t kc[2][NP];
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
          for (int p = 0; p < NP; ++p)
            kc[j][p] = *reinterpret_cast<const f16x8_t*>(kr + p * KT * RB + (kx ^ (32 * (s0 + j))));
        if constexpr (NP == 2) {
#pragma unroll
          for (int j = 0; j < 2; ++j) s2[j] = mfma32_f16(kc[j][1], qh[s0 + j], s2[j]);
        }
        // a quarter of V's copies (one buffer: this tile's, free since the
        // last barrier; two: the next tile's K and V) between the products:
        // issued together they hold a wave until the load path took them
        if constexpr (DB) {
          if (more) {
#pragma unroll
            for (int t = s0 / 2; t < NL; t += 4) {
              copy1(t, tk + KT, kbuf[(it + 1) & 1], khead, false);
              copy1(t, tk + KT, vbuf[(it + 1) & 1], vhead, true);
            }
          }
        } else {
#pragma unroll
          for (int t = s0 / 2; t < NL; t += 4) copy1(t, tk, vbuf[0], vhead, true);
        }
#pragma unroll
        for (int j = 0; j < 2; ++j) s2[j] = mfma32_f16(kc[j][0], ql[s0 + j], s2[j]);
#pragma unroll
        for (int j = 0; j < 2; ++j) s2[j] = mfma32_f16(kc[j][0], qh[s0 + j], s2[j]);
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        f32x4 y;
#pragma unroll
        for (int e = 0; e < 4; ++e) y[e] = s2[0][4 * i + e] + s2[1][4 * i + e];
        *reinterpret_cast<f32x4*>(s_st + (s_sw ^ (32 * i))) = y;
      }
    }
    lds_barrier();  // A: the shares are in LDS, K's buffer is free
    // K's copies of the next tile between the softmax's steps
    auto next_k = [&](int t) {
      if constexpr (!DB) {
        if (more) {
#pragma unroll
          for (int i = 0; i < NL / 4; ++i) copy1(t * (NL / 4) + i, tk + KT, kbuf[0], khead, false);
        }
      }
    };
    {  // 2. softmax of the owned rows
      float sv[KPL];
      {
        f32x4 t = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int s = 0; s < NSL; ++s) {
          const f32x4 y = *reinterpret_cast<const f32x4*>(s_ld + s * (RPO * 128) + (16 * oc ^ o_sw));
          t = s ? t + y : y;
        }
        next_k(0);
#pragma unroll
        for (int e = 0; e < 4; ++e) sv[e] = t[e];
      }
      const int k0 = tk + KPL * oc;
      const bool full = __builtin_amdgcn_ballot_w64(tk < rt0 || tk + KT > rnn) == 0;
      next_k(1);
#pragma unroll
      for (int e = 0; e < KPL; ++e) mark = fmaf(ku[e] + vu[e], 0.f, mark);
      uint32_t yh[KPL / 2], yl[KPL / 2];
      const float fac = softmax_tile<KPL>(
          sv, ku, vu, qunit, rs, full, [](float x) { return group_max<LPR>(x); },
          [&](int e) { return k0 + e < rt0 || k0 + e >= rnn; }, yh, yl);
      next_k(2);
      next_k(3);
      char* d = p_st + (oc >> 1) * 256 + (oc & 1) * 8;
      *reinterpret_cast<u32x2*>(d) = u32x2{yh[0], yh[1]};
      *reinterpret_cast<u32x2*>(d + 1024) = u32x2{yl[0], yl[1]};
      if (oc == 0)
        *reinterpret_cast<f32x4*>(region(sl) + 2048 + 16 * orr) = f32x4{fac, 0.f, 0.f, 0.f};
    }
    if constexpr (!DB) {  // V of this tile is in LDS; K of the next may be in flight
      if (more)
        wait_vmcnt<NL>();
      else
        wait_vmcnt<0>();
    }
    lds_barrier();  // B: P is in LDS
    {  // 3. O^T += V^T . P^T of this slice
      if (more) load_units(tk + KT);  // waited for where the copies are, below
      __builtin_amdgcn_sched_barrier(0);
      const float fac = (*reinterpret_cast<const f32x4*>(region(my_ow) + 2048 + 16 * my_rr))[0];
      f16x8_t yh[2], yl[2];
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        yh[j] = *reinterpret_cast<const f16x8_t*>(p_ld + (2 * j + hh) * 256);
        yl[j] = *reinterpret_cast<const f16x8_t*>(p_ld + 1024 + (2 * j + hh) * 256);
      }
      // transposed reads: 16-lane group (2*h + x) reads keys 16j + 8h + 4u ..
      // +3 (lane/4 of it) of the block's 16 columns 16x .. +15
      const int l16 = lane & 15;
      const char* vr = vb + (8 * hh + (l16 >> 2)) * RB + 256 * sl + 32 * ((lane >> 4) & 1) +
                       16 * ((l16 & 3) >> 1) + 8 * (l16 & 1);
      const int vx = 64 * (l16 >> 2);  // the rows' swizzle (64-byte steps)
      // a tile's sum on its own (the small products first), then one addition to
      // o, under the next block's products: o takes a rounding a tile instead of
      // one a product (error: the kernel's head)
      f32x16 t[2];
#pragma unroll
      for (int b = 0; b < 4; ++b) {
        f16x8_t av[2][NP];
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
          for (int p = 0; p < NP; ++p) {
            i16x4_t t2[2];
#pragma unroll
            for (int u = 0; u < 2; ++u)
              t2[u] = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                  (__attribute__((address_space(3))) i16x4_t*)(
                      vr + p * KT * RB + (16 * j + 4 * u) * RB + ((64 * b) ^ vx)));
            av[j][p] = __builtin_bit_cast(
                f16x8_t, __builtin_shufflevector(t2[0], t2[1], 0, 1, 2, 3, 4, 5, 6, 7));
          }
        f32x16 x;
#pragma unroll
        for (int i = 0; i < 16; ++i) x[i] = 0.f;
        if constexpr (NP == 2) {
#pragma unroll
          for (int j = 0; j < 2; ++j) x = mfma32_f16(av[j][1], yh[j], x);
        }
#pragma unroll
        for (int j = 0; j < 2; ++j) x = mfma32_f16(av[j][0], yl[j], x);
#pragma unroll
        for (int j = 0; j < 2; ++j) x = mfma32_f16(av[j][0], yh[j], x);
        t[b & 1] = x;
        if (b > 0) {
#pragma unroll
          for (int i = 0; i < 16; ++i) o[b - 1][i] = fmaf(o[b - 1][i], fac, t[(b - 1) & 1][i]);
          asm volatile("" : "+v"(o[b - 1]));  // (else all of them sink to the loop's end)
        }
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int i = 0; i < 16; ++i) o[3][i] = fmaf(o[3][i], fac, t[1][i]);
    }
#pragma unroll
    for (int e = 0; e < KPL; ++e)
      asm volatile("" : "+v"(ku[e]), "+v"(vu[e]));  // the units' wait falls here
    wait_vmcnt<0>();  // the next tile's copies (one buffer: K's) are in LDS
    lds_barrier();    // C: V, P and the shares may be overwritten
  }

  // (every wave met the same units: the workgroup decides alike)
  if (__builtin_amdgcn_ballot_w64(mark != 0.f) != 0) {
    own_rows<D>(own_args(), h, r0 + (QB / 8) * w, QB / 8, kt_s, kt_s + ntile * KT, sp);
    return;
  }
  // the rows' (l, m, wsh) from their owners to the waves that hold their o
  rs.l = group_sum<LPR>(rs.l);
  if (oc == 0)
    *reinterpret_cast<f32x4*>(region(sl) + 16 * orr) = f32x4{rs.l, rs.m, (float)rs.wsh, 0.f};
  lds_barrier();
  const f32x4 st = *reinterpret_cast<const f32x4*>(region(my_ow) + 16 * my_rr);
  const int row = r0 + 32 * rg + c32;
  if (row >= rows) return;
  const int m = row / G, g = row - m * G;
  const int64_t slot = (int64_t)m * a.nq + h * G + g;
  const int sh = -(int)st[2];
  if (a.nsplit > 1) {
    const int64_t ps = slot * a.nsplit + sp;
    float* po = a.part_o + ps * D + 128 * sl + 4 * hh;
#pragma unroll
    for (int b = 0; b < 4; ++b)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        f32x4 y;
#pragma unroll
        for (int e = 0; e < 4; ++e) y[e] = ldexpf(o[b][4 * i + e], sh);
        *reinterpret_cast<f32x4*>(po + 32 * b + 8 * i) = y;
      }
    if (sl == 0 && hh == 0) {
      a.part_ml[2 * ps] = st[0] > 0.f ? st[1] * kLn2 : -INFINITY;
      a.part_ml[2 * ps + 1] = st[0];
    }
  } else {
    const float inv = st[0] > 0.f ? 1.f / st[0] : 0.f;  // no key: O = 0 (gemm.h:438)
    float* po = a.o + slot * a.dh;
    const bool v4 = (a.dh & 3) == 0;
#pragma unroll
    for (int b = 0; b < 4; ++b)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int e0 = 128 * sl + 32 * b + 8 * i + 4 * hh;
        f32x4 y;
#pragma unroll
        for (int e = 0; e < 4; ++e) y[e] = div_by(ldexpf(o[b][4 * i + e], sh), st[0], inv);
        if (v4) {
          if (e0 < a.dh) *reinterpret_cast<f32x4*>(po + e0) = y;
        } else {
          if (e0 < a.dh) *reinterpret_cast<f32x2*>(po + e0) = f32x2{y[0], y[1]};
          if (e0 + 2 < a.dh) *reinterpret_cast<f32x2*>(po + e0 + 2) = f32x2{y[2], y[3]};
        }
      }
  }
}

template <int D, typename T>
SplitFn split_of(bool paged) {
  return paged ? wide_split_kernel<D, T, true> : wide_split_kernel<D, T, false>;
}

}  // namespace

SplitFn prefill_wide_split(int D, int kv_dtype, bool paged) {
  auto of = [&](auto d) -> SplitFn {
    constexpr int N = decltype(d)::value;
    if (kv_dtype == MOLOT_KV_Q8) return split_of<N, q8_t>(paged);
    if (kv_dtype == MOLOT_KV_BF16) return split_of<N, bf16_t>(paged);
    return split_of<N, float>(paged);
  };
  if (D == 64) return of(std::integral_constant<int, 64>{});
  if (D == 128) return of(std::integral_constant<int, 128>{});
  return of(std::integral_constant<int, 512>{});
}

PfFn prefill_wide_fn(int D, int kv_dtype) {
  if (D != 512) return nullptr;
  return kv_dtype == MOLOT_KV_F32 ? prefill_wide_kernel<512, 2> : prefill_wide_kernel<512, 1>;
}
