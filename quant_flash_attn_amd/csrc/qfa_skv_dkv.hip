// dKV of the shared-KV attention for query blocks of any length (33 to 128 queries of many heads: qfa_skv_pass.hip):
//     P = exp(sm_scale * Q KV^T - LSE),  dS = sm_scale * P o (dO KV^T - delta),  dKV = P^T dO + dS^T Q,  delta = rowsum(O o dO)
// (quant_flash_attn.py:104-166).
//
// A wave owns 32 keys: their codes, expanded once to binary16 integers code - zero_point (exact), are B operands in
// registers, their dKV^T accumulators too.  Q and dO rows lie in LDS in slabs of 32 bytes and are read both ways: as rows
// for S and dP, transposed for the two accumulations.
//   KEEP    all queries fit (128): the rows are copied and delta is formed once, then every wave walks over its key tiles by
//           itself, the next tile's codes on their way while it works -- no barrier.
//   cycle   longer query blocks: a workgroup takes 128 keys, blocks of 64 queries alternate between the halves of the row
//           area, two barriers per 64 queries.
// The kernel before it copied and summed the rows once per 128 keys, met at two barriers per 32 queries (52 % of its time was
// waiting) and removed the codes' offset by two more MFMAs per block.  Measured, that one -> this (us, one GPU): 5247 heads, 97 x 689
// 941 -> 668 at head_dim 128, 497 -> 327 at 64; 512 heads, 512 x 4096 1565 -> 1180 and 842 -> 599.  Up to 64 queries it had its rows
// resident too and was 7 to 9 % faster at 128 (1470 heads, 47 x 2737: 532 against 572; so many heads go to qfa_skv_pass.hip now).
// What bounds it: at 512 queries the matrix pipe is busy 45 % at 1.89 GHz, issue stalls 37 %; the S and dP of the next block
// beside the vector work of this one (32 registers more) changed nothing.  At 97 x 689 it is busy 33 % with 41 % waits: 16 KB
// of rows and 16 KB transposed out of LDS for 32 products, and the last block of 32 queries holds one.
#include "qfa_host.h"
#include "qfa_skv_common.h"

namespace qfa {

struct SkvDkvArgs {
  const _Float16 *q, *o, *dout;
  const int8_t *codes; const void *scale; const int8_t *zp;
  const float *lse;
  void *dkv;
  const float *grad_scale;     // nullable device scalar: dkv is multiplied by it before rounding
  int64_t H;
  int Nq, Nk, BH, grad_bf16, scale_dtype;
  int direct, q_bf16, do_bf16;   // resident rows only: q, o and dO as the caller has them, dO scaled here (no grad_scale)
  int wgs_per_bh, tiles_per_wg;
  int64_t sqb, sqh, sqn, scb, sch, scn, sob, soh, son, sdob, sdoh, sdon, sdkb, sdkh, sdkn;
  float sm_scale, sm_scale_log2;
};

template <int D> struct SkvDkvGeom {
  static constexpr int RB = 4, ROWS = 32 * RB;     // blocks of 32 queries, rows that fit
  static constexpr int CPR = D / 16, SLAB = ROWS * 32 + 128, MAT = CPR * SLAB;   // slabs, one matrix
  static constexpr int OFF_STAT = 2 * MAT, OFF_STAGE = OFF_STAT + 2 * ROWS * 4, STAGE = 32 * 64;
  static constexpr int TOTAL = OFF_STAGE + 4 * STAGE;
};

template <int D, bool KEEP> __global__ __launch_bounds__(256, D == 256 ? 1 : D == 128 ? 2 : 3) void skv_dkv_kernel(SkvDkvArgs a) {
  typedef SkvDkvGeom<D> GM;
  constexpr int CPR = GM::CPR, SLAB = GM::SLAB, DB = D / 32, KD = D / 16, RB = GM::RB;
  __shared__ __attribute__((aligned(256))) unsigned char smem[GM::TOTAL];

  const XcdBlock id(a.BH, a.wgs_per_bh);
  if (!id.live) return;
  const int bh = id.bh, part = id.sub;
  const int64_t b = index_div(bh, a.H), h = bh - b * a.H;
  const int tid = threadIdx.x, lane = tid % 64, lr = lane % 32, g = lane / 32;
  const int wave = __builtin_amdgcn_readfirstlane(tid / 64);
  const int nqb = (a.Nq + 31) / 32, ntiles = (a.Nk + 31) / 32;
  const int64_t tk0 = (int64_t)bh * a.Nk, tq0 = (int64_t)bh * a.Nq;
  const unsigned char *codes_bh = reinterpret_cast<const unsigned char *>(a.codes + b * a.scb + h * a.sch);
  const _Float16 *q_bh = a.q + b * a.sqb + h * a.sqh, *d_bh = a.dout + b * a.sdob + h * a.sdoh, *o_bh = a.o + b * a.sob + h * a.soh;
  float *stat = reinterpret_cast<float *>(smem + GM::OFF_STAT);   // -lse in log2 units, -delta * sm_scale

  // ---- rows of query block qb -> block `at` of the row area; rows past Nq arrive as zeros
  auto copy_rows = [&](int qb, int at) __attribute__((always_inline)) {
    const int rows = min(32, a.Nq - 32 * qb), r = lane / 2;
    const rsrc_t rq = make_rsrc(q_bh + (int64_t)32 * qb * a.sqn, (unsigned)(((rows - 1) * (int)a.sqn + D) * 2));
    const rsrc_t rd = make_rsrc(d_bh + (int64_t)32 * qb * a.sdon, (unsigned)(((rows - 1) * (int)a.sdon + D) * 2));
    const int half = ((lane % 2) ^ (r >> 3 & 1)) * 16;
    const int oq = r * (int)a.sqn * 2 + half, od = r * (int)a.sdon * 2 + half;
#pragma unroll
    for (int i = 0; i < CPR / 4; ++i) {
      const int s = wave + 4 * i;
      unsigned char *dst = smem + s * SLAB + at * 1024;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rq, (lptr_t)dst, 16, oq + s * 32, 0, 0, 0);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rd, (lptr_t)(dst + GM::MAT), 16, od + s * 32, 0, 0, 0);
    }
  };
  // delta and LSE of RPT-row groups: 256 / TPR rows from row r0 of the sequence on, in rows a0.. of the row area; O comes
  // and the LSE from memory (`of`, `lse`, loaded before), dO from the row area
  constexpr int TPR = KEEP ? 2 : 4, OC = D / 8 / TPR;   // threads per row, 8-element chunks per thread
  auto load_o = [&](int r0, u32x4 (&of)[OC], float &lse) __attribute__((always_inline)) {
    const int row = min(r0 + tid / TPR, a.Nq - 1);
    lse = a.lse[tq0 + row];
#pragma unroll
    for (int k = 0; k < OC; ++k) of[k] = *reinterpret_cast<const u32x4 *>(o_bh + (int64_t)row * a.son + 8 * (tid % TPR + TPR * k));
  };
  auto dout_of = [&](int ra, int k) __attribute__((always_inline)) -> u32x4 {   // chunk k of a thread's row
    const int c = tid % TPR + TPR * k;
    return *reinterpret_cast<const u32x4 *>(smem + GM::MAT + c / 2 * SLAB + ra * 32 + (((c % 2) ^ (ra >> 3 & 1)) << 4));
  };
  auto set_stat = [&](int r0, int ra, float delta, float lse) __attribute__((always_inline)) {
    if (tid % TPR != 0) return;
    const bool live = r0 + tid / TPR < a.Nq;
    stat[ra] = live ? -lse * kLog2e : -INFINITY;   // padding rows: p = 0
    stat[GM::ROWS + ra] = live ? -a.sm_scale * delta : 0.f;
  };
  auto stats = [&](int r0, int a0, const u32x4 (&of)[OC], float lse) __attribute__((always_inline)) {
    const int ra = a0 + tid / TPR;
    float sum = 0.f;
#pragma unroll
    for (int k = 0; k < OC; ++k) {
      const u32x4 dv = dout_of(ra, k);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const unsigned dw = dv[e], ow = of[k][e];
        sum += lo_to_f32<_Float16>(ow) * lo_to_f32<_Float16>(dw) + hi_to_f32<_Float16>(ow) * hi_to_f32<_Float16>(dw);
      }
    }
#pragma unroll
    for (int m = 1; m < TPR; m *= 2) sum += __shfl_xor(sum, m, 64);
    set_stat(r0, ra, sum, lse);
  };

  // ---- a tile of 32 keys: codes on their way (raw), then as B operands (column = key lr; k-steps 2j, 2j + 1 and k-group g
  // hold columns 32j + 16g + {0..7} and {8..15})
  u32x4 raw[D / 32];
  unsigned raw_z = 0u, raw_s = 0u;
  auto load_tile = [&](int t) __attribute__((always_inline)) {
    const int rows = min(32, a.Nk - 32 * t);
    const rsrc_t rk = make_rsrc(codes_bh + (int64_t)32 * t * a.scn, (unsigned)((rows - 1) * (int)a.scn + D));
#pragma unroll
    for (int j = 0; j < D / 32; ++j)
      raw[j] = __builtin_amdgcn_raw_buffer_load_b128(rk, lr * (int)a.scn + (2 * j + g) * 16, 0, 0);
    const int key = min(32 * t + lr, a.Nk - 1);
    raw_z = (unsigned char)a.zp[tk0 + key];
    if (a.scale_dtype == QFA_F32) raw_s = static_cast<const unsigned *>(a.scale)[tk0 + key];
    else raw_s = static_cast<const unsigned short *>(a.scale)[tk0 + key];
  };
  u32x4 cb[KD];
  float a_sk = 0.f, sm_k = 0.f;
  auto expand_tile = [&]() __attribute__((always_inline)) {
    const unsigned nz = 0xe400u | (raw_z ^ 0x80u), nz2 = nz | nz << 16;   // -(1152 + zero_point), twice
    const f16x2 neg = __builtin_bit_cast(f16x2, nz2);
#pragma unroll
    for (int j = 0; j < D / 32; ++j)
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        const u32x4 m = expand_codes(raw[j][2 * k], raw[j][2 * k + 1]);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const unsigned me = m[e];
          cb[2 * j + k][e] = __builtin_bit_cast(unsigned, __builtin_bit_cast(f16x2, me) + neg);
        }
      }
    const unsigned sw = raw_s;
    const float sk = a.scale_dtype == QFA_F32 ? __builtin_bit_cast(float, sw)
                     : a.scale_dtype == QFA_F16 ? lo_to_f32<_Float16>(sw) : lo_to_f32<__bf16>(sw);
    a_sk = a.sm_scale_log2 * sk;
    sm_k = a.sm_scale * sk;
  };

  // ---- per-lane offsets inside a block of rows: rows (lane = row lr, slab g, half 0 or 1), transposing reads (rows
  // 4g + {0..3} of slabs u; rows 8 further have their halves swapped)
  const int s16 = lane % 16, u16 = lane / 16 % 2;
  const int row_l = g * SLAB + lr * 32 + ((lr >> 3 & 1) << 4);
  const unsigned tr_l = lds_addr(smem) + u16 * SLAB + (4 * g + s16 / 4) * 32 + (s16 % 4 / 2) * 16 + (s16 % 2) * 8;

  f32x16 acc[DB];
  auto clear = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[db][v] = 0.f;
  };
  // contributions of the query block at block `at` of the row area
  auto add_block = [&](int at) __attribute__((always_inline)) {
    const unsigned char *rows = smem + at * 1024;
    f32x16 s, dp;
#pragma unroll
    for (int v = 0; v < 16; ++v) s[v] = 0.f, dp[v] = 0.f;
#pragma unroll
    for (int m = 0; m < KD; ++m) {
      const unsigned char *p = rows + m / 2 * 2 * SLAB + (row_l ^ (m % 2 * 16));
      s = mfma_h(*reinterpret_cast<const u32x4 *>(p), cb[m], s);
      dp = mfma_h(*reinterpret_cast<const u32x4 *>(p + GM::MAT), cb[m], dp);
    }
    const unsigned tr = tr_l + at * 1024;
    u32x2 fr[2][2][2];   // [dO, Q][16-query half][rows, rows + 8]
    auto request = [&](int db) __attribute__((always_inline)) {
#pragma unroll
      for (int hh = 0; hh < 2; ++hh) {
        const unsigned x = tr + 2 * db * SLAB + hh * 512;
        constexpr int IMM = GM::MAT < 65536 ? GM::MAT : 0;   // (what fits an instruction's offset)
        fr[0][hh][0] = lds_read_tr16_async<IMM>(x + (GM::MAT - IMM));
        fr[0][hh][1] = lds_read_tr16_async<IMM>((x ^ 16) + 256 + (GM::MAT - IMM));
        fr[1][hh][0] = lds_read_tr16_async<0>(x);
        fr[1][hh][1] = lds_read_tr16_async<0>((x ^ 16) + 256);
      }
    };
    request(0);
    u32x4 pf[2], df[2];
#pragma unroll
    for (int aa = 0; aa < 4; ++aa) {
      const f32x4 nl = *reinterpret_cast<const f32x4 *>(stat + 32 * at + 8 * aa + 4 * g);
      const f32x4 nd = *reinterpret_cast<const f32x4 *>(stat + GM::ROWS + 32 * at + 8 * aa + 4 * g);
      float p[4], ds[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        p[e] = __builtin_amdgcn_exp2f(__builtin_fmaf(a_sk, s[4 * aa + e], nl[e]));
        ds[e] = p[e] * __builtin_fmaf(sm_k, dp[4 * aa + e], nd[e]);
      }
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        pf[aa / 2][2 * (aa % 2) + e] = pack_h2(p[2 * e], p[2 * e + 1]);
        df[aa / 2][2 * (aa % 2) + e] = pack_h2(ds[2 * e], ds[2 * e + 1]);
      }
    }
#pragma unroll
    for (int db = 0; db < DB; ++db) {
      lds_wait_all();
      u32x2 now[2][2][2];
#pragma unroll
      for (int x = 0; x < 8; ++x) now[x / 4][x / 2 % 2][x % 2] = tie(fr[x / 4][x / 2 % 2][x % 2]);
      if (db + 1 < DB) request(db + 1);
#pragma unroll
      for (int hh = 0; hh < 2; ++hh) {
        const u32x2(&d)[2] = now[0][hh], (&q)[2] = now[1][hh];
        acc[db] = mfma_h(u32x4{d[0][0], d[0][1], d[1][0], d[1][1]}, pf[hh], acc[db]);
        acc[db] = mfma_h(u32x4{q[0][0], q[0][1], q[1][0], q[1][1]}, df[hh], acc[db]);
      }
    }
  };
  float osc = a.grad_scale ? *a.grad_scale : 1.0f;
  // the tile's rows leave through 2 KB of LDS as whole 128-byte lines: 64 columns of 16 rows at a time
  auto write_tile = [&](int t, unsigned char *stage) __attribute__((always_inline)) {
    unsigned short *out = static_cast<unsigned short *>(a.dkv) + b * a.sdkb + h * a.sdkh + (int64_t)32 * t * a.sdkn;
    const int rows = a.Nk - 32 * t;
    int w = lr % 16 * 128 + 8 * g, r = lane / 8 * 128 + ((lane % 8 ^ lane / 8) << 4);
    asm volatile("" : "+v"(w), "+v"(r));
#pragma unroll
    for (int db = 0; db < DB; db += 2)
#pragma unroll
      for (int hf = 0; hf < 2; ++hf) {
        if (lr / 16 == hf) {
#pragma unroll
          for (int x = 0; x < 8; ++x) {
            const f32x16 &c = acc[db + x / 4];
            const int v = 4 * (x % 4);
            const float x0 = c[v] * osc, x1 = c[v + 1] * osc, x2 = c[v + 2] * osc, x3 = c[v + 3] * osc;
            const u32x2 o2 = a.grad_bf16 ? u32x2{pack2<__bf16>(x0, x1), pack2<__bf16>(x2, x3)}
                                         : u32x2{pack2<_Float16>(x0, x1), pack2<_Float16>(x2, x3)};
            *reinterpret_cast<u32x2 *>(stage + w + ((x ^ (lr % 8)) << 4)) = o2;
          }
        }
        // (a wave's LDS operations complete in order)
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          const u32x4 x = *reinterpret_cast<const u32x4 *>(stage + r + i * 1024);
          const int j = 16 * hf + 8 * i + lane / 8;
          if (j < rows) *reinterpret_cast<u32x4 *>(out + (int64_t)j * a.sdkn + 32 * db + 8 * (lane % 8)) = x;
        }
      }
  };

  if (KEEP) {
    int t = part * a.tiles_per_wg + wave;
    const int t_end = min(ntiles, (part + 1) * a.tiles_per_wg);
    const int key0 = part * a.tiles_per_wg * 32;
    const KeyScaleMax scales(a.scale, a.scale_dtype, tk0 + key0, a.direct ? min(a.tiles_per_wg * 32, a.Nk - key0) : 1, tid);
    if (t < t_end) load_tile(t);
    for (int qb = 0; qb < nqb; ++qb) copy_rows(qb, qb);
    u32x4 of[OC];
    float lse;
    load_o(0, of, lse);
    dma_wait();
    __syncthreads();
    if (a.direct) {   // cast and scaled in place: a thread has 16 bytes of every slab
      const bool live = tid < 64 * nqb;
      unsigned char *mine = smem + tid * 16;
      float *red = reinterpret_cast<float *>(smem + GM::OFF_STAGE);
      u32x4 w[CPR];
#pragma unroll
      for (int s = 0; s < CPR; ++s) w[s] = live ? *reinterpret_cast<const u32x4 *>(mine + GM::MAT + s * SLAB) : u32x4{0u, 0u, 0u, 0u};
      if (a.q_bf16) {
#pragma unroll
        for (int i = 0; i < OC; ++i) of[i] = half_of_bf16(of[i]);
      }
      // delta of the rows as they came: times 2^k it is that of the scaled ones, and what bounds k where O comes from all keys
      // of the head and the scales from a part of them
      u32x4 dr[OC];
#pragma unroll
      for (int i = 0; i < OC; ++i) dr[i] = dout_of(tid / TPR, i);
      float delta = dot_dout(of, dr, a.do_bf16);
#pragma unroll
      for (int m = 1; m < TPR; m *= 2) delta += __shfl_xor(delta, m, 64);
      const float md = a.wgs_per_bh > 1 && tid / TPR < a.Nq ? finite_abs(a.sm_scale * delta) : 0.f;
      const int k = block_dout_exponent(max_abs_dout(w, a.do_bf16), scales.get(), md, red);
      set_stat(0, tid / TPR, delta * exp2_neg(-k), lse);
      scale_dout(w, a.do_bf16, k);
      osc = exp2_neg(k);
      if (live) {
#pragma unroll
        for (int s = 0; s < CPR; ++s) *reinterpret_cast<u32x4 *>(mine + GM::MAT + s * SLAB) = w[s];
        if (a.q_bf16) {
#pragma unroll
          for (int s = 0; s < CPR; ++s) {
            u32x4 *q = reinterpret_cast<u32x4 *>(mine + s * SLAB);
            *q = half_of_bf16(*q);
          }
        }
      }
    } else {
      stats(0, 0, of, lse);
    }
    __syncthreads();
    for (; t < t_end; t += 4) {
      expand_tile();
      if (t + 4 < t_end) load_tile(t + 4);
      clear();
      for (int qb = 0; qb < nqb; ++qb) add_block(qb);
      write_tile(t, smem + GM::OFF_STAGE + wave * GM::STAGE);
    }
    return;
  }

  // ---- cycle: 64 queries (HB blocks) at a time in the halves of the row area
  constexpr int HB = RB / 2;
  const int t = part * 4 + wave;
  const bool t_ok = t < ntiles;   // (a wave without a tile still takes part in copies and barriers)
  const int ngroups = (nqb + HB - 1) / HB;
  u32x4 of[OC];
  float lse;
  auto fetch = [&](int grp) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < HB; ++i)
      if (HB * grp + i < nqb) copy_rows(HB * grp + i, HB * (grp & 1) + i);
    load_o(32 * HB * grp, of, lse);
  };
  if (t_ok) load_tile(t);
  fetch(0);
  if (t_ok) expand_tile();
  clear();
  for (int grp = 0; grp < ngroups; ++grp) {
    dma_wait();
    __syncthreads();   // the group's rows have landed
    stats(32 * HB * grp, 32 * HB * (grp & 1), of, lse);
    __syncthreads();   // its statistics are there, and everybody is done with the group before it
    if (grp + 1 < ngroups) fetch(grp + 1);
    if (t_ok)
      for (int i = 0; i < HB; ++i)
        if (HB * grp + i < nqb) add_block(HB * (grp & 1) + i);
  }
  if (t_ok) write_tile(t, smem + GM::OFF_STAGE + wave * GM::STAGE);
}

template <int D> static int launch_d(const SkvAttnArgs &x, hipStream_t st) {
  SkvDkvArgs a;
  a.q = static_cast<const _Float16 *>(x.q); a.o = static_cast<const _Float16 *>(x.o);
  a.dout = static_cast<const _Float16 *>(x.dout);
  a.codes = x.codes; a.scale = x.scale; a.zp = x.zp; a.lse = x.lse; a.dkv = x.dkv;
  a.grad_scale = x.grad_scale; a.grad_bf16 = x.grad_dtype == QFA_BF16; a.scale_dtype = x.scale_dtype;
  a.direct = x.direct; a.q_bf16 = x.io_dtype == QFA_BF16; a.do_bf16 = x.dout_dtype == QFA_BF16;
  a.H = x.H; a.Nq = (int)x.Nq; a.Nk = (int)x.Nk;
  a.sqb = x.sqb; a.sqh = x.sqh; a.sqn = x.sqn; a.scb = x.scb; a.sch = x.sch; a.scn = x.scn;
  a.sob = x.sob; a.soh = x.soh; a.son = x.son; a.sdob = x.sdob; a.sdoh = x.sdoh; a.sdon = x.sdon;
  a.sdkb = x.sdkb; a.sdkh = x.sdkh; a.sdkn = x.sdkn;
  a.sm_scale = x.sm_scale;
  a.sm_scale_log2 = x.sm_scale * kLog2e;
  if (x.B * x.H > 0x7fffffffLL) return set_error(QFA_EUNSUPPORTED, "attn_bwd_shared_kv: too many (batch, head) pairs");
  a.BH = (int)(x.B * x.H);
  const bool keep = x.Nq <= SkvDkvGeom<D>::ROWS;
  // resident rows: a workgroup walks over as many chunks of four tiles as leave about 2048 workgroups
  const int64_t chunks = (x.Nk + 127) / 128;
  int64_t cpw = 1;
  if (keep) {
    const int64_t want = (chunks * a.BH + 2047) / 2048;
    cpw = want < 1 ? 1 : want > chunks ? chunks : want;
  }
  a.wgs_per_bh = (int)((chunks + cpw - 1) / cpw);
  a.tiles_per_wg = (int)(4 * cpw);
  const int64_t total = xcd_grid(a.BH, a.wgs_per_bh);
  if (total > 0x7fffffffLL) return set_error(QFA_EUNSUPPORTED, "attn_bwd_shared_kv: too many blocks for one launch");
  if (keep) skv_dkv_kernel<D, true><<<dim3((unsigned)total), dim3(256), 0, st>>>(a);
  else skv_dkv_kernel<D, false><<<dim3((unsigned)total), dim3(256), 0, st>>>(a);
  return check_launch("qfa_attn_bwd_shared_kv (dKV)");
}

int launch_skv_dkv(const SkvAttnArgs &x, hipStream_t st) {
  return x.D == 128 ? launch_d<128>(x, st) : launch_d<64>(x, st);
}

}  // namespace qfa
