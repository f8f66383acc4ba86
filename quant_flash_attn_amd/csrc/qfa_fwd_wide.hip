// Forward kernel with one wave per SIMD (see qfa_fwd.hip for the contract and the arithmetic: INT8 scores, zero-point
// correction as one extra MFMA, reference maximum that is only moved when a running sum says so).
//
// A workgroup is 4 waves; a wave owns QB blocks of 32 queries, whose O^T accumulators live in AccVGPRs by hand (qfa_acc.h).
// Keys stream through LDS in tiles of 64, three buffers, one barrier per tile; the LDS layout is the slab layout of the
// backward kernels (qfa_bwd_dkv.inc).  A step (32 keys) is one straight line whose MFMAs come in the order
//     P.V of the previous step, all but its last fragment  |  S of the next step  |  last fragment of P.V
// with the vector work of this step's P dealt to them at an even pace.  Every LDS request is issued three fragments before
// its use, behind the compiler's back, and waited for by count (LDS returns in order).
//
// QB is 1 at head_dim 256 and 2 at 128: eight accumulator tiles either way.  At head_dim 256 the compiler's version of
// qfa_fwd.hip moved scores and accumulators between the register files, 3800 moves in the kernel.  Bound by the waits for
// the tiles (27 % of a wave's time: with 53 KB per tile three buffers leave a copy one tile's time to land) and by the
// instructions one wave can issue; the matrix pipe is busy 44 % of the time (4096 x 4096, 32 heads of 256: 467 us at 2.03 GHz,
// 589 TFLOP/s, from 590 us).  Fragments requested seven MFMAs ahead instead of three changed nothing; at head_dim 128 two waves
// per SIMD of one block each were 4 - 6 % slower than qfa_fwd.hip.
//
// Scores start from a bias whose sum is a float already and the correction takes the bias out (qfa_acc.h): no conversion,
// and one MFMA less than the biased accumulators of qfa_fwd.hip.
#include <type_traits>

#include "qfa_acc.h"
#include "qfa_bwd_common.h"
#include "qfa_fwd_common.h"

namespace qfa {

template <int D> struct FwdWideSmem {
  static constexpr int TILE = 64, SLAB = TILE * 32 + 128;
  static constexpr int OFF_K = 0, OFF_V = OFF_K + D / 32 * SLAB, OFF_C = OFF_V + D / 16 * SLAB,
                       BUF = OFF_C + TILE * 8 + TILE * 4;   // constants: correction digits (2 dwords per key), key scale
  static_assert(BUF % 256 == 0 && 3 * BUF <= 160 * 1024, "three tile buffers");
};

template <typename T, int D, int QB, bool CAUSAL, bool SPLIT> __global__ __launch_bounds__(256, 1) void fwd_wide_kernel(FwdArgs a) {
#ifdef __HIP_DEVICE_COMPILE__   // (with the body in view the host pass of this compiler emits no launch stub)
  typedef FwdWideSmem<D> SM;
  constexpr int TILE = SM::TILE, NSTEP = TILE / 32, SLAB = SM::SLAB;
  constexpr int KS = D / 32, DB = D / 32, KD = D / 16;
  constexpr int QUERIES = 32 * QB;   // queries per wave
  __shared__ __attribute__((aligned(256))) unsigned char smem[3 * SM::BUF];

  // ---- block -> (batch*head, query block): as in qfa_fwd.hip, longest rows first and a group of heads at a time
  const int L = blockIdx.x;
  const int vid = (L % 8) * a.blocks_per_xcd + (L / 8);
  if (vid >= a.total_blocks) return;
  int bh = vid / a.mblocks;
  int mb = vid % a.mblocks;
  int split = 0, key0 = 0;
  if (SPLIT) {   // the keys of a query block in a.splits parts, as in qfa_fwd.hip
    split = bh % a.splits;
    bh /= a.splits;
    key0 = split * a.keys_per_split;
  }
  const int Nk = SPLIT ? min(a.keys_per_split, a.Nk - key0) : a.Nk;
  if (CAUSAL && !SPLIT) {
    const int gsz = 1 << a.group_log2;
    const int pb = bh >> a.group_log2 << a.group_log2;
    if (pb + gsz <= a.total_blocks / a.mblocks) {
      const int idx = (bh - pb) * a.mblocks + mb;
      bh = pb + (idx & (gsz - 1));
      mb = idx >> a.group_log2;
    }
    mb = a.mblocks - 1 - mb;
  }
  const int64_t b = index_div(bh, a.H), h = bh - b * a.H;
  const int m0 = mb * 4 * QUERIES;
  const int tid = threadIdx.x, lane = tid % 64, lr = lane % 32, g = lane / 32;
  const int wave = __builtin_amdgcn_readfirstlane(tid / 64);
  const int q_first = m0 + wave * QUERIES;

  const int8_t *qc_bh = a.qc + b * a.sqb + h * a.sqh;
  const unsigned char *kc_bh = reinterpret_cast<const unsigned char *>(a.kc + b * a.skb + h * a.skh + key0 * a.skn);
  const unsigned char *v_bh = reinterpret_cast<const unsigned char *>(reinterpret_cast<const T *>(a.v) + b * a.svb + h * a.svh + key0 * a.svn);
  const int64_t tq0 = (int64_t)bh * a.Nq, tk0 = (int64_t)bh * a.Nk + key0;

  const int coff = CAUSAL ? a.Nk - a.Nq - key0 : 0;   // causal: query i keeps keys j <= i + coff (mask aligned to the last key)
  const int ntiles = ((CAUSAL ? min(Nk, m0 + 4 * QUERIES + coff) : Nk) + TILE - 1) / TILE;
  const int wtiles = q_first >= a.Nq ? 0 : ((CAUSAL ? min(Nk, q_first + QUERIES + coff) : Nk) + TILE - 1) / TILE;

  // ---- tile copies (direct to LDS); the per-key constants through registers, key = lane, the same in every wave
  typedef SlabCopy<TILE, KS> CopyK;
  typedef SlabCopy<TILE, KD> CopyV;
  const CopyK cp_k(lane, (unsigned)a.skn);
  const CopyV cp_v(lane, (unsigned)a.svn * 2u);
  constexpr int PIECES = CopyK::N + CopyV::N;
  const rsrc_t rs_sk = make_rsrc(a.sk + tk0, (unsigned)Nk * 4u);
  const rsrc_t rs_rk = make_rsrc(a.rk + tk0, (unsigned)Nk * 4u);
  const rsrc_t rs_zk = make_rsrc(a.zk + tk0, (unsigned)Nk);
  struct TileDesc { rsrc_t k, v; unsigned char *dst; };
  auto tile_desc = [&](int t) __attribute__((always_inline)) -> TileDesc {
    const int rows = t < ntiles ? min(TILE, Nk - TILE * t) : 0;
    return {cp_k.desc(kc_bh + (int64_t)t * TILE * a.skn, rows), cp_v.desc(v_bh + (int64_t)t * TILE * a.svn * 2, rows),
            smem + t % 3 * SM::BUF};
  };
  auto copy_piece = [&](const TileDesc &d, int i) __attribute__((always_inline)) {   // i: a compile-time constant everywhere
    if (i < CopyK::N) cp_k.piece(i, d.k, d.dst + SM::OFF_K, wave);
    else cp_v.piece(i - CopyK::N, d.v, d.dst + SM::OFF_V, wave);
  };
  auto copy_tile = [&](int t) __attribute__((always_inline)) {
    const TileDesc d = tile_desc(t);
#pragma unroll
    for (int i = 0; i < PIECES; ++i) copy_piece(d, i);
  };
  float c_sk;
  int c_rk, c_zk;
  auto load_kc = [&](int t) __attribute__((always_inline)) {   // (keys past the end read as zero and are masked)
    c_sk = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rs_sk, lane * 4, t * TILE * 4, 0));
    c_rk = __builtin_amdgcn_raw_buffer_load_b32(rs_rk, lane * 4, t * TILE * 4, 0);
    c_zk = (int)(signed char)__builtin_amdgcn_raw_buffer_load_b8(rs_zk, lane, t * TILE, 0);
  };
  auto store_kc = [&](int buf) __attribute__((always_inline)) {
    *reinterpret_cast<u32x2 *>(smem + buf + SM::OFF_C + lane * 8) = u32x2{base128_pair<T>(c_rk), pack2<T>((float)c_zk, (float)c_zk)};
    *reinterpret_cast<float *>(smem + buf + SM::OFF_C + TILE * 8 + lane * 4) = c_sk;
  };
  copy_tile(0);
  copy_tile(1);
  load_kc(0);

  // ---- this lane's queries: codes as B operands for the whole kernel, correction operand
  constexpr int SH = D > 128 ? 8 : 7;   // bits per digit of rq - D*zq (see qfa_fwd.hip)
  i32x4 qf[QB][KS];
  u32x2 corr_q[QB];
  float a_i[QB];
  int k_hi[QB];      // last key that the lane's query sees
#pragma unroll
  for (int qb = 0; qb < QB; ++qb) {
    const int qi = q_first + 32 * qb + lr, qc = min(qi, a.Nq - 1);
    k_hi[qb] = CAUSAL ? min(qc + coff, Nk - 1) : Nk - 1;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
      qf[qb][ks] = *reinterpret_cast<const i32x4 *>(qc_bh + (int64_t)qc * a.sqn + ks * 32 + g * 16);
    const int zq = (int)a.zq[tq0 + qc], c = a.rq[tq0 + qc] - D * zq;
    const int hi = c >> SH, lo = c & ((1 << SH) - 1);
    corr_q[qb][0] = g == 0 ? pack2<T>((float)(-zq), (float)(-zq)) : pack2<T>((float)(-(hi * (1 << SH))), (float)(-lo));
    corr_q[qb][1] = g == 0 ? QFA_BIAS_B(T) : 0u;
    a_i[qb] = a.sq[tq0 + qc] * a.sm_scale_log2;   // > 0
  }
  store_kc(0);
  load_kc(1);

  // ---- per-lane read offsets (see qfa_bwd_dkv.inc): rows, transposing reads
  const int row_l = slab_row(lr, g);
  const int s16 = lane % 16, u16 = (lane / 16) % 2;
  const int tr_l = u16 * SLAB + (4 * g + s16 / 4) * 32 + ((s16 % 4) / 2) * 16 + (s16 % 2) * 8;
  const unsigned lds0 = lds_addr(smem);
  const unsigned k_l = lds0 + SM::OFF_K + row_l, v_l = lds0 + SM::OFF_V + tr_l, ck_l = lds0 + SM::OFF_C + (2 * lr + g) * 4,
                 sk_l = lds0 + SM::OFF_C + TILE * 8 + 16 * g;

  // accumulators: O^T of (query block qb, columns 32db) in tile qb * DB + db
  static_assert(QB * DB == 8, "eight tiles, then the V fragments");
  acc_zero<8>();

  i32x16 bias, si[QB];     // si: scores of the step in work, biased integers without the zero-point term
#pragma unroll
  for (int v = 0; v < 16; ++v) bias[v] = QFA_BIAS_BITS;
  typedef u32x4 Prob[QB][2];
  Prob pf[2];              // probabilities of the previous step and of this one, by turns
#pragma unroll
  for (int qb = 0; qb < QB; ++qb)
#pragma unroll
    for (int hh = 0; hh < 2; ++hh) pf[0][qb][hh] = u32x4{0u, 0u, 0u, 0u};

  float m_ref[QB], nm[QB], l_run[QB];   // reference maximum of u = score / a_i, -a_i * m_ref, the lane's share of the row sum
#pragma unroll
  for (int qb = 0; qb < QB; ++qb) { m_ref[qb] = -INFINITY; nm[qb] = 0.f; l_run[qb] = 0.f; }

  auto ld = [&](int off) -> u32x4 { return *reinterpret_cast<const u32x4 *>(smem + off); };

  // scores of step (tile buffer buf, part mbk) of query block qb from scratch: u = score / a_i, masked; their maximum
  auto scores = [&](int qb, int t, int buf, int mbk, float (&u)[16]) __attribute__((always_inline)) -> float {
    i32x16 s = bias;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
      s = mfma_i8(__builtin_bit_cast(i32x4, ld(buf + SM::OFF_K + row_l + mbk * 1024 + ks * SLAB)), qf[qb][ks], s);
    const unsigned dg = *reinterpret_cast<const unsigned *>(smem + buf + SM::OFF_C + (2 * lr + g) * 4 + mbk * 256);
    const f32x16 f = mfma_16b_k8<T>(u32x2{dg, QFA_BIAS_A(T)}, corr_q[qb], __builtin_bit_cast(f32x16, s));
    float mt = -INFINITY;
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      const int jl = 32 * mbk + 8 * (v / 4) + 4 * g + v % 4;
      const float x = f[v] * *reinterpret_cast<const float *>(smem + buf + SM::OFF_C + TILE * 8 + jl * 4);
      u[v] = TILE * t + jl <= k_hi[qb] ? x : -INFINITY;
      mt = fmaxf(mt, u[v]);
    }
    return mt;
  };

  // LDS fragments in the order of their use: P.V of the previous step 0 .. XA-1, S of the next step, P.V fragment XA (NX-1),
  // then P.V of the next step; V fragments are two requests, K fragments one.  Position n is requested behind the first MFMA
  // of position n - AHEAD.
  constexpr int NX = 2 * DB, XA = NX - 1, XZ = XA + KS, NF = XZ + 1, SLOTS = QB * NF, RING = 4,
                AHEAD = RING - 1;
  static_assert(NF % RING == 0 && XA - AHEAD >= RING, "a step starts with the fragment registers where the one before left them");
  u32x4 fk[RING];          // K fragments (V fragments: AccVGPRs, they are in flight where a step may branch)
  unsigned dg_k;           // correction digits of the step's key row
  auto request_v = [&](unsigned v0, auto n_tag, auto pos_tag) __attribute__((always_inline)) {   // hh = n / DB, db = n % DB
    constexpr int n = decltype(n_tag)::value;
    acc_request<decltype(pos_tag)::value % RING, 2 * (n % DB) * SLAB + 16 * (n / DB) * 32>(v0, v0 ^ 16u);
  };

  // One step: 32 keys (part mbk of the tile in buffer `buf`) against the wave's queries.  `nbuf`: buffer of the next step;
  // v_prev: the lane's address of the V rows of the previous step; vis: which query blocks saw any of its keys.
  auto body = [&](int t, int buf, int nbuf, unsigned v_prev, auto mbk_tag, auto masked_tag, const Prob &pin, Prob &pout)
                  __attribute__((always_inline)) {
    constexpr bool MASKED = decltype(masked_tag)::value;
    constexpr int mbk = decltype(mbk_tag)::value;
    constexpr bool LAST = mbk == NSTEP - 1;
    const int nmbk = LAST ? 0 : mbk + 1;
    const unsigned v_cur = v_l + buf + mbk * 1024, k_next = k_l + nbuf + nmbk * 1024;
    const int j0 = TILE * t + 32 * mbk;
    constexpr int P_LO = AHEAD * QB, HALF = 16 * QB;   // (the scales are there at position AHEAD)
    f32x16 f[QB];
    f32x4 sk[4];          // key scales of rows 8aa + 4g + {0..3}
    float x0, x1, l[QB];
    // 16 QB half items: scaling of a pair of scores and packing of the pair before it (even), exponentials (odd)
    auto pack_pair = [&](auto x_tag) __attribute__((always_inline)) {
      constexpr int x = decltype(x_tag)::value, qb = x / 8, y = x % 8;
      const unsigned w = pack2<T>(x0, x1);
      pout[qb][y / 4][y % 4] = w;
      l[qb] = y == 0 ? dot2_ones_keep<T>(w, l_run[qb]) : dot2_ones<T>(w, l[qb]);   // sum of the rounded pair, fp32
    };
    auto half_item = [&](auto i_tag) __attribute__((always_inline)) {
      constexpr int i = decltype(i_tag)::value, x = i / 2, qb = x / 8, v = 2 * (x % 8);
      if constexpr (i % 2 == 0) {
        if constexpr (x > 0) pack_pair(ic<x - 1>{});
        x0 = __builtin_fmaf(a_i[qb], f[qb][v] * sk[v / 4][v % 4], nm[qb]);
        x1 = __builtin_fmaf(a_i[qb], f[qb][v + 1] * sk[v / 4][v % 4 + 1], nm[qb]);
      } else {
        x0 = __builtin_amdgcn_exp2f(x0);
        x1 = __builtin_amdgcn_exp2f(x1);
        if constexpr (MASKED) {
          const int j = j0 + 4 * g + 8 * (v / 4) + v % 4;
          x0 = j <= k_hi[qb] ? x0 : 0.f;
          x1 = j + 1 <= k_hi[qb] ? x1 : 0.f;
        }
      }
    };
    TileDesc td;
    constexpr int BAR = RING, CSLOTS = SLOTS - QB * BAR;   // the turn of the tile is behind BAR fragments, the copies behind it
    auto work = [&](auto slot_tag) __attribute__((always_inline)) {
      constexpr int s = decltype(slot_tag)::value;
      if constexpr (s >= P_LO) {
        constexpr int n = SLOTS - P_LO, i0_ = (s - P_LO) * HALF / n, i1_ = (s - P_LO + 1) * HALF / n;
        static_for<i1_ - i0_>([&](auto k) __attribute__((always_inline)) { half_item(ic<i0_ + decltype(k)::value>{}); });
      }
      if constexpr (LAST && s >= QB * BAR) {
        constexpr int c = s - QB * BAR, p0 = c * PIECES / CSLOTS, p1 = (c + 1) * PIECES / CSLOTS;
        static_for<p1 - p0>([&](auto p) __attribute__((always_inline)) { copy_piece(td, p0 + decltype(p)::value); });
      }
    };
    auto request = [&](auto n_tag) __attribute__((always_inline)) {
      constexpr int n = decltype(n_tag)::value;
      if constexpr (n < XA) request_v(v_prev, n_tag, n_tag);
      else if constexpr (n < XZ) fk[n % RING] = lds_read_b128_async<(n - XA) * SLAB>(k_next);
      else if constexpr (n == XZ) request_v(v_prev, ic<XA>{}, n_tag);
      else request_v(v_cur, ic<n - NF>{}, n_tag);
    };
    // requests that may still be in flight at position n: those of the AHEAD - 1 positions behind it (the constants come on
    // top: they are only waited for longer)
    auto later = [](int n) constexpr {
      int c = 0;
      for (int i = n + 1; i < n + AHEAD; ++i) c += i >= XA && i < XZ ? 1 : 2;
      return c;
    };
    // query blocks that saw none of the previous step's keys skip its P.V: their probabilities are zeros, and V may hold
    // anything there
    bool vis[QB];
#pragma unroll
    for (int qb = 0; qb < QB; ++qb) vis[qb] = !MASKED || !CAUSAL || j0 - 32 <= q_first + 32 * qb + 31 + coff;
    auto pv = [&](auto n_tag, auto pos_tag, auto qb_tag) __attribute__((always_inline)) {
      constexpr int n = decltype(n_tag)::value, pos = decltype(pos_tag)::value, qb = decltype(qb_tag)::value;
      if (!MASKED || vis[qb]) acc_mfma_frag<T, qb * DB + n % DB, pos % RING>(pin[qb][n / DB]);
    };

    if constexpr (LAST) {   // the next tile has landed as far as this wave copied it
      dma_wait();
      store_kc(nbuf);
      td = tile_desc(t + 2);
    }
#pragma unroll
    for (int qb = 0; qb < QB; ++qb) f[qb] = mfma_16b_k8<T>(u32x2{dg_k, QFA_BIAS_A(T)}, corr_q[qb], __builtin_bit_cast(f32x16, si[qb]));
    static_for<NF>([&](auto n_tag) __attribute__((always_inline)) {
      constexpr int n = decltype(n_tag)::value;
      // the turn of the tile: position n - 1 was requested behind the constants' stores, so these are done too; the buffer of
      // the previous tile was last read in the step before this one; the first read of the next tile is still to come
      if constexpr (LAST && n == BAR) {
        asm volatile("s_barrier" ::: "memory");
        load_kc(t + 2);
      }
      if constexpr (n >= XA && n < XZ) lds_wait_for<later(n)>(fk[n % RING]);
      else lds_wait_for<later(n)>();
      if constexpr (n == AHEAD) lds_tie(sk);
      static_for<QB>([&](auto qb_tag) __attribute__((always_inline)) {
        constexpr int qb = decltype(qb_tag)::value;
        QFA_FENCE();
        if constexpr (n < XA) pv(ic<n>{}, n_tag, qb_tag);
        else if constexpr (n < XZ) si[qb] = mfma_i8(__builtin_bit_cast(i32x4, fk[n % RING]), qf[qb][n - XA], n == XA ? bias : si[qb]);
        else pv(ic<XA>{}, n_tag, qb_tag);
        QFA_FENCE();
        if constexpr (qb == 0) {
          // constants, each in front of a request that is waited for before their use
          if constexpr (n == XZ - AHEAD) dg_k = lds_read_b32_async(ck_l + nbuf + nmbk * 256);
          if constexpr (n == 0)
            static_for<4>([&](auto aa) __attribute__((always_inline)) {
              sk[decltype(aa)::value] = __builtin_bit_cast(f32x4, lds_read_b128_async<decltype(aa)::value * 32>(sk_l + buf + mbk * 128));
            });
          request(ic<n + AHEAD>{});
        }
        work(ic<QB * n + qb>{});
      });
    });
    pack_pair(ic<8 * QB - 1>{});
    lds_tie(dg_k);   // (arrived: the last fragment was requested behind it)
    QFA_FENCE();
    // Some lane's sum left the range below (its scores outgrew the reference by about 2^60, or overflowed): the step's scores
    // are formed again, the reference moved -- at least far enough to bring the sum so far back to order one -- and with it
    // O and the row sum.  The tile is still in LDS.
    bool over = false;
#pragma unroll
    for (int qb = 0; qb < QB; ++qb) over |= !(l[qb] <= 0x1p60f);
    if (__builtin_expect(__builtin_amdgcn_ballot_w64(over) != 0, 0)) {
      acc_settle();
      static_for<QB>([&](auto qb_tag) __attribute__((always_inline)) {
        constexpr int qb = decltype(qb_tag)::value;
        float u[16];
        float mt = fmaxf(scores(qb, t, buf, mbk, u), m_ref[qb] + __log2f(fmaxf(l_run[qb], 1.0f)) / a_i[qb]);
        const float m_new = fmaxf(m_ref[qb], max_across_halves(mt));
        float alpha = __builtin_amdgcn_exp2f(a_i[qb] * (m_ref[qb] - m_new));
        if (SPLIT && m_ref[qb] == m_new) alpha = 1.0f;   // also of a row without keys: -inf both
        m_ref[qb] = m_new;
        nm[qb] = SPLIT && m_new == -INFINITY ? 0.f : -a_i[qb] * m_new;
        l[qb] = l_run[qb] * alpha;
        acc_scale<qb * DB, DB>(alpha);
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const float p0 = __builtin_amdgcn_exp2f(__builtin_fmaf(a_i[qb], u[2 * e], nm[qb]));
          const float p1 = __builtin_amdgcn_exp2f(__builtin_fmaf(a_i[qb], u[2 * e + 1], nm[qb]));
          pout[qb][e / 4][e % 4] = pack2<T>(p0, p1);
          l[qb] = dot2_ones<T>(pout[qb][e / 4][e % 4], l[qb]);
        }
      });
      acc_settle();
    }
#pragma unroll
    for (int qb = 0; qb < QB; ++qb) l_run[qb] = l[qb];
  };

  dma_wait();
  __syncthreads();
  int t = 0, buf = 0, nbuf = SM::BUF;
  if (wtiles > 0) {
    // the first step: reference maximum (every query sees key 0, or no key of its split), raw scores, constants and first fragments
#pragma unroll
    for (int qb = 0; qb < QB; ++qb) {
      float u[16];
      m_ref[qb] = max_across_halves(scores(qb, 0, 0, 0, u));
      nm[qb] = SPLIT && m_ref[qb] == -INFINITY ? 0.f : -a_i[qb] * m_ref[qb];
      si[qb] = bias;
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) si[qb] = mfma_i8(__builtin_bit_cast(i32x4, ld(row_l + SM::OFF_K + ks * SLAB)), qf[qb][ks], si[qb]);
    }
    dg_k = lds_read_b32_async(ck_l);
    lds_wait_for<0>(dg_k);
    unsigned v_prev = v_l;     // (the probabilities are zero: the product adds nothing)
    static_for<AHEAD>([&](auto n) __attribute__((always_inline)) { request_v(v_prev, n, n); });
    // full tiles, then masked ones (diagonal, ragged end)
    auto tiles = [&](int t_end, auto masked_tag) __attribute__((always_inline)) {
      for (; t < t_end; ++t) {
        static_for<NSTEP>([&](auto mbk_tag) __attribute__((always_inline)) {
          constexpr int mbk = decltype(mbk_tag)::value;
          body(t, buf, mbk == NSTEP - 1 ? nbuf : buf, v_prev, mbk_tag, masked_tag, pf[mbk % 2], pf[(mbk + 1) % 2]);
          v_prev = v_l + buf + mbk * 1024;
        });
        const int b2 = 3 * SM::BUF - buf - nbuf;
        buf = nbuf;
        nbuf = b2;
      }
    };
    tiles(min(wtiles, min(Nk / TILE, CAUSAL ? (q_first + coff + 1) / TILE : wtiles)), std::false_type{});
    tiles(wtiles, std::true_type{});
    // P.V of the last step (fragments 0 .. AHEAD-1 are under way)
    const int j_last = TILE * wtiles - 32;
    static_for<NX>([&](auto n_tag) __attribute__((always_inline)) {
      constexpr int n = decltype(n_tag)::value;
      lds_wait_for<2 * (NX - 1 - n < AHEAD - 1 ? NX - 1 - n : AHEAD - 1)>();
      static_for<QB>([&](auto qb_tag) __attribute__((always_inline)) {
        constexpr int qb = decltype(qb_tag)::value;
        if (!CAUSAL || j_last <= q_first + 32 * qb + 31 + coff)
          acc_mfma_frag<T, qb * DB + n % DB, n % RING>(pf[0][qb][n / DB]);
      });
      if constexpr (n + AHEAD < NX) request_v(v_prev, ic<n + AHEAD>{}, ic<n + AHEAD>{});
    });
  }
  for (; t < ntiles; ++t) {   // tiles that only other waves see
    dma_wait();
    lds_barrier();
    copy_tile(t + 2);
  }
  dma_wait();
  acc_settle();
  __syncthreads();   // the tile buffers are done with: the output stages overlay them
  static_assert(4 * 32 * 2 * D <= 3 * SM::BUF, "output staging fits the tile buffers");
  unsigned char *stage = smem + wave * (32 * 2 * D);
  T *o_bh = reinterpret_cast<T *>(a.o) + b * a.sob + h * a.soh;
  static_for<QB>([&](auto qb_tag) __attribute__((always_inline)) {
    constexpr int qb = decltype(qb_tag)::value;
    const float l_tot = l_run[qb] + swap32_f(l_run[qb]);
    const int qi = q_first + 32 * qb + lr;
    if constexpr (SPLIT) {
      const int64_t at = tq0 * a.splits + split;
      acc_store_rows_f32<D, qb * DB>(1.0f, a.po + at * D, (int64_t)a.splits * D, q_first + 32 * qb, a.Nq, lane);
      if (qi < a.Nq && g == 0) *reinterpret_cast<f32x2 *>(a.pml + 2 * (at + (int64_t)qi * a.splits)) = f32x2{a_i[qb] * m_ref[qb], l_tot};
      return;
    }
    if (a.o32) acc_store_rows_f32<D, qb * DB>(1.0f / l_tot, a.o32 + tq0 * D, D, q_first + 32 * qb, a.Nq, lane);
    if (a.o) acc_store_rows<T, D, qb * DB>(1.0f / l_tot, stage, o_bh, a.son, q_first + 32 * qb, a.Nq, lane, a.o_once);
    if (qi < a.Nq && g == 0) a.lse[tq0 + qi] = (a_i[qb] * m_ref[qb] + __log2f(l_tot)) * kLn2;
  });
#endif
}

template <typename T, int D, int QB> static int launch_wide(FwdArgs a, int64_t BH, bool causal, hipStream_t st) {
  a.mblocks = (a.Nq + 128 * QB - 1) / (128 * QB);
  const int64_t total = (int64_t)a.mblocks * BH * a.splits;
  if (total > 0x3fffffffLL) return set_error(QFA_EUNSUPPORTED, "attn_fwd: too many query blocks for one launch");
  a.total_blocks = (int)total;
  a.blocks_per_xcd = (a.total_blocks + 7) / 8;
  const dim3 grid((unsigned)(a.blocks_per_xcd * 8));
  if constexpr (D == 256) {
    if (a.splits > 1) {
      if (causal) fwd_wide_kernel<T, D, QB, true, true><<<grid, dim3(256), 0, st>>>(a);
      else fwd_wide_kernel<T, D, QB, false, true><<<grid, dim3(256), 0, st>>>(a);
      return check_launch("qfa_attn_fwd");
    }
    if (causal) fwd_wide_kernel<T, D, QB, true, false><<<grid, dim3(256), 0, st>>>(a);
    else fwd_wide_kernel<T, D, QB, false, false><<<grid, dim3(256), 0, st>>>(a);
  } else {
    if (causal) return set_error(QFA_EUNSUPPORTED, "attn_fwd: no wide kernel for a mask at this head_dim");
    fwd_wide_kernel<T, D, QB, false, false><<<grid, dim3(256), 0, st>>>(a);
  }
  return check_launch("qfa_attn_fwd");
}

template <typename T, int D> int launch_fwd_wide(FwdArgs a, int64_t BH, bool causal, hipStream_t st) {
  return launch_wide<T, D, D == 128 ? 2 : 1>(a, BH, causal, st);
}
template int launch_fwd_wide<__bf16, 128>(FwdArgs, int64_t, bool, hipStream_t);
template int launch_fwd_wide<__bf16, 256>(FwdArgs, int64_t, bool, hipStream_t);
template int launch_fwd_wide<_Float16, 128>(FwdArgs, int64_t, bool, hipStream_t);
template int launch_fwd_wide<_Float16, 256>(FwdArgs, int64_t, bool, hipStream_t);

}  // namespace qfa
