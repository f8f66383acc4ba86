// Shared-KV attention for query blocks of more than 16 queries: forward and dQ on tiles of keys that the whole workgroup
// expands once.  (The backward of 33 to 128 queries of many heads: qfa_skv_pass.hip.)
//     O = softmax(sm_scale * Q K^^T) K^,   dQ = dS K^,   K^ = V^ = scale * (codes - zero_point)  per token
// (quant_flash_attn.py:22-83 and 104-166; Q and dO stay in binary16).
//
// Why kernels of their own.  The 16-query kernels expand every code twice per 16 queries (row operands and transposed
// operands): 560 vector instructions per 32 x 32 block of scores in the forward beside 18 MFMAs' worth of products.  Here the
// four waves together turn a tile of 64 keys into binary16 integers code - zero_point (exact) in LDS; both operand orders come
// out of that tile (plain and transposing reads), nothing has to be corrected afterwards, and a block takes 114 vector
// instructions and 16 MFMAs.
//
// Work split.  A wave takes 32 queries.  Four waves side by side (128 queries) leave every tile expanded once for all of them;
// two (64 queries) share the keys of a tile with the other two and their partial results meet in LDS.  With few workgroups the
// keys are split over several of them (qfa_skv_plan.cpp).  The codes of the tile after the next are on their way in registers
// while a tile is worked on.  The forward makes the scores of the next block beside the probabilities of this one (three
// tiles in LDS); the same pipeline in dQ costs 35 KB more LDS and gained nothing (head_dim 128, before the scaling moved in: 384
// against 421 us).
//
// What bounds them.  Long blocks (512 heads, 512 queries, 4096 keys of 128): the forward's matrix pipe is busy 47 % and its vector
// pipe 54 % of the time at 1.86 GHz, 42 % of the LDS cycles are used, dQ 47, 49 and 28 %; one workgroup per CU already reaches
// nine tenths of what two do: power and issue, not latency.  Short ones (5247 heads, 97 queries, 689 keys): matrix pipe 39 and 38 %,
// waits 27 and 36 %: eleven tiles between a workgroup's start and end, and the fourth block of 32 queries holds one.
// Measured, 16-query kernels -> these (us, one GPU): 5247 heads, 97 x 689: forward 538 -> 298, dQ with the scaling of dO 679 -> 439
// at head_dim 128, 333 -> 186 and 420 -> 248 at 64; 512 heads, 512 x 4096: 1069 -> 566 and 1141 -> 831 (128), 670 -> 349 and 732 ->
// 476 (64); 256 heads of 256: forward 997 -> 601 (dQ stays with the 16-query kernel).
#include <type_traits>

#include "qfa_host.h"
#include "qfa_merge.h"
#include "qfa_skv_tile.h"

namespace qfa {

struct SkvTileArgs {
  const void *q; const int8_t *codes; const void *scale; const int8_t *zp;
  void *o; float *lse;
  const _Float16 *dout; void *dq; const float *grad_scale;   // dQ only
  int direct, do_bf16;   // dQ: q, o (io_bf16) and dO as the caller has them, dO scaled here (grad_scale is not used)
  int64_t H;
  int Nq, Nk, BH;
  int io_bf16, scale_dtype, grad_bf16;
  int64_t sqb, sqh, sqn, scb, sch, scn, sob, soh, son, sdob, sdoh, sdon, sdqb, sdqh, sdqn;
  float sm_scale, sm_scale_log2;
  int qwgs, bpw;               // workgroups per (batch, head) and blocks of 32 queries per workgroup (at most QW)
  int splits, tiles_per_split; // forward: workgroups that share the keys
  float *po, *pml;
};

// A wave takes 32 queries; QW waves side by side take different queries, the 4 / QW groups of them different keys of a tile.
template <int D, int QW> struct SkvTileGeom {
  static constexpr int KW = 4 / QW;
  static constexpr int NB = QW == 4 ? 2 : 1;      // blocks of 32 keys per wave and tile
  static constexpr int TK = 32 * NB * KW;         // keys per tile
  static constexpr int CPR = D / 16;              // 16-code chunks per row = slabs of 16 columns
  static constexpr int SLAB = TK * 32 + 128;      // a slab: 32 bytes of every row; slabs are 128 bytes apart modulo 256
  static constexpr int TILE = CPR * SLAB, BUF = TILE + TK * 4;   // expanded tile, key scales
  static constexpr int MERGE = (D / 2 + 2) * 256; // partial result of a wave: O^T accumulators, m, l
  static_assert((KW - 1) * QW * MERGE <= 2 * BUF && 4 * 64 * D <= 2 * BUF, "merge and output areas overlay the tiles");
};
template <int D, int QW> __global__ __launch_bounds__(256, D == 256 ? 1 : D == 128 ? 2 : 3) void skv_tile_fwd_kernel(SkvTileArgs a) {
  typedef SkvTileGeom<D, QW> GM;
  constexpr int TK = GM::TK, NB = GM::NB, KW = GM::KW, DB = D / 32, KD = D / 16;
  constexpr bool AHEAD = NB == 2;   // row fragments requested a body ahead (the next tile's second block is in LDS by then)
  // A tile's codes are on their way for one tile of products, or (EARLY) go to LDS in the middle of a tile and are requested a tile
  // earlier; the second tile's are requested beside the first's (BOTH) or behind them.  At head_dim 256 with four waves side by side,
  // one wave per SIMD, nobody fills that wait (256 heads, 512 x 4096: 752 -> 601 us; 1584 heads, 97 x 689: 275 -> 224).  With four
  // waves at 128 and 64, two and three per SIMD, EARLY costs 2 and 14 %; with two waves it gains up to 4 % there (5247 heads, 40 x 300 of
  // 128: 121 -> 116) and nothing at 256, where BOTH costs 5 % of short calls (256 heads, 64 x 512: 25.0 -> 26.2)
  constexpr bool EARLY = D == 256 ? NB == 2 : NB == 1, BOTH = D < 256 || NB == 2;
  constexpr int VA = D == 256 ? 4 : D == 128 ? 3 : 2;   // blocks of 32 columns of the transposed fragments requested ahead
  __shared__ __attribute__((aligned(256))) unsigned char smem[3 * GM::BUF];

  const XcdBlock id(a.BH, a.qwgs * a.splits);
  if (!id.live) return;
  const int64_t b = index_div(id.bh, a.H), h = id.bh - b * a.H;
  const int tid = threadIdx.x, lane = tid % 64, lr = lane % 32, g = lane / 32;
  const int wave = __builtin_amdgcn_readfirstlane(tid / 64);
  const int split = id.sub / a.qwgs;
  // (turned by the workgroup: waves without queries should not all sit on the same SIMD)
  const int slot = (wave + id.bh + id.sub) % QW, kw = wave / QW;
  const int qb = id.sub % a.qwgs * a.bpw + slot;
  const bool active = slot < a.bpw && 32 * qb < a.Nq;

  const unsigned char *codes_bh = reinterpret_cast<const unsigned char *>(a.codes + b * a.scb + h * a.sch);
  const int64_t tk0 = (int64_t)id.bh * a.Nk, tq0 = (int64_t)id.bh * a.Nq;
  const int t0 = split * a.tiles_per_split, nt = min(a.tiles_per_split, (a.Nk + TK - 1) / TK - t0);

  typedef SkvTileStage<D, TK, GM::SLAB> Stage;
  Stage st, st1;
  st.init((unsigned)a.scn, tid);
  auto issue = [&](Stage &x, int t) __attribute__((always_inline)) {
    const int64_t k0 = (int64_t)(t0 + t) * TK;
    x.issue(codes_bh + k0 * a.scn, a.scale, a.scale_dtype == QFA_F32, a.zp, tk0 + k0, a.scn, a.Nk - (int)k0);
  };
  st1 = st;
  issue(st, 0);
  if (BOTH && nt > 1) issue(st1, 1);

  const int qi = 32 * qb + lr;
  u32x4 qf[KD];
  skv_load_row<D>(a.q, b * a.sqb + h * a.sqh + (int64_t)min(qi, a.Nq - 1) * a.sqn, a.io_bf16, g, qf);
  const SkvTileReads<GM::SLAB> rd(lane);

  f32x16 acc[DB];
#pragma unroll
  for (int db = 0; db < DB; ++db)
#pragma unroll
    for (int v = 0; v < 16; ++v) acc[db][v] = 0.f;
  const float a_s = a.sm_scale_log2;
  // Key j enters with w_j = scale_j * sm_scale * log2(e): the exponent of p is s_j * w_j - m, and w_j serves as V's scale
  // too, its constant factor a_s taken out of the sums at the end.  The reference sits where that factor times p is a power
  // of two, so that p' = p * w_j of the key it is taken from is its scale itself, exact in binary16.
  const float limit = 16.0f / a_s;   // a_s * p <= 2^4: p' stays inside binary16 for any fp16 K
  const float unit = -__log2f(a_s);
  float m_ref = NO_KEY, nm = unit - NO_KEY, l_run = 0.f;   // m_ref in log2 units
  f32x16 s;      // scores of the block in work, in code units
  f32x4 sk[4];   // its w

  u32x4 kf[KD];   // rows of the keys whose scores are made next
  auto request_keys = [&](const unsigned char *p) __attribute__((always_inline)) {
#pragma unroll
    for (int m = 0; m < KD; ++m) kf[m] = rd.rows(p, m);
  };
  auto scores = [&]() __attribute__((always_inline)) {
    f32x16 r;
#pragma unroll
    for (int v = 0; v < 16; ++v) r[v] = 0.f;
#pragma unroll
    for (int m = 0; m < KD; ++m) r = mfma_h(kf[m], qf[m], r);
    return r;
  };
  // w of 32 keys from row kr of the tile in buf
  auto request_w = [&](const unsigned char *buf, int kr) __attribute__((always_inline)) {
#pragma unroll
    for (int aa = 0; aa < 4; ++aa) sk[aa] = *reinterpret_cast<const f32x4 *>(buf + GM::TILE + (kr + 8 * aa + 4 * g) * 4);
  };
  // krem: keys that exist from the block's first on
  auto mask = [&](int krem) __attribute__((always_inline)) {
    if (krem < 32) {
#pragma unroll
      for (int v = 0; v < 16; ++v) s[v] = 8 * (v / 4) + 4 * g + v % 4 >= krem ? -INFINITY : s[v];
    }
  };
  u32x4 pf[2];
  auto probs = [&]() __attribute__((always_inline)) -> float {
    float sum = 0.f;
#pragma unroll
    for (int x = 0; x < 8; ++x) {
      const int v = 2 * x;
      const float p0 = __builtin_amdgcn_exp2f(__builtin_fmaf(s[v], sk[v / 4][v % 4], nm)),
                  p1 = __builtin_amdgcn_exp2f(__builtin_fmaf(s[v + 1], sk[v / 4][v % 4 + 1], nm));
      sum += p0 + p1;
      pf[x / 4][x % 4] = pack_h2(p0 * sk[v / 4][v % 4], p1 * sk[v / 4][v % 4 + 1]);
    }
    return sum;
  };
  // One block of 32 keys (rows kr of buf), whose scaled scores are in s; those of the next one (rows nkr of nbuf) are made
  // beside its probabilities
  auto body = [&](const unsigned char *buf, int kr, const unsigned char *nbuf, int nkr, int nkrem, const unsigned char *nnext) __attribute__((always_inline)) {
    const unsigned char *p = buf + kr * 32;
    if (!AHEAD) request_keys(nbuf + nkr * 32);
    u32x4 vf[DB][2];
#pragma unroll
    for (int db = 0; db < VA; ++db)
#pragma unroll
      for (int hh = 0; hh < 2; ++hh) vf[db][hh] = rd.cols(p, db, hh);
    const f32x16 r = scores();
    float sum = probs();
    __builtin_amdgcn_sched_barrier(0);
    if (__builtin_amdgcn_ballot_w64(!(sum <= limit)) != 0) {
      float mt = s[0] * sk[0][0];
#pragma unroll
      for (int v = 1; v < 16; ++v) mt = fmaxf(mt, s[v] * sk[v / 4][v % 4]);
      const float m_new = fmaxf(m_ref, max_across_halves(mt));
      const float alpha = __builtin_amdgcn_exp2f(m_ref - m_new);
      m_ref = m_new;
      nm = unit - m_new;
      l_run *= alpha;
#pragma unroll
      for (int db = 0; db < DB; ++db)
#pragma unroll
        for (int v = 0; v < 16; ++v) acc[db][v] *= alpha;
      sum = probs();
    }
    l_run += sum;
    __builtin_amdgcn_sched_barrier(0);
    if (AHEAD) request_keys(nnext);
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
      for (int hh = 0; hh < 2; ++hh) {
        if (db >= VA) vf[db][hh] = rd.cols(p, db, hh);
        acc[db] = mfma_h(vf[db][hh], pf[hh], acc[db]);
      }
    s = r;
    request_w(nbuf, nkr);
    __builtin_amdgcn_sched_barrier(0);
    mask(nkrem);
  };

  st.commit(smem, a.scale_dtype, a_s);
  if (nt > 1) {
    Stage &second = BOTH ? st1 : st;
    if (!BOTH) issue(second, 1);
    second.commit(smem + GM::BUF, a.scale_dtype, a_s);
  }
  if (EARLY && nt > 2) issue(st, 2);
  __syncthreads();
  const int kr0 = 32 * NB * kw;
  int left = a.Nk - t0 * TK - kr0;   // keys that exist from the wave's first row of the tile on
  if (active) {
    request_keys(smem + kr0 * 32);
    s = scores();
    request_w(smem, kr0);
    mask(left);
    if (AHEAD) request_keys(smem + (kr0 + 32) * 32);
  }
  int cur = 0;
  for (int t = 0; t < nt; ++t) {
    const int nxt = cur + 1 == 3 ? 0 : cur + 1, wr = nxt + 1 == 3 ? 0 : nxt + 1;
    const unsigned char *buf = smem + cur * GM::BUF, *nbuf = smem + nxt * GM::BUF;
    if (!EARLY && t + 2 < nt) issue(st, t + 2);
    if (active && NB == 2) body(buf, kr0, buf, kr0 + 32, left - 32, nbuf + kr0 * 32);
    if (EARLY && t + 2 < nt) {
      st.commit(smem + wr * GM::BUF, a.scale_dtype, a_s);
      if (t + 3 < nt) issue(st, t + 3);
    }
    if (active) body(buf, kr0 + 32 * (NB - 1), nbuf, kr0, left - TK, nbuf + (kr0 + 32) * 32);
    left -= TK;
    if (!EARLY && t + 2 < nt) st.commit(smem + wr * GM::BUF, a.scale_dtype, a_s);
    __syncthreads();
    cur = nxt;
  }

  float l = a_s * (l_run + swap32_f(l_run));
  float *mine = reinterpret_cast<float *>(smem) + slot * (GM::MERGE / 4) + lane;
  if (KW > 1) {
    if (kw > 0 && active) {
      float *dst = mine + (kw - 1) * QW * (GM::MERGE / 4);
#pragma unroll
      for (int db = 0; db < DB; ++db)
#pragma unroll
        for (int v = 0; v < 16; ++v) dst[(16 * db + v) * 64] = acc[db][v];
      dst[16 * DB * 64] = m_ref;
      dst[(16 * DB + 1) * 64] = l;
    }
    __syncthreads();
    if (kw > 0) return;
  }
  if (!active) return;
  if (KW > 1) {
    float m_all = m_ref;
#pragma unroll
    for (int w = 0; w < KW - 1; ++w) m_all = fmaxf(m_all, mine[w * QW * (GM::MERGE / 4) + 16 * DB * 64]);
    const float s0 = __builtin_amdgcn_exp2f(m_ref - m_all);
    l *= s0;
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[db][v] *= s0;
#pragma unroll
    for (int w = 0; w < KW - 1; ++w) {
      const float *src = mine + w * QW * (GM::MERGE / 4);
      const float sw = __builtin_amdgcn_exp2f(src[16 * DB * 64] - m_all);
      l += src[(16 * DB + 1) * 64] * sw;
#pragma unroll
      for (int db = 0; db < DB; ++db)
#pragma unroll
        for (int v = 0; v < 16; ++v) acc[db][v] += src[(16 * db + v) * 64] * sw;
    }
    m_ref = m_all;
  }
  if (a.splits > 1) {   // hand the unnormalised result to the merge kernel
    if (qi < a.Nq) {
      const int64_t at = (tq0 + qi) * a.splits + split;
#pragma unroll
      for (int db = 0; db < DB; ++db)
#pragma unroll
        for (int aa = 0; aa < 4; ++aa)
          *reinterpret_cast<f32x4 *>(a.po + at * D + 32 * db + 8 * aa + 4 * g) =
              f32x4{acc[db][4 * aa], acc[db][4 * aa + 1], acc[db][4 * aa + 2], acc[db][4 * aa + 3]};
      if (g == 0) *reinterpret_cast<f32x2 *>(a.pml + 2 * at) = f32x2{m_ref, l};
    }
    return;
  }
  if (g == 0 && qi < a.Nq) a.lse[tq0 + qi] = (m_ref + __log2f(l)) * kLn2;
  // (the wave's own part of the merge area, or of the tiles that nobody reads any more)
  unsigned char *stage = smem + (KW > 1 ? slot * GM::MERGE : wave * 64 * D);
  const float inv = 1.0f / l;
  unsigned short *o = static_cast<unsigned short *>(a.o) + b * a.sob + h * a.soh;
  if (a.io_bf16) store_tile_rows<__bf16, D>(acc, inv, stage, reinterpret_cast<__bf16 *>(o), a.son, 32 * qb, a.Nq, lane);
  else store_tile_rows<_Float16, D>(acc, inv, stage, reinterpret_cast<_Float16 *>(o), a.son, 32 * qb, a.Nq, lane);
}

template <int D, int QW> __global__ __launch_bounds__(256, D == 256 ? 1 : D == 128 ? 2 : 3) void skv_tile_dq_kernel(SkvTileArgs a) {
  typedef SkvTileGeom<D, QW> GM;
  constexpr int TK = GM::TK, NB = GM::NB, KW = GM::KW, DB = D / 32, KD = D / 16;
  __shared__ __attribute__((aligned(256))) unsigned char smem[2 * GM::BUF];

  const XcdBlock id(a.BH, a.qwgs * a.splits);
  if (!id.live) return;
  const int64_t b = index_div(id.bh, a.H), h = id.bh - b * a.H;
  const int tid = threadIdx.x, lane = tid % 64, lr = lane % 32, g = lane / 32;
  const int wave = __builtin_amdgcn_readfirstlane(tid / 64);
  const int split = id.sub / a.qwgs;
  const int slot = (wave + id.bh + id.sub) % QW, kw = wave / QW;
  const int qb = id.sub % a.qwgs * a.bpw + slot;
  const bool active = slot < a.bpw && 32 * qb < a.Nq;

  const unsigned char *codes_bh = reinterpret_cast<const unsigned char *>(a.codes + b * a.scb + h * a.sch);
  const int64_t tk0 = (int64_t)id.bh * a.Nk, tq0 = (int64_t)id.bh * a.Nq;
  const int t0 = split * a.tiles_per_split, nt = min(a.tiles_per_split, (a.Nk + TK - 1) / TK - t0);

  SkvTileStage<D, TK, GM::SLAB> st;
  st.init((unsigned)a.scn, tid);
  auto issue = [&](int t) __attribute__((always_inline)) {
    const int64_t k0 = (int64_t)(t0 + t) * TK;
    st.issue(codes_bh + k0 * a.scn, a.scale, a.scale_dtype == QFA_F32, a.zp, tk0 + k0, a.scn, a.Nk - (int)k0);
  };
  issue(0);

  const int qi = 32 * qb + lr, qi_c = min(qi, a.Nq - 1);
  u32x4 qf[KD], dof[KD];
  const KeyScaleMax scales(a.scale, a.scale_dtype, tk0 + (int64_t)t0 * TK, a.direct ? min(nt * TK, a.Nk - t0 * TK) : 1, tid);
  skv_load_row<D>(a.q, b * a.sqb + h * a.sqh + (int64_t)qi_c * a.sqn, a.io_bf16, g, qf);
  int dout_k = 0;   // direct: dO is scaled by 2^dout_k
  skv_load_row<D>(a.dout, b * a.sdob + h * a.sdoh + (int64_t)qi_c * a.sdon, 0, g, dof);
  const float lse = a.lse[tq0 + qi_c];
  float delta = 0.f;
  {
    u32x4 of[KD];
    skv_load_row<D>(a.o, b * a.sob + h * a.soh + (int64_t)qi_c * a.son, a.io_bf16, g, of);
    // A power of two of the workgroup's own queries, their delta and its keys.  The reduction in front of the first tile costs this
    // kernel a little (99 x 53 heads, 97 x 689, fp16, when it moved in: 442 -> 456 us), but it takes the place of two launches, more
    // in bf16: the call 1480 -> 1417 and 1519 -> 1426 us; 14 heads, 100 x 1872 (bound by launches): 84 -> 54 to 76.
    if (a.direct) {
      __shared__ float red[12];
      float md = 0.f;
      if (a.splits > 1) {   // O comes from all keys of the head, the scales from a part of them
        md = dot_dout(of, dof, a.do_bf16);
        md = finite_abs(a.sm_scale * (md + swap32_f(md)));
      }
      dout_k = block_dout_exponent(max_abs_dout(dof, a.do_bf16), scales.get(), md, red);
      scale_dout(dof, a.do_bf16, dout_k);
    }
#pragma unroll
    for (int m = 0; m < KD; ++m)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const unsigned ow = of[m][e], dw = dof[m][e];
        delta += lo_to_f32<_Float16>(ow) * lo_to_f32<_Float16>(dw) + hi_to_f32<_Float16>(ow) * hi_to_f32<_Float16>(dw);
      }
    delta += swap32_f(delta);
  }
  const float a_s = a.sm_scale_log2, sm = a.sm_scale;
  const float nlse2 = qi < a.Nq ? -lse * kLog2e : -INFINITY;   // padding rows: p = 0
  const SkvTileReads<GM::SLAB> rd(lane);

  f32x16 acc[DB];
#pragma unroll
  for (int db = 0; db < DB; ++db)
#pragma unroll
    for (int v = 0; v < 16; ++v) acc[db][v] = 0.f;

  // 32 keys from row kr of the tile in `buf`; krem: keys that exist from there on
  auto block = [&](const unsigned char *buf, int kr, int krem, auto masked_tag) __attribute__((always_inline)) {
    constexpr bool MASKED = decltype(masked_tag)::value;
    const unsigned char *p = buf + kr * 32;
    f32x16 s, dp;
#pragma unroll
    for (int v = 0; v < 16; ++v) s[v] = 0.f, dp[v] = 0.f;
#pragma unroll
    for (int m = 0; m < KD; ++m) {
      const u32x4 k = rd.rows(p, m);
      s = mfma_h(k, qf[m], s);
      dp = mfma_h(k, dof[m], dp);
    }
    u32x4 xf[2];
#pragma unroll
    for (int aa = 0; aa < 4; ++aa) {
      const f32x4 sk = *reinterpret_cast<const f32x4 *>(buf + GM::TILE + (kr + 8 * aa + 4 * g) * 4);
      float x[4];
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        float pr = __builtin_amdgcn_exp2f(__builtin_fmaf(a_s * sk[v], s[4 * aa + v], nlse2));
        if (MASKED && 8 * aa + 4 * g + v >= krem) pr = 0.f;
        x[v] = pr * __builtin_fmaf(sk[v], dp[4 * aa + v], -delta) * (sm * sk[v]);
      }
      xf[aa / 2][2 * (aa % 2)] = pack_h2(x[0], x[1]);
      xf[aa / 2][2 * (aa % 2) + 1] = pack_h2(x[2], x[3]);
    }
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
      for (int hh = 0; hh < 2; ++hh) acc[db] = mfma_h(rd.cols(p, db, hh), xf[hh], acc[db]);
  };

  st.commit(smem, a.scale_dtype, 1.0f);
  wait_loads();
  __syncthreads();
  for (int t = 0; t < nt; ++t) {
    unsigned char *buf = smem + (t & 1) * GM::BUF;
    if (t + 1 < nt) issue(t + 1);
    if (active) {
      const int left = a.Nk - (t0 + t) * TK - 32 * NB * kw;
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) {
        if (left >= 32 * (nb + 1)) block(buf, 32 * (NB * kw + nb), 32, std::false_type{});
        else if (left > 32 * nb) block(buf, 32 * (NB * kw + nb), left - 32 * nb, std::true_type{});
      }
    }
    if (t + 1 < nt) st.commit(smem + ((t + 1) & 1) * GM::BUF, a.scale_dtype, 1.0f);
    __syncthreads();
  }

  float *mine = reinterpret_cast<float *>(smem) + slot * (GM::MERGE / 4) + lane;
  if (KW > 1) {
    if (kw > 0 && active) {
      float *dst = mine + (kw - 1) * QW * (GM::MERGE / 4);
#pragma unroll
      for (int db = 0; db < DB; ++db)
#pragma unroll
        for (int v = 0; v < 16; ++v) dst[(16 * db + v) * 64] = acc[db][v];
    }
    __syncthreads();
    if (kw > 0) return;
  }
  if (!active) return;
#pragma unroll
  for (int w = 0; w < KW - 1; ++w) {
    const float *src = mine + w * QW * (GM::MERGE / 4);
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[db][v] += src[(16 * db + v) * 64];
  }
  if (a.splits > 1) {   // partial result for the sum
    const float part = exp2_neg(dout_k);   // (the sum applies grad_scale)
    if (qi < a.Nq) {
      const int64_t at = (tq0 + qi) * a.splits + split;
#pragma unroll
      for (int db = 0; db < DB; ++db)
#pragma unroll
        for (int aa = 0; aa < 4; ++aa)
          *reinterpret_cast<f32x4 *>(a.po + at * D + 32 * db + 8 * aa + 4 * g) =
              f32x4{acc[db][4 * aa] * part, acc[db][4 * aa + 1] * part, acc[db][4 * aa + 2] * part, acc[db][4 * aa + 3] * part};
    }
    return;
  }
  const float osc = a.grad_scale ? *a.grad_scale : exp2_neg(dout_k);
  unsigned char *stage = smem + (KW > 1 ? slot * GM::MERGE : wave * 64 * D);
  unsigned short *dq = static_cast<unsigned short *>(a.dq) + b * a.sdqb + h * a.sdqh;
  if (a.grad_bf16) store_tile_rows<__bf16, D>(acc, osc, stage, reinterpret_cast<__bf16 *>(dq), a.sdqn, 32 * qb, a.Nq, lane);
  else store_tile_rows<_Float16, D>(acc, osc, stage, reinterpret_cast<_Float16 *>(dq), a.sdqn, 32 * qb, a.Nq, lane);
}

// ---------------------------------------------------------------------------------------------- launch
static SkvTileArgs skv_tile_args(const SkvAttnArgs &x, int qw) {
  SkvTileArgs a;
  a.q = x.q; a.codes = x.codes; a.scale = x.scale; a.zp = x.zp; a.o = x.o; a.lse = x.lse;
  a.dout = static_cast<const _Float16 *>(x.dout); a.dq = x.dq; a.grad_scale = x.grad_scale;
  a.direct = x.direct; a.do_bf16 = x.dout_dtype == QFA_BF16;
  a.H = x.H; a.Nq = (int)x.Nq; a.Nk = (int)x.Nk; a.BH = (int)(x.B * x.H);
  a.io_bf16 = x.io_dtype == QFA_BF16; a.scale_dtype = x.scale_dtype; a.grad_bf16 = x.grad_dtype == QFA_BF16;
  a.sqb = x.sqb; a.sqh = x.sqh; a.sqn = x.sqn; a.scb = x.scb; a.sch = x.sch; a.scn = x.scn;
  a.sob = x.sob; a.soh = x.soh; a.son = x.son; a.sdob = x.sdob; a.sdoh = x.sdoh; a.sdon = x.sdon;
  a.sdqb = x.sdqb; a.sdqh = x.sdqh; a.sdqn = x.sdqn;
  a.sm_scale = x.sm_scale;
  a.sm_scale_log2 = x.sm_scale * kLog2e;
  const int nb = (int)((x.Nq + 31) / 32);
  a.qwgs = (nb + qw - 1) / qw;
  a.bpw = (nb + a.qwgs - 1) / a.qwgs;   // 5 blocks: 3 + 2, not 4 + 1
  a.splits = 1;
  a.tiles_per_split = 0x7fffffff;
  a.po = a.pml = nullptr;
  return a;
}
template <int D> static int launch_fwd_d(const SkvAttnArgs &x, const SkvTilePlan &p, hipStream_t st) {
  SkvTileArgs a = skv_tile_args(x, p.qw);
  a.sm_scale_log2 = a.sm_scale_log2 < 0x1p-60f ? 0x1p-60f : a.sm_scale_log2;   // (key scales are multiplied by it)
  if (p.splits > 1) {   // (the caller has seen to the workspace)
    a.splits = p.splits;
    a.tiles_per_split = p.tiles;
    a.po = static_cast<float *>(x.workspace);
    a.pml = a.po + x.B * x.H * x.Nq * a.splits * (int64_t)D;
  }
  const int64_t total = xcd_grid(a.BH, (int64_t)a.qwgs * a.splits), rows = x.B * x.H * x.Nq;
  if (x.B * x.H > 0x7fffffffLL || total > 0x7fffffffLL || (a.splits > 1 && rows > 0x7fffffffLL))
    return set_error(QFA_EUNSUPPORTED, "attn_fwd_shared_kv: too many query blocks for one launch");
  if (p.qw == 4) skv_tile_fwd_kernel<D, 4><<<dim3((unsigned)total), dim3(256), 0, st>>>(a);
  else skv_tile_fwd_kernel<D, 2><<<dim3((unsigned)total), dim3(256), 0, st>>>(a);
  if (int e = check_launch("qfa_attn_fwd_shared_kv")) return e;
  if (a.splits > 1) {
    const SplitMergeArgs m = {a.po, a.pml, a.o, a.lse, a.H, a.sob, a.soh, a.son, a.Nq, a.splits, x.io_dtype, nullptr};
    return launch_split_merge<D>(m, rows, "qfa_attn_fwd_shared_kv (merge)", st);
  }
  return 0;
}
template <int D> static int launch_dq_d(const SkvAttnArgs &x, const SkvTilePlan &p, hipStream_t st) {
  SkvTileArgs a = skv_tile_args(x, p.qw);
  if (p.splits > 1) {   // (the caller has seen to the workspace)
    a.splits = p.splits;
    a.tiles_per_split = p.tiles;
    a.po = static_cast<float *>(x.workspace);
  }
  const int64_t total = xcd_grid(a.BH, (int64_t)a.qwgs * a.splits);
  if (total > 0x7fffffffLL) return set_error(QFA_EUNSUPPORTED, "attn_bwd_shared_kv: too many query blocks for one launch");
  if (p.qw == 4) skv_tile_dq_kernel<D, 4><<<dim3((unsigned)total), dim3(256), 0, st>>>(a);
  else skv_tile_dq_kernel<D, 2><<<dim3((unsigned)total), dim3(256), 0, st>>>(a);
  if (int e = check_launch("qfa_attn_bwd_shared_kv (dQ)")) return e;
  return a.splits > 1 ? launch_split_sum(x, a.splits, st) : 0;
}
int launch_skv_tile_fwd(const SkvAttnArgs &x, const SkvTilePlan &p, hipStream_t st) {
  return x.D == 256 ? launch_fwd_d<256>(x, p, st) : x.D == 128 ? launch_fwd_d<128>(x, p, st) : launch_fwd_d<64>(x, p, st);
}
int launch_skv_tile_dq(const SkvAttnArgs &x, const SkvTilePlan &p, hipStream_t st) {
  return x.D == 256 ? launch_dq_d<256>(x, p, st) : x.D == 128 ? launch_dq_d<128>(x, p, st) : launch_dq_d<64>(x, p, st);
}

}  // namespace qfa
