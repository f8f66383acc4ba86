// Backward of the shared-KV attention in one pass at head_dim 64, for query blocks of 33 to 128; the counterpart of qfa_skv_pass.hip,
// where the arithmetic and the way of P and dS through LDS are described.
//
// At this width a wave's operands -- Q and dO rows, 32 columns of dO^T and Q^T for all queries -- and its accumulators fit 256
// registers and a workgroup 52 KB of LDS, so two workgroups run on a CU and fill each other's waits: scheduled by the compiler, one
// buffer of P and dS, two barriers a tile.  (Written out with one wave per SIMD, as at 128, it took 590 us for 5247 heads, 97 x 689,
// this one 440, the two kernels it stands for 580; where it is taken: skv_pass_takes.
// Exponentials and vector work take longer than the products here, and one wave issues an instruction every 4 cycles.)
#include "qfa_host.h"
#include "qfa_skv_tile.h"

namespace qfa {

// QW waves side by side on the queries, KW on the keys of a tile
template <int QW> struct SkvPass64Geom {
  static constexpr int D = 64, KW = 4 / QW, ROWS = 32 * QW, TK = 64, CPR = D / 16;      // queries, keys per tile, slabs of 16 columns
  static constexpr int SLAB = TK * 32 + 128, TILE = CPR * SLAB, BUF = TILE + TK * 4;   // expanded tile, key scales
  static constexpr int PSLAB = ROWS * 32 + 128, PMAT = TK / 16 * PSLAB;                 // P, dS: slabs of 16 keys
  static constexpr int OFF_P = 2 * BUF, TOTAL = OFF_P + 2 * PMAT;
  static constexpr int MERGE = D / 2 * 256;   // a wave's dQ^T
  static_assert(CPR * PSLAB <= PMAT, "the rows of dO and Q pass through the buffers of P and dS");
  static_assert((KW - 1) * QW * MERGE <= TOTAL && 4 * 64 * D <= TOTAL, "dQ leaves through LDS");
};

// G: type of the gradients
template <typename G, int QW> __global__ __launch_bounds__(256, 2) void skv_pass64_kernel(SkvPassArgs a) {
  typedef SkvPass64Geom<QW> GM;
  constexpr int D = GM::D, TK = GM::TK, KW = GM::KW, DB = D / 32, KD = D / 16, KQ = 2 * QW, PSLAB = GM::PSLAB;
  __shared__ __attribute__((aligned(256))) unsigned char smem[GM::TOTAL];

  const XcdBlock id(a.BH, 1);
  if (!id.live) return;
  const int64_t b = index_div(id.bh, a.H), h = id.bh - b * a.H;
  const int tid = threadIdx.x, lane = tid % 64, lr = lane % 32, g = lane / 32;
  const int wave = __builtin_amdgcn_readfirstlane(tid / 64);
  // S, dP, dQ: block of queries, of keys (KW == 1: both); turned by the head, waves without queries should not share a SIMD
  const int qb = (wave + (KW == 1 ? id.bh : 0)) % QW, kw = wave / QW;
  const int wd = wave % 2, wk = wave / 2;     // dKV: block of 32 columns, of 32 keys
  const bool active = 32 * qb < a.Nq;

  const unsigned char *codes_bh = reinterpret_cast<const unsigned char *>(a.codes + b * a.scb + h * a.sch);
  const int64_t tk0 = (int64_t)id.bh * a.Nk, tq0 = (int64_t)id.bh * a.Nq;
  const int nt = (a.Nk + TK - 1) / TK;

  SkvTileStage<D, TK, GM::SLAB> st;
  st.init((unsigned)a.scn, tid);
  auto issue = [&](int t) __attribute__((always_inline)) {
    const int64_t k0 = (int64_t)t * TK;
    st.issue(codes_bh + k0 * a.scn, a.scale, a.scale_dtype == QFA_F32, a.zp, tk0 + k0, a.scn, a.Nk - (int)k0);
  };
  issue(0);
  const SkvTileReads<GM::SLAB> rd(lane);
  // P and dS: this lane's query as a row (the 8-byte pieces of rows 16-31 of a block are swapped: 32 lanes that write 8 bytes each
  // hit all banks once); transposing reads of the wave's keys
  const int p_row = (32 * qb + lr) * 32 + ((lr >> 3 & 1) << 4) + 8 * (g ^ (lr >> 4));
  const int p_tr = skv_tile_off<PSLAB>(4 * g + lane % 16 / 4, lane / 16 % 2 + 2 * wk, lane % 4 / 2) + lane % 2 * 8;

  u32x4 qf[KD], dof[KD];
  float nlse2, nd, osc;
  {
    const int qi = 32 * qb + lr, qi_c = min(qi, a.Nq - 1);
    const KeyScaleMax scales(a.scale, a.scale_dtype, tk0, a.direct ? a.Nk : 1, tid);
    u32x4 of[KD];
    skv_load_row<D>(a.dout, b * a.sdob + h * a.sdoh + (int64_t)qi_c * a.sdon, 0, g, dof);
    skv_load_row<D>(a.o, b * a.sob + h * a.soh + (int64_t)qi_c * a.son, a.io_bf16, g, of);
    skv_load_row<D>(a.q, b * a.sqb + h * a.sqh + (int64_t)qi_c * a.sqn, a.io_bf16, g, qf);
    const float lse = a.lse[tq0 + qi_c];
    if (qi >= a.Nq) {   // rows past the end: zeros, which add nothing to dKV whatever the last row holds
#pragma unroll
      for (int m = 0; m < KD; ++m) qf[m] = dof[m] = of[m] = u32x4{0u, 0u, 0u, 0u};
    }
    int dout_k = 0;   // direct: dO is scaled by 2^dout_k
    if (a.direct) {
      dout_k = block_dout_exponent(max_abs_dout(dof, a.do_bf16), scales.get(), 0.f, reinterpret_cast<float *>(smem));
      scale_dout(dof, a.do_bf16, dout_k);
      __syncthreads();   // (the maxima are where the tiles go)
    }
    osc = a.grad_scale ? *a.grad_scale : exp2_neg(dout_k);
    float delta = dot_dout(of, dof, 0);
    delta += swap32_f(delta);
    nlse2 = qi < a.Nq ? -lse * kLog2e : -INFINITY;   // p = 0
    nd = -a.sm_scale * delta;
    if (kw == 0) {
#pragma unroll
      for (int m = 0; m < KD; ++m) {
        unsigned char *row = smem + GM::OFF_P + skv_tile_off<PSLAB>(32 * qb + lr, m, g);
        *reinterpret_cast<u32x4 *>(row) = dof[m];
        *reinterpret_cast<u32x4 *>(row + GM::PMAT) = qf[m];
      }
    }
    st.commit(smem, a.scale_dtype, 1.0f);
  }
  wait_loads();
  if (nt > 1) issue(1);
  __syncthreads();
  // A operands of dKV: columns 32wd + lr of dO and Q
  u32x4 dot[KQ], qt[KQ];
  {
    const SkvTileReads<PSLAB> rp(lane);
    const int o = rp.tr[0] ^ wd << 4;
    auto cols = [&](const unsigned char *c) -> u32x4 {
      const u32x2 x = lds_read_tr16(c + o), y = lds_read_tr16(c + 256 + (o ^ 16));
      return u32x4{x[0], x[1], y[0], y[1]};
    };
#pragma unroll
    for (int j = 0; j < KQ; ++j) {
      const unsigned char *p = smem + GM::OFF_P + 2 * wd * PSLAB + j * 512;
      dot[j] = cols(p);
      qt[j] = cols(p + GM::PMAT);
    }
  }
  __syncthreads();
  if (!active) {   // P and dS of queries that do not exist stay zero
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int c = 0; c < 4; ++c)
        if (KW == 1 || c / 2 == kw) *reinterpret_cast<u32x4 *>(smem + GM::OFF_P + i * GM::PMAT + c * PSLAB + (32 * qb + lr) * 32 + 16 * g) = u32x4{0u, 0u, 0u, 0u};
  }

  f32x16 acc[DB];
#pragma unroll
  for (int db = 0; db < DB; ++db)
#pragma unroll
    for (int v = 0; v < 16; ++v) acc[db][v] = 0.f;
  const float a_s = a.sm_scale_log2, sm = a.sm_scale;

  // P and dS of block kb (32 keys) of the tile in `buf`, and their dQ.  krem: keys that exist from the block's first on
  auto block = [&](const unsigned char *buf, int kb, int krem, auto masked_tag) __attribute__((always_inline)) {
    constexpr bool MASKED = decltype(masked_tag)::value;
    const unsigned char *p = buf + kb * 1024;
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
    unsigned char *pw = smem + GM::OFF_P + 2 * kb * PSLAB;
    const int pr = p_row ^ kb << 4;
#pragma unroll
    for (int aa = 0; aa < 4; ++aa) {
      const f32x4 sk = *reinterpret_cast<const f32x4 *>(buf + GM::TILE + (32 * kb + 8 * aa + 4 * g) * 4);
      float pv[4], ds[4], x[4];
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        pv[v] = __builtin_amdgcn_exp2f(__builtin_fmaf(a_s * sk[v], s[4 * aa + v], nlse2));
        ds[v] = pv[v] * __builtin_fmaf(sm * sk[v], dp[4 * aa + v], nd);
        x[v] = ds[v] * sk[v];
        if (MASKED && 8 * aa + 4 * g + v >= krem) x[v] = 0.f;   // (keys past the end: their rows of dKV are not stored)
      }
      unsigned char *w = pw + aa / 2 * PSLAB + (pr ^ aa % 2 << 4);
      *reinterpret_cast<u32x2 *>(w) = u32x2{pack_h2(pv[0], pv[1]), pack_h2(pv[2], pv[3])};
      *reinterpret_cast<u32x2 *>(w + GM::PMAT) = u32x2{pack_h2(ds[0], ds[1]), pack_h2(ds[2], ds[3])};
      xf[aa / 2][2 * (aa % 2)] = pack_h2(x[0], x[1]);
      xf[aa / 2][2 * (aa % 2) + 1] = pack_h2(x[2], x[3]);
    }
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
      for (int hh = 0; hh < 2; ++hh) acc[db] = mfma_h(rd.cols(p, db, hh), xf[hh], acc[db]);
  };

  unsigned short *dkv_bh = static_cast<unsigned short *>(a.dkv) + b * a.sdkb + h * a.sdkh + 32 * wd;
  const int out_l = lr * (int)a.sdkn * 2 + 16 * g;
  for (int t = 0; t < nt; ++t) {
    const unsigned char *buf = smem + (t & 1) * GM::BUF;
    const int left = a.Nk - t * TK;
    if (active) {
#pragma unroll
      for (int i = 0; i < 2 / KW; ++i) {
        const int kb = KW == 2 ? kw : i;
        if (left >= TK) block(buf, kb, 32, std::false_type{});
        else if (left > 32 * kb) block(buf, kb, left - 32 * kb, std::true_type{});
      }
    }
    if (t + 1 < nt) {
      st.commit(smem + (~t & 1) * GM::BUF, a.scale_dtype, 1.0f);
      if (t + 2 < nt) issue(t + 2);
    }
    lds_barrier();   // P and dS are there, and the next tile
    if (left > 32 * wk) {
      f32x16 c;
#pragma unroll
      for (int v = 0; v < 16; ++v) c[v] = 0.f;
#pragma unroll
      for (int j = 0; j < KQ; ++j) {
        const int o = p_tr ^ (j & 1) * 8;
        auto frag = [&](const unsigned char *p) -> u32x4 {
          const u32x2 x = lds_read_tr16(p + o), y = lds_read_tr16(p + 256 + (o ^ 16));
          return u32x4{x[0], x[1], y[0], y[1]};
        };
        c = mfma_h(dot[j], frag(smem + GM::OFF_P + j * 512), c);
        c = mfma_h(qt[j], frag(smem + GM::OFF_P + GM::PMAT + j * 512), c);
      }
      // 16 bytes of a row per lane: the halves of the wave exchange quads of columns
      const int rows = min(32, left - 32 * wk);
      const rsrc_t rs = make_rsrc(dkv_bh + (int64_t)(t * TK + 32 * wk) * a.sdkn, (unsigned)((rows - 1) * (int)a.sdkn * 2 + 64));
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        unsigned w[4];
#pragma unroll
        for (int x = 0; x < 4; ++x) w[x] = pack2<G>(c[8 * i + 2 * x] * osc, c[8 * i + 2 * x + 1] * osc);
        swap_halves(w[0], w[2]);
        swap_halves(w[1], w[3]);
        __builtin_amdgcn_raw_buffer_store_b128(u32x4{w[0], w[1], w[2], w[3]}, rs, out_l + 32 * i, 0, 0);
      }
    }
    lds_barrier();   // P and dS have been read
  }
  if (KW > 1) {
    float *mine = reinterpret_cast<float *>(smem) + qb * (GM::MERGE / 4) + lane;
    if (kw > 0 && active) {
#pragma unroll
      for (int db = 0; db < DB; ++db)
#pragma unroll
        for (int v = 0; v < 16; ++v) mine[(16 * db + v) * 64] = acc[db][v];
    }
    __syncthreads();
    if (kw > 0 || !active) return;
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[db][v] += mine[(16 * db + v) * 64];
  }
  if (!active) return;
  G *dq = static_cast<G *>(a.dq) + b * a.sdqb + h * a.sdqh;
  store_tile_rows<G, D>(acc, osc, smem + qb * (KW > 1 ? GM::MERGE : 64 * D), dq, a.sdqn, 32 * qb, a.Nq, lane);
}

template <int QW> static void launch_qw(const SkvPassArgs &a, unsigned grid, bool grad_bf16, hipStream_t st) {
  if (grad_bf16) skv_pass64_kernel<__bf16, QW><<<dim3(grid), dim3(256), 0, st>>>(a);
  else skv_pass64_kernel<_Float16, QW><<<dim3(grid), dim3(256), 0, st>>>(a);
}

int launch_skv_pass(const SkvAttnArgs &x, hipStream_t st) {
  SkvPassArgs a;
  a.q = x.q; a.codes = x.codes; a.scale = x.scale; a.zp = x.zp; a.o = x.o; a.lse = x.lse; a.dout = x.dout;
  a.dq = x.dq; a.dkv = x.dkv; a.grad_scale = x.grad_scale;
  a.H = x.H; a.Nq = (int)x.Nq; a.Nk = (int)x.Nk; a.BH = (int)(x.B * x.H);
  a.io_bf16 = x.io_dtype == QFA_BF16; a.scale_dtype = x.scale_dtype;
  a.direct = x.direct; a.do_bf16 = x.dout_dtype == QFA_BF16;
  a.sqb = x.sqb; a.sqh = x.sqh; a.sqn = x.sqn; a.scb = x.scb; a.sch = x.sch; a.scn = x.scn;
  a.sob = x.sob; a.soh = x.soh; a.son = x.son; a.sdob = x.sdob; a.sdoh = x.sdoh; a.sdon = x.sdon;
  a.sdqb = x.sdqb; a.sdqh = x.sdqh; a.sdqn = x.sdqn; a.sdkb = x.sdkb; a.sdkh = x.sdkh; a.sdkn = x.sdkn;
  a.sm_scale = x.sm_scale;
  a.sm_scale_log2 = x.sm_scale * kLog2e;
  const unsigned grid = (unsigned)xcd_grid(x.B * x.H, 1);
  const bool bf16 = x.grad_dtype == QFA_BF16;
  if (x.D == 128) return launch_skv_pass128(a, grid, bf16, st);
  if (a.Nq > 64) launch_qw<4>(a, grid, bf16, st);
  else launch_qw<2>(a, grid, bf16, st);
  return check_launch("qfa_attn_bwd_shared_kv (one pass)");
}

}  // namespace qfa
