// Backward of the shared-KV attention in one pass at head_dim 128, for query blocks of 33 to 128:
//     P = exp(sm_scale * Q KV^T - LSE),  dS = sm_scale * P o (dO KV^T - delta),  dQ = dS KV,  dKV = P^T dO + dS^T Q
// (quant_flash_attn.py:104-166).
//
// A workgroup takes a (batch, head) and expands a tile of 64 keys at a time into LDS (qfa_skv_tile.h).  A wave has 32 queries, whose
// Q and dO rows are B operands in registers and whose dQ^T accumulators are AccVGPRs: four waves side by side take both blocks of 32
// keys of a tile (up to 128 queries), two side by side one block each (up to 64).  S^T and dP^T leave P and dS in the lanes as the B
// operand of dQ^T += KV^T.(dS scale).  dKV is contracted over the queries of all waves: P and dS go through LDS as binary16
// [query][key] tiles and come back transposed, with dO^T and Q^T -- 64 columns per wave, for 32 keys -- as A operands that stay in
// AccVGPRs for the whole kernel.  So a code is expanded once, and S, dP and the exponentials are formed once, where the two kernels
// (skv_tile_dq_kernel, skv_dkv_kernel) do all of it twice: 5 products per pair of query and key instead of 7.
//
// One wave per SIMD, written out as in qfa_bwd_dq.inc.  A step (32 keys per wave) is one straight line of MFMAs in the order
//     dQ of the previous step and, in turn, S and dP of the next one  |  dKV of the previous tile
// and the vector work of this step's P and dS, the expansion of the tile after the next and the way of the finished dKV rows to
// memory are dealt to them, so that no product waits for the vector work it depends on.  One barrier per tile: four or five buffers
// of keys, two of P and dS.
//
// What bounds it: the instructions one wave can issue.  A lone wave takes 4 cycles for any instruction, scalar ones and waits too,
// 12 for an LDS read whatever its width, 13 for an MFMA: the 680 of a tile (four waves side by side) come to the 4870 cycles that it
// takes, its products to 2560; without the vector work the loop runs at the products' pace, so LDS bandwidth is not it.  A workgroup's
// start is 16000 cycles (8700 of them until its rows are there), its end 4600.  Measured against the two kernels (us, one GPU): 5247
// heads, 97 x 689: 1100 -> 785; 64 x 689: 800 -> 580; 256 heads, 128 x 4096: 310 -> 188; 512 heads, 40 x 3000: 275 -> 192.
// Tried and not kept: fragments requested seven ahead instead of three; eight waves (two per SIMD, 32 keys each, scheduled by the
// compiler, 255 registers, Q from LDS): 922 us; the next workgroup's rows requested into the L2 by this one: no change.
#include <type_traits>

#include "qfa_acc.h"
#include "qfa_skv_tile.h"

namespace qfa {

template <int QW> struct SkvPassGeom {
  static constexpr int D = 128, KW = 4 / QW, NB = 2 / KW;   // QW waves side by side on the queries, KW on the keys; blocks per wave
  static constexpr int ROWS = 32 * QW, TK = 64, CPR = D / 16;                         // queries, keys of a tile, slabs of 16 columns
  static constexpr int SLAB = TK * 32 + 128, TILE = CPR * SLAB, BUF = TILE + 3 * TK * 4;   // expanded tile, factors of the keys
  static constexpr int PSLAB = ROWS * 32 + 128, PMAT = TK / 16 * PSLAB, PBUF = 2 * PMAT;   // P, dS: slabs of 16 keys
  // tiles in LDS: the previous step's, this one's, those whose rows the next step and (where a step is a tile) the first requests of
  // the one behind it read, the one that is written
  static constexpr int NBUF = NB == 2 ? 4 : 5;
  static constexpr int OFF_P = NBUF * BUF, TOTAL = OFF_P + 2 * PBUF;
  static constexpr int MERGE = D / 2 * 256;   // a wave's dQ^T
  static_assert(CPR * PSLAB <= PBUF, "Q and dO rows pass through the buffers of P and dS");
  static_assert(TOTAL <= 160 * 1024 && 4 * 64 * D <= OFF_P && (KW - 1) * QW * MERGE <= OFF_P, "LDS of a CU; dQ leaves through the tiles");
};

// dout_exponent of 256 threads' m and ms (block_dout_exponent without shuffles: rows of 16 lanes by DPP, the rest from LDS); red: 32
// floats of LDS that nobody uses
__device__ __forceinline__ int skv_pass_exponent(float m, float ms, float *red) {
  const auto row_max = [](float x) __attribute__((always_inline)) {
    x = fmaxf(x, dpp_f<0xB1>(x));
    x = fmaxf(x, dpp_f<0x4E>(x));
    x = fmaxf(x, dpp_f<0x141>(x));
    return fmaxf(x, dpp_f<0x140>(x));
  };
  m = row_max(m);
  ms = row_max(ms);
  if (threadIdx.x % 16 == 0) {
    red[threadIdx.x / 16] = m;
    red[16 + threadIdx.x / 16] = ms;
  }
  __syncthreads();
  m = ms = 0.f;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const f32x4 x = *reinterpret_cast<const f32x4 *>(red + 4 * i), y = *reinterpret_cast<const f32x4 *>(red + 16 + 4 * i);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      m = fmaxf(m, x[e]);
      ms = fmaxf(ms, y[e]);
    }
  }
  return __builtin_amdgcn_readfirstlane(dout_exponent(m, ms));
}

// S: type of the key scales, G: of the gradients
template <typename S, typename G, int QW> __global__ __launch_bounds__(256, 1) void skv_pass_kernel(SkvPassArgs a) {
#ifdef __HIP_DEVICE_COMPILE__   // (with the body in view the host pass of this compiler emits no launch stub)
  typedef SkvPassGeom<QW> GM;
  constexpr int D = GM::D, TK = GM::TK, KW = GM::KW, NB = GM::NB, DB = D / 32, KD = D / 16, RT = 2, KQ = 2 * QW, PSLAB = GM::PSLAB;
  __shared__ __attribute__((aligned(256))) unsigned char smem[GM::TOTAL];

  const XcdBlock id(a.BH, 1);
  if (!id.live) return;
  const int64_t b = index_div(id.bh, a.H), h = id.bh - b * a.H;
  const int tid = threadIdx.x, lane = tid % 64, lr = lane % 32, g = lane / 32;
  const int wave = __builtin_amdgcn_readfirstlane(tid / 64);
  const int qb = wave % QW, kw = wave / QW;   // block of queries; of keys, with two waves side by side
  const int wd = wave % 2, wk = wave / 2;     // of dKV: half of the columns, block of 32 keys of a tile
  const int64_t tk0 = (int64_t)id.bh * a.Nk, tq0 = (int64_t)id.bh * a.Nq;
  const int nt = (a.Nk + TK - 1) / TK;

  // ---- a thread's share of a tile on its way: two chunks of 16 codes, their rows' zero points, a key scale.  Descriptors of the
  // whole head: what lies past its end arrives as zeros, and the offsets just go on
  typedef SkvTileStage<D, TK, GM::SLAB> Stage;
  static_assert(Stage::N == 2, "chunks per thread");
  Stage st;
  st.init((unsigned)a.scn, tid);
  const rsrc_t rk = make_rsrc(a.codes + b * a.scb + h * a.sch, (unsigned)((a.Nk - 1) * (int)a.scn + D));
  const rsrc_t rz = make_rsrc(a.zp + tk0, (unsigned)a.Nk), rs = make_rsrc(static_cast<const S *>(a.scale) + tk0, (unsigned)(a.Nk * (int)sizeof(S)));
  unsigned s_at = lane * sizeof(S);
  auto issue = [&](Stage &x) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      x.w[i] = __builtin_amdgcn_raw_buffer_load_b128(rk, (int)(st.off + (unsigned)i * st.row_step), 0, 0);
      x.z[i] = (unsigned char)__builtin_amdgcn_raw_buffer_load_b8(rz, st.row + Stage::STEP * i, 0, 0);
    }
    if constexpr (sizeof(S) == 4) x.s = __builtin_amdgcn_raw_buffer_load_b32(rs, (int)s_at, 0, 0);
    else x.s = (unsigned short)__builtin_amdgcn_raw_buffer_load_b16(rs, (int)s_at, 0, 0);
    st.off += TK * (unsigned)a.scn;
    st.row += TK;
    s_at += TK * sizeof(S);
  };
  // what the scores, dP and dS of a key are multiplied by: a table each, written by a wave each
  const float a_s = a.sm_scale_log2, sm = a.sm_scale, factor = wave == 0 ? 1.0f : wave == 1 ? a_s : sm;
  auto commit_scale = [&](const Stage &x, unsigned char *buf) __attribute__((always_inline)) {
    if (wave < 3) *reinterpret_cast<float *>(buf + GM::TILE + tid * 4) = scale_to_f32<S>(x.s) * factor;
  };
  const SkvTileReads<GM::SLAB> rd(lane);
  // per-lane offsets in a buffer of P and dS: this lane's query as a row (the 8-byte pieces of rows 16-31 of a block are swapped: 32
  // lanes that write 8 bytes each hit all banks once); transposing reads of the wave's keys
  const int p_row = ((32 * qb + lr) * 32 + ((lr >> 3 & 1) << 4) + 8 * (g ^ (lr >> 4))) ^ (NB == 1 ? kw << 4 : 0);
  const int s16 = lane % 16, p_tr = skv_tile_off<PSLAB>(4 * g + s16 / 4, lane / 16 % 2 + 2 * wk, s16 % 4 / 2) + s16 % 2 * 8;

  u32x4 qf[KD], dof[KD];
  float nlse2, nd, osc;
  {
    Stage first[GM::NBUF - 2];
    static_for<GM::NBUF - 2>([&](auto i) __attribute__((always_inline)) {
      first[decltype(i)::value] = st;
      issue(first[decltype(i)::value]);
    });
    // Rows of dO, O and Q as they lie in memory, whole rows of 256 bytes (as B operands straight from memory, 32 bytes of each of 32
    // rows at a time, they kept the address unit busy for 4 us); the 16-byte piece c of row r is at c ^ r % 16.  Rows past the end
    // arrive as zeros, which add nothing to dKV whatever the last row holds
    constexpr int RW = GM::ROWS / 4, OFF_O = (GM::NBUF - 2) * GM::BUF;   // rows that a wave copies
    auto copy_rows = [&](const void *p, int64_t stride, int dst) __attribute__((always_inline)) {
      const rsrc_t r = make_rsrc(p, (unsigned)((a.Nq - 1) * (int)stride * 2 + 2 * D));
#pragma unroll
      for (int i = 0; i < RW / 4; ++i) {
        const int row = RW * wave + 4 * i + lane / 16;
        __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (lptr_t)(smem + dst + (RW * wave + 4 * i) * 2 * D), 16,
                                                 row * (int)stride * 2 + ((lane % 16 ^ row % 16) << 4), 0, 0, 0);
      }
    };
    copy_rows(static_cast<const unsigned short *>(a.dout) + b * a.sdob + h * a.sdoh, a.sdon, GM::OFF_P + GM::PBUF);
    copy_rows(static_cast<const unsigned short *>(a.o) + b * a.sob + h * a.soh, a.son, OFF_O);
    copy_rows(static_cast<const unsigned short *>(a.q) + b * a.sqb + h * a.sqh, a.sqn, GM::OFF_P);
    const int qi = 32 * qb + lr;
    const float lse = a.lse[tq0 + min(qi, a.Nq - 1)];
    float ms = 0.f;
    if (a.direct) {   // the largest of the head's key scales
      const S *sc = static_cast<const S *>(a.scale) + tk0;
      for (int j0 = 0; j0 < a.Nk; j0 += 4 * 256) {
        S x[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) x[i] = sc[min(j0 + 256 * i + tid, a.Nk - 1)];
#pragma unroll
        for (int i = 0; i < 4; ++i) ms = fmaxf(ms, fabsf((float)x[i]));
      }
    }
    dma_wait();
    if (QW == 2) __syncthreads();   // (with four waves side by side each copied its own queries)
    u32x4 of[KD];
    auto rows = [&](int at, u32x4 (&f)[KD]) __attribute__((always_inline)) {
#pragma unroll
      for (int m = 0; m < KD; ++m) f[m] = *reinterpret_cast<const u32x4 *>(smem + at + (32 * qb + lr) * 2 * D + (((2 * m + g) ^ lr % 16) << 4));
    };
    rows(GM::OFF_P + GM::PBUF, dof);
    rows(OFF_O, of);
    rows(GM::OFF_P, qf);
    if (a.io_bf16) {
#pragma unroll
      for (int m = 0; m < KD; ++m) {
        of[m] = half_of_bf16(of[m]);
        qf[m] = half_of_bf16(qf[m]);
      }
    }
    int dout_k = 0;   // direct: dO is scaled by 2^dout_k
    if (a.direct) {
      dout_k = skv_pass_exponent(max_abs_dout(dof, a.do_bf16), ms, reinterpret_cast<float *>(smem + OFF_O + GM::ROWS * 2 * D));
      scale_dout(dof, a.do_bf16, dout_k);
    } else {
      __syncthreads();   // everybody has its rows: they lie in another order from here on
    }
    osc = a.grad_scale ? *a.grad_scale : exp2_neg(dout_k);
    float delta = dot_dout(of, dof, 0);
    delta += swap32_f(delta);
    nlse2 = qi < a.Nq ? -lse * kLog2e : -INFINITY;   // p = 0
    nd = -sm * delta;
    if (kw == 0) {
#pragma unroll
      for (int m = 0; m < KD; ++m) {
        unsigned char *row = smem + GM::OFF_P + skv_tile_off<PSLAB>(32 * qb + lr, m, g);
        *reinterpret_cast<u32x4 *>(row) = qf[m];
        *reinterpret_cast<u32x4 *>(row + GM::PBUF) = dof[m];
      }
    }
    static_for<GM::NBUF - 2>([&](auto i_tag) __attribute__((always_inline)) {
      constexpr int i = decltype(i_tag)::value;
      first[i].commit_chunk(smem + i * GM::BUF, 0);
      first[i].commit_chunk(smem + i * GM::BUF, 1);
      commit_scale(first[i], smem + i * GM::BUF);
    });
    issue(st);
  }
  lds_barrier();

  // ---- AccVGPRs: dQ^T (columns 32db) in tile db; dKV^T of the tile in work (columns 32r of the wave's half) behind them, that of the
  // last tile at the end; in between the constant operands, columns 32r of the wave's half times queries 16j .. 16j + 15 of dO^T and Q^T
  constexpr int C0 = 16 * DB, A0 = C0 + 16 * RT, C1 = 256 - 16 * RT;
  static_assert(A0 + 8 * RT * KQ <= C1, "a wave has 256 AccVGPRs");
  {
    const SkvTileReads<PSLAB> rp(lane);
    unsigned c[RT];
#pragma unroll
    for (int r = 0; r < RT; ++r) c[r] = lds_addr(smem + GM::OFF_P + 2 * (wd * RT + r) * PSLAB + rp.tr[r]);
    static_for<2 * RT * KQ>([&](auto i_tag) __attribute__((always_inline)) {
      constexpr int i = decltype(i_tag)::value, mat = i / (RT * KQ), r = i / KQ % RT, j = i % KQ;   // mat 0: dO, 1: Q
      acc_request_const<A0 + 4 * i, (mat == 0 ? GM::PBUF : 0) + j * 512>(c[r], c[r] ^ 16u);
    });
  }
  static_for<DB>([&](auto i) __attribute__((always_inline)) { acc_zero_tile<decltype(i)::value, 16>(); });

  f32x16 sv[2], dp[2];   // scores and dP of the step in work and of the next one, by turns
  u32x4 xf[2][2];        // dS scale of the previous step and of this one, by turns
  f32x4 tk[2], ta[2], ts[2];   // factors of key rows 8aa + 4g + {0..3}: aa % 2
  constexpr int RING = 4, AHEAD = RING - 1;
  u32x4 fr[RING];
  auto ld_scale = [&](int kblk, int aa) __attribute__((always_inline)) {   // kblk: offset of a block's first row (32 bytes a row, 4 a factor)
    tk[aa % 2] = *reinterpret_cast<const f32x4 *>(smem + kblk + 32 * aa + 16 * g);
    if constexpr (QW == 4) {
      ta[aa % 2] = *reinterpret_cast<const f32x4 *>(smem + kblk + TK * 4 + 32 * aa + 16 * g);
      ts[aa % 2] = *reinterpret_cast<const f32x4 *>(smem + kblk + TK * 8 + 32 * aa + 16 * g);
    }
  };
  // the rows of a finished tile of dKV, 16 bytes of a row per lane: the halves of the wave exchange quads of columns
  const rsrc_t ro = make_rsrc(static_cast<unsigned short *>(a.dkv) + b * a.sdkb + h * a.sdkh, (unsigned)((a.Nk - 1) * (int)a.sdkn * 2 + 2 * D));
  int out_at = (32 * wk + lr - 2 * TK) * (int)a.sdkn * 2 + D * wd + 16 * g;   // (of the tile two before the one in work)
  unsigned ow[4];
  auto out_quad = [&](auto i_tag) __attribute__((always_inline)) {
    constexpr int i = decltype(i_tag)::value, R = 4 * i;
    const float x0 = acc_read_reg<R>() * osc, x1 = acc_read_reg<R + 1>() * osc, x2 = acc_read_reg<R + 2>() * osc, x3 = acc_read_reg<R + 3>() * osc;
    ow[i % 2 * 2] = pack2<G>(x0, x1);
    ow[i % 2 * 2 + 1] = pack2<G>(x2, x3);
  };
  auto out_store = [&](rsrc_t r, auto i_tag) __attribute__((always_inline)) {   // quads 2i and 2i + 1
    swap_halves(ow[0], ow[2]);
    swap_halves(ow[1], ow[3]);
    __builtin_amdgcn_raw_buffer_store_b128(u32x4{ow[0], ow[1], ow[2], ow[3]}, r, out_at + 32 * decltype(i_tag)::value, 0, 0);
  };
  constexpr int OQ = 4 * RT;

  // LDS fragments of a step in the order of their use: dQ and S / dP in turn, dKV; requested AHEAD of it
  constexpr int NSD = KD, NDK = 8, NF = 2 * NSD + NDK;
  static_assert(NF % RING == 0, "a step starts with the fragment registers where the one before left them");
  static_assert(NDK * NB == 2 * KQ && 2 * DB == KD, "fragments of dKV per step; of dQ as many as of S");
  constexpr int S2 = 3 * NSD, SLOTS = S2 + RT * NDK;   // MFMA slots: dQ, S, dP | dKV
  auto cols_of = [&](int off, auto n_tag) __attribute__((always_inline)) -> u32x4 {   // hh = n / DB, db = n % DB
    constexpr int n = decltype(n_tag)::value;
    return rd.cols(smem + off, n % DB, n / DB);
  };
  auto pd_frag = [&](int pbuf, auto n_tag) __attribute__((always_inline)) -> u32x4 {   // queries 16 (n / 2) on of P (n even) or dS
    constexpr int n = decltype(n_tag)::value, off = n % 2 * GM::PMAT + n / 2 * 512, odd = n / 2 % 2 * 8;
    const u32x2 x = lds_read_tr16(smem + pbuf + (p_tr ^ odd) + off), y = lds_read_tr16(smem + pbuf + (p_tr ^ odd ^ 16) + off + 256);
    return u32x4{x[0], x[1], y[0], y[1]};
  };

  // One step of tile t (in kbuf): its block KB (NB == 2) or kw.  kprev, kcur, knext, knext2: first rows of the blocks of the previous
  // step, this one and the next two; snext: factors of the next step's block; pin, pout: P and dS of the tile before and of this one
  auto body = [&](int t, int kbuf, int kprev, int kcur, int knext, int knext2, int scur, int snext, int pin, int pout, auto par_tag)
                  __attribute__((always_inline)) {
    constexpr int CUR = decltype(par_tag)::value, NXT = 1 - CUR, KB = NB == 2 ? CUR : 0;
    // ---- vector work: 8 pairs of P and dS in four items each
    float e0, e1, t0, t1;
    unsigned pp[2], pd[2];
    unsigned char *pw = smem + pout + 2 * (NB == 2 ? KB : kw) * PSLAB;
    auto item = [&](auto i_tag) __attribute__((always_inline)) {
      constexpr int i = decltype(i_tag)::value, x = i / 4, aa = x / 2, e = 2 * (x % 2), v = 4 * aa + e;
      if constexpr (i % 4 == 0) {
        e0 = __builtin_fmaf(QW == 4 ? ta[aa % 2][e] : a_s * tk[aa % 2][e], sv[CUR][v], nlse2);
        e1 = __builtin_fmaf(QW == 4 ? ta[aa % 2][e + 1] : a_s * tk[aa % 2][e + 1], sv[CUR][v + 1], nlse2);
      } else if constexpr (i % 4 == 1) {
        e0 = __builtin_amdgcn_exp2f(e0);
        e1 = __builtin_amdgcn_exp2f(e1);
      } else if constexpr (i % 4 == 2) {
        t0 = __builtin_fmaf(QW == 4 ? ts[aa % 2][e] : sm * tk[aa % 2][e], dp[CUR][v], nd);
        t1 = __builtin_fmaf(QW == 4 ? ts[aa % 2][e + 1] : sm * tk[aa % 2][e + 1], dp[CUR][v + 1], nd);
        pp[e / 2] = pack_h2(e0, e1);
      } else {
        t0 *= e0;
        t1 *= e1;
        pd[e / 2] = pack_h2(t0, t1);
        // (keys past the end have a scale of zero, and whatever their P and dS are they must not reach dQ; their dKV is not stored)
        t0 = mul_zero_wins(t0, tk[aa % 2][e]);
        t1 = mul_zero_wins(t1, tk[aa % 2][e + 1]);
        xf[NXT][aa / 2][2 * (aa % 2) + e / 2] = pack_h2(t0, t1);
        if constexpr (e == 2) {
          unsigned char *w = pw + aa / 2 * PSLAB + (p_row ^ ((aa % 2 ^ KB) << 4));
          *reinterpret_cast<u32x2 *>(w) = u32x2{pp[0], pp[1]};
          *reinterpret_cast<u32x2 *>(w + GM::PMAT) = u32x2{pd[0], pd[1]};
          if constexpr (aa < 2) ld_scale(scur, aa + 2);
        }
      }
    };
    constexpr bool OUT = NB == 1 || KB == 0, COMMIT = NB == 1 || KB == 1;
    rsrc_t ors = ro;
    if constexpr (OUT) {
      if (t < 2) ors = make_rsrc(a.dkv, 0u);   // (there is no such tile)
    }
    unsigned char *kw2 = smem + (kbuf < 2 * GM::BUF ? kbuf + (GM::NBUF - 2) * GM::BUF : kbuf - 2 * GM::BUF);
    auto work = [&](auto s_tag) __attribute__((always_inline)) {
      constexpr int s = decltype(s_tag)::value, i0 = s * 32 / SLOTS, i1 = (s + 1) * 32 / SLOTS;
      static_for<i1 - i0>([&](auto k) __attribute__((always_inline)) { item(ic<i0 + decltype(k)::value>{}); });
      if constexpr (OUT) {   // dKV rows of the tile before the previous one (its accumulators are free from S2 on)
        constexpr int W0 = 3;
        static_assert(W0 + 2 * OQ + 2 <= S2, "read before they are written again");
        if constexpr (s >= W0 && s < W0 + 2 * OQ && (s - W0) % 2 == 0) out_quad(ic<C0 / 4 + (s - W0) / 2>{});
        if constexpr (s > W0 && s < W0 + 2 * OQ && (s - W0) % 4 == 3) out_store(ors, ic<(s - W0) / 4>{});
      }
      if constexpr (COMMIT) {   // the tile NBUF - 2 further, and the one behind it on its way
        if constexpr (s == S2) st.commit_chunk(kw2, 0);
        if constexpr (s == S2 + 5) st.commit_chunk(kw2, 1);
        if constexpr (s == S2 + 10) {
          commit_scale(st, kw2);
          issue(st);
        }
      }
    };
    auto request = [&](auto n_tag) __attribute__((always_inline)) {
      constexpr int n = decltype(n_tag)::value, i = n / 2;
      if constexpr (n < 2 * NSD && n % 2 == 0) fr[n % RING] = cols_of(kprev, ic<i>{});
      else if constexpr (n < 2 * NSD) fr[n % RING] = rd.rows(smem + knext, i);
      else if constexpr (n < NF) fr[n % RING] = pd_frag(pin, ic<KB * NDK + n - 2 * NSD>{});
      else if constexpr (n % 2 == 0) fr[n % RING] = cols_of(kcur, ic<(n - NF) / 2>{});
      else fr[n % RING] = rd.rows(smem + knext2, (n - NF) / 2);
    };
    static_for<NF>([&](auto n_tag) __attribute__((always_inline)) {
      constexpr int n = decltype(n_tag)::value, m = n / 2;
      if constexpr (n < 2 * NSD && n % 2 == 0) {
        QFA_FENCE();
        acc_mfma<_Float16, m % DB, 16>(fr[n % RING], xf[CUR][m / DB]);
        QFA_FENCE();
        work(ic<3 * m>{});
        request(ic<n + AHEAD>{});
      } else if constexpr (n < 2 * NSD) {
        f32x16 zero;
#pragma unroll
        for (int v = 0; v < 16; ++v) zero[v] = 0.f;
        QFA_FENCE();
        sv[NXT] = mfma_h(fr[n % RING], qf[m], m == 0 ? zero : sv[NXT]);
        QFA_FENCE();
        work(ic<3 * m + 1>{});
        request(ic<n + AHEAD>{});
        QFA_FENCE();
        dp[NXT] = mfma_h(fr[n % RING], dof[m], m == 0 ? zero : dp[NXT]);
        QFA_FENCE();
        work(ic<3 * m + 2>{});
      } else {
        constexpr int i = n - 2 * NSD, j = (NB == 2 ? KB * QW : 0) + i / 2, mat = i % 2;
        static_for<RT>([&](auto r_tag) __attribute__((always_inline)) {
          constexpr int r = decltype(r_tag)::value;
          QFA_FENCE();
          acc_mfma_const<C0 + 16 * r, A0 + 4 * ((mat * RT + r) * KQ + j), KB == 0 && i == 0>(fr[n % RING]);
          QFA_FENCE();
          work(ic<S2 + RT * i + r>{});
          if constexpr (r == 0) request(ic<n + AHEAD>{});
        });
      }
    });
    ld_scale(snext, 0);
    ld_scale(snext, 1);
    if constexpr (OUT) out_at += TK * (int)a.sdkn * 2;
    QFA_FENCE();
  };

  // ---- the first step: its scores; the step before it adds nothing (dS is zero, the keys are those of the first tile)
  const int kw_row = NB == 1 ? kw * 1024 : 0, kw_s = GM::TILE + (NB == 1 ? kw * 128 : 0);
  {
#pragma unroll
    for (int v = 0; v < 16; ++v) sv[0][v] = dp[0][v] = 0.f;
#pragma unroll
    for (int m = 0; m < KD; ++m) {
      const u32x4 k = rd.rows(smem + kw_row, m);
      sv[0] = mfma_h(k, qf[m], sv[0]);
      dp[0] = mfma_h(k, dof[m], dp[0]);
    }
    xf[0][0] = xf[0][1] = u32x4{0u, 0u, 0u, 0u};
    static_for<AHEAD>([&](auto n_tag) __attribute__((always_inline)) {
      constexpr int n = decltype(n_tag)::value;
      if constexpr (n % 2 == 0) fr[n] = cols_of(kw_row, ic<n / 2>{});
      else fr[n] = rd.rows(smem + (NB == 2 ? 1024 : GM::BUF + kw_row), n / 2);
    });
    ld_scale(kw_s, 0);
    ld_scale(kw_s, 1);
  }
  lds_barrier();   // the constant operands are there: the buffers of P and dS are free
  int kbuf = 0, kprev = kw_row, pout = GM::OFF_P, t = 0;
  auto next_of = [&](int buf) __attribute__((always_inline)) -> int { return buf == (GM::NBUF - 1) * GM::BUF ? 0 : buf + GM::BUF; };
  // tile t with parity PAR (two blocks per wave: both of them)
  auto tile = [&](auto par_tag) __attribute__((always_inline)) {
    const int knext = next_of(kbuf), pin = 2 * GM::OFF_P + GM::PBUF - pout;
    if constexpr (NB == 2) {
      body(t, kbuf, kprev, kbuf, kbuf + 1024, knext, kbuf + kw_s, kbuf + kw_s + 128, pin, pout, ic<0>{});
      body(t, kbuf, kbuf, kbuf + 1024, knext, knext + 1024, kbuf + kw_s + 128, knext + kw_s, pin, pout, ic<1>{});
      kprev = kbuf + 1024;
    } else {
      body(t, kbuf, kprev, kbuf + kw_row, knext + kw_row, next_of(knext) + kw_row, kbuf + kw_s, knext + kw_s, pin, pout, par_tag);
      kprev = kbuf + kw_row;
    }
    kbuf = knext;
    pout = pin;
    ++t;
    lds_barrier();
  };
  if constexpr (NB == 2) {
    while (t < nt) tile(ic<0>{});
  } else {
    for (;;) {
      tile(ic<0>{});
      if (t == nt) {   // (this step left its dS where the odd ones do)
        xf[0][0] = xf[1][0];
        xf[0][1] = xf[1][1];
        break;
      }
      tile(ic<1>{});
      if (t == nt) break;
    }
  }

  // ---- what is left: dQ of the last step; dKV of the last tile, and under its products the rows of the tile before and dQ's way to
  // the wave's stage, in the two buffers behind the last tile's
  static_for<NSD>([&](auto n_tag) __attribute__((always_inline)) {
    constexpr int n = decltype(n_tag)::value;
    acc_mfma<_Float16, n % DB, 16>(cols_of(kprev, n_tag), xf[0][n / DB]);
  });
  acc_settle();
  const int pin = 2 * GM::OFF_P + GM::PBUF - pout;
  // (zero wins over dS where a key's scale is zero, also where the key exists: what is not finite in a query's dS, because its dO or LSE
  // is not, reaches its dQ here)
  const float osc_q = __builtin_isfinite(nd) && nlse2 == nlse2 ? osc : __builtin_nanf("");
  unsigned char *stage = smem + (wave < 2 ? kbuf : next_of(kbuf)) + wave % 2 * 64 * D;
  static_assert(2 * 64 * D <= GM::BUF && GM::ROWS * 2 * D + 128 <= 2 * GM::BUF, "two stages in a buffer");
  const rsrc_t before = nt > 1 ? ro : make_rsrc(a.dkv, 0u);
  u32x4 ef[3];
  static_for<2>([&](auto n) __attribute__((always_inline)) { ef[decltype(n)::value] = pd_frag(pin, n); });
  static_for<2 * KQ>([&](auto n_tag) __attribute__((always_inline)) {
    constexpr int n = decltype(n_tag)::value, j = n / 2, mat = n % 2;
    if constexpr (n + 2 < 2 * KQ) ef[(n + 2) % 3] = pd_frag(pin, ic<n + 2>{});
    static_for<RT>([&](auto r_tag) __attribute__((always_inline)) {
      constexpr int r = decltype(r_tag)::value, s = RT * n + r;
      QFA_FENCE();
      acc_mfma_const<C1 + 16 * r, A0 + 4 * ((mat * RT + r) * KQ + j), n == 0>(ef[n % 3]);
      QFA_FENCE();
      if constexpr (s < OQ) {
        out_quad(ic<C0 / 4 + s>{});
        if constexpr (s % 2 == 1) out_store(before, ic<s / 2>{});
      }
      if constexpr (KW == 1 && s >= 8 && s < 8 + 4 * DB) {   // quad aa of columns 32db: as store_tile_rows lays them down
        constexpr int q = s - 8, R = 4 * q;
        const float x0 = acc_read_reg<R>() * osc_q, x1 = acc_read_reg<R + 1>() * osc_q, x2 = acc_read_reg<R + 2>() * osc_q, x3 = acc_read_reg<R + 3>() * osc_q;
        *reinterpret_cast<u32x2 *>(stage + lr * 2 * D + ((q ^ lr % 16) * 16) + 8 * g) = u32x2{pack2<G>(x0, x1), pack2<G>(x2, x3)};
      }
    });
  });
  out_at += TK * (int)a.sdkn * 2;
  G *dq = static_cast<G *>(a.dq) + b * a.sdqb + h * a.sdqh;
  if constexpr (KW == 1) {
    const int rows = a.Nq - 32 * qb;   // (none for a wave without queries)
    const rsrc_t rq = make_rsrc(dq + (int64_t)32 * qb * a.sdqn, rows > 0 ? (unsigned)((min(rows, 32) - 1) * (int)a.sdqn * 2 + 2 * D) : 0u);
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int row = 4 * i + lane / 16;
      const u32x4 w = *reinterpret_cast<const u32x4 *>(stage + row * 2 * D + ((lane % 16 ^ row % 16) * 16));
      __builtin_amdgcn_raw_buffer_store_b128(w, rq, row * (int)a.sdqn * 2 + lane % 16 * 16, 0, 0);
    }
  }
  acc_settle();
  static_for<OQ>([&](auto i) __attribute__((always_inline)) {
    out_quad(ic<C1 / 4 + decltype(i)::value>{});
    if constexpr (decltype(i)::value % 2 == 1) out_store(ro, ic<decltype(i)::value / 2>{});
  });
  if constexpr (KW > 1) {
    lds_barrier();   // the tiles are done with: dQ leaves through them
    float *mine = reinterpret_cast<float *>(smem) + qb * (GM::MERGE / 4) + lane;
    f32x16 x[DB] = {acc_read<0>(), acc_read<1>(), acc_read<2>(), acc_read<3>()};
    if (kw > 0) {
#pragma unroll
      for (int i = 0; i < 16 * DB; ++i) mine[i * 64] = x[i / 16][i % 16];
    }
    __syncthreads();
    if (kw > 0 || 32 * qb >= a.Nq) return;
#pragma unroll
    for (int i = 0; i < 16 * DB; ++i) x[i / 16][i % 16] += mine[i * 64];
    store_tile_rows<G, D>(x, osc_q, smem + qb * GM::MERGE, dq, a.sdqn, 32 * qb, a.Nq, lane);
  }
#endif
}

template <typename S, typename G> static void launch_sg(const SkvPassArgs &a, unsigned grid, hipStream_t st) {
  if (a.Nq > 64) skv_pass_kernel<S, G, 4><<<dim3(grid), dim3(256), 0, st>>>(a);
  else skv_pass_kernel<S, G, 2><<<dim3(grid), dim3(256), 0, st>>>(a);
}
int launch_skv_pass128(const SkvPassArgs &a, unsigned grid, bool grad_bf16, hipStream_t st) {
  if (a.scale_dtype == QFA_F32) grad_bf16 ? launch_sg<float, __bf16>(a, grid, st) : launch_sg<float, _Float16>(a, grid, st);
  else grad_bf16 ? launch_sg<_Float16, __bf16>(a, grid, st) : launch_sg<_Float16, _Float16>(a, grid, st);
  return check_launch("qfa_attn_bwd_shared_kv (one pass)");
}

}  // namespace qfa
