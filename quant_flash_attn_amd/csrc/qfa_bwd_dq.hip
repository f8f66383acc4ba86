// dQ:  S^T = Kc.Qc^T (INT8 MFMA), P = exp2(.), dP^T = V.dO^T, dS = P o (dP - delta), dQ^T += Kz^T.dS
// with Kz the dequantized K rounded to 16 bits, for one block of queries over all keys that they see.
//
// The counterpart of the dK / dV kernel (qfa_bwd_dkv.hip; the LDS layout is described there): a workgroup is 4 waves, a wave
// owns QB blocks of 32 queries -- their codes and dO rows are B operands in registers for the whole kernel, their dQ^T
// accumulators live in AccVGPRs by hand -- and keys stream through LDS in tiles of 64 (32 at head_dim 256), three buffers,
// one barrier per tile.
//
// A step (32 keys) is one straight line.  Its MFMAs come in the order
//     dQ of the previous step, all but its last fragment  |  dP  |  S of the next step  |  last fragment of dQ
// and the vector work of this step's P and dS is dealt to them at an even pace, so that no product waits for the vector work
// that it depends on, and no vector work for a product just issued (the last fragment of dQ covers the latency of S).
//
// Two blocks of queries per wave at head_dim 128 (one where that would leave the chip empty: launch_dq), because the A
// operands come out of LDS at 1 KB per MFMA: with one block the LDS reads take as long as the products.  At head_dim 256 the
// operands and accumulators of one block fill the registers; at 64 two waves of one block share a SIMD, since its exponentials
// take longer than its products.  Bound by the instructions a wave can issue (74 vector instructions beside 21 MFMAs of 32
// cycles per 32 x 32 block; matrix pipe busy 72 % at 1.85 GHz on the long sequence below, 54 % on the causal one), then by power.
// Measured, this kernel alone against the one before it (32 queries per wave, scheduled by the compiler, no bias trick):
// 16384 x 16384, 16 heads of 128: 2890 -> 2200 us; 4096 causal, 128 heads of 128: 789 -> 650; 64 heads of 256: 1276 -> 789
// (less since: see the turn of the tile); 2048 causal, 256 heads of 64: 251 -> 226.
#include <type_traits>

#include "qfa_acc.h"
#include "qfa_bwd_common.h"

namespace qfa {

template <int D> struct DqSmem : BwdSlab<D> {
  static constexpr int SLAB = BwdSlab<D>::SLAB;
  static constexpr int OFF_K = 0, OFF_V = OFF_K + D / 32 * SLAB, OFF_KT = OFF_V + D / 16 * SLAB,
                       OFF_C = OFF_KT + BwdWs<D>::T_BYTES, C_COPY = (BwdWs<D>::CK_BYTES + 1023) / 1024 * 1024,
                       BUF = OFF_C + C_COPY;
  static_assert(3 * BUF <= 160 * 1024, "three tile buffers");
};

// QB: 32-query blocks per wave
template <typename T, int D, int QB, bool CAUSAL> __global__ __launch_bounds__(256, D == 64 ? 2 : 1) void bwd_dq_kernel(BwdArgs a) {
#ifdef __HIP_DEVICE_COMPILE__   // (with the body in view the host pass of this compiler emits no launch stub)
  typedef BwdWs<D> WS;
  typedef DqSmem<D> SM;
  constexpr int TILE = WS::TILE, NSTEP = TILE / 32;   // keys per tile, steps of 32 per tile
  constexpr int KS = D / 32, DB = D / 32, KD = D / 16, SLAB = SM::SLAB;
  constexpr int QUERIES = 32 * QB;   // queries per wave
  __shared__ __attribute__((aligned(256))) unsigned char smem[3 * SM::BUF];

  const int L = blockIdx.x;
  const int vid = (L % 8) * a.blocks_per_xcd + (L / 8);
  if (vid >= a.total_blocks) return;
  int bh = vid / a.nblocks;
  int mb = vid % a.nblocks;
  if (CAUSAL) {
    // longest rows first, 2^group_log2 heads at a time (ids cycle through the heads of a group): with one
    // head after the other the last head's long blocks start while the chip is already draining
    const int GL = a.group_log2;
    const int pb = bh >> GL << GL;
    if (pb + (1 << GL) <= a.total_blocks / a.nblocks) {
      const int idx = (bh - pb) * a.nblocks + mb;
      bh = pb + (idx & ((1 << GL) - 1));
      mb = idx >> GL;
    }
    mb = a.nblocks - 1 - mb;
  }
  const int64_t b = index_div(bh, a.H), h = bh - b * a.H;
  // this workgroup's keys: key0 .. key0 + Nk - 1, a sequence of its own whose mask is shifted
  const int key0 = blockIdx.y * a.per_split, Nk = min(a.per_split, a.Nk - key0);
  const int m0 = mb * 4 * QUERIES;
  const int tid = threadIdx.x, lane = tid % 64, lr = lane % 32, g = lane / 32;
  const int wave = __builtin_amdgcn_readfirstlane(tid / 64);
  const int q_first = m0 + wave * QUERIES;

  const int8_t *qc_bh = a.qc + b * a.sqb + h * a.sqh;
  const unsigned char *kc_bh = reinterpret_cast<const unsigned char *>(a.kc + b * a.skb + h * a.skh + key0 * a.skn);
  const unsigned char *v_bh = reinterpret_cast<const unsigned char *>(reinterpret_cast<const T *>(a.v) + b * a.svb + h * a.svh + key0 * a.svn);
  const T *do_bh = reinterpret_cast<const T *>(a.dout) + b * a.sdob + h * a.sdoh;
  const unsigned char *wsk_bh = a.ws_k + ((int64_t)bh * a.tiles_k + key0 / TILE) * WS::K_BLOB;
  const unsigned char *wsq_bh = a.ws_q + (int64_t)bh * a.tiles_q * WS::Q_BLOB;

  const int coff = CAUSAL ? a.Nk - a.Nq - key0 : 0;   // causal: query i keeps keys j <= i + coff (mask aligned to the last key)
  const int ntiles = ((CAUSAL ? min(Nk, m0 + 4 * QUERIES + coff) : Nk) + TILE - 1) / TILE;
  const int wtiles = q_first >= a.Nq ? 0 : ((CAUSAL ? min(Nk, q_first + QUERIES + coff) : Nk) + TILE - 1) / TILE;

  // ---- tile copies (direct to LDS)
  typedef SlabCopy<TILE, KS> CopyK;
  typedef SlabCopy<TILE, KD> CopyV;
  typedef BlobCopy<WS::T_BYTES, SM::C_COPY> CopyB;
  const CopyK cp_k(lane, (unsigned)a.skn);
  const CopyV cp_v(lane, (unsigned)a.svn * 2u);
  // pieces of a tile; with one step per tile the FIRST of them, the codes and the constants, are what the turn of the tile waits for
  constexpr int PIECES = CopyK::N + CopyV::N + CopyB::N, FIRST = NSTEP == 1 ? CopyK::N + 1 : PIECES;
  struct TileDesc { rsrc_t k, v, b; unsigned char *dst; };
  auto tile_desc = [&](int t) __attribute__((always_inline)) -> TileDesc {
    const int rows = t < ntiles ? min(TILE, Nk - TILE * t) : 0;
    return {cp_k.desc(kc_bh + (int64_t)t * TILE * a.skn, rows), cp_v.desc(v_bh + (int64_t)t * TILE * a.svn * 2, rows),
            make_rsrc(wsk_bh + (int64_t)t * WS::K_BLOB, rows > 0 ? (unsigned)WS::K_BLOB : 0u), smem + t % 3 * SM::BUF};
  };
  auto copy_piece = [&](const TileDesc &d, int i) __attribute__((always_inline)) {   // i: a compile-time constant everywhere
    if constexpr (FIRST < PIECES) {
      if (i < FIRST - 1) cp_k.piece(i, d.k, d.dst + SM::OFF_K, wave);
      else if (i == FIRST - 1) CopyB::piece(CopyB::N - 1, d.b, d.dst + SM::OFF_KT, d.dst + SM::OFF_C, wave, lane);
      else if (i < FIRST + CopyV::N) cp_v.piece(i - FIRST, d.v, d.dst + SM::OFF_V, wave);
      else CopyB::piece(i - FIRST - CopyV::N, d.b, d.dst + SM::OFF_KT, d.dst + SM::OFF_C, wave, lane);
      return;
    }
    if (i < CopyV::N) cp_v.piece(i, d.v, d.dst + SM::OFF_V, wave);
    else if (i < CopyV::N + CopyK::N) cp_k.piece(i - CopyV::N, d.k, d.dst + SM::OFF_K, wave);
    else CopyB::piece(i - CopyV::N - CopyK::N, d.b, d.dst + SM::OFF_KT, d.dst + SM::OFF_C, wave, lane);
  };
  auto copy_tile = [&](int t) __attribute__((always_inline)) {
    const TileDesc d = tile_desc(t);
#pragma unroll
    for (int i = 0; i < PIECES; ++i) copy_piece(d, i);
  };
  copy_tile(0);
  copy_tile(1);

  // ---- this lane's queries: codes and dO rows as B operands for the whole kernel, constants prepared by prep_q
  i32x4 qf[QB][KS];
  u32x4 dof[QB][KD];
  u32x2 corr_q[QB];
  f32x16 nd[QB];     // -delta: dP - delta comes out of the MFMAs
  float a_i[QB], nlse[QB];
  int k_hi[QB];      // last key that the lane's query sees
#pragma unroll
  for (int qb = 0; qb < QB; ++qb) {
    const int qi = q_first + 32 * qb + lr, qc = min(qi, a.Nq - 1);
    k_hi[qb] = CAUSAL ? min(qc + coff, Nk - 1) : Nk - 1;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
      qf[qb][ks] = *reinterpret_cast<const i32x4 *>(qc_bh + (int64_t)qc * a.sqn + ks * 32 + g * 16);
#pragma unroll
    for (int kd = 0; kd < KD; ++kd)
      dof[qb][kd] = *reinterpret_cast<const u32x4 *>(do_bh + (int64_t)qc * a.sdon + kd * 16 + g * 8);
    const unsigned *cq = reinterpret_cast<const unsigned *>(wsq_bh + (int64_t)(qc / TILE) * WS::Q_BLOB + WS::T_BYTES);
    const int ql = qc % TILE;
    corr_q[qb] = u32x2{cq[2 * ql + g], g ? 0u : QFA_BIAS_B(T)};
    a_i[qb] = __builtin_bit_cast(float, cq[2 * TILE + ql]);
    nlse[qb] = __builtin_bit_cast(float, cq[3 * TILE + ql]);
    const float d = __builtin_bit_cast(float, cq[4 * TILE + ql]);
#pragma unroll
    for (int v = 0; v < 16; ++v) nd[qb][v] = d;
  }

  const int row_l = slab_row(lr, g);   // this lane's read offset in a slab (row lr, k-group g)

  // accumulators: dQ^T of (query block qb, columns 32db) in tile qb * DB + db
  constexpr int ACC = QB * DB;
  acc_zero<ACC>();

  i32x16 bias, si[QB];     // si: scores of the step in work, biased integers without the zero-point term
#pragma unroll
  for (int v = 0; v < 16; ++v) bias[v] = QFA_BIAS_BITS;
  u32x4 ds[2][QB][2];      // dS of the previous step and of this one, by turns
#pragma unroll
  for (int qb = 0; qb < QB; ++qb)
#pragma unroll
    for (int hh = 0; hh < 2; ++hh) ds[0][qb][hh] = u32x4{0u, 0u, 0u, 0u};

  auto ld = [&](int off) -> u32x4 { return *reinterpret_cast<const u32x4 *>(smem + off); };
  auto ldf = [&](int off) -> f32x4 { return *reinterpret_cast<const f32x4 *>(smem + off); };

  // What a step finds in registers, requested at the end of the previous one: the first fragments of Kz^T of the previous
  // step, the correction operand, and the scales of the first key rows
  constexpr int NX = 2 * DB, NP = KD;      // fragments of dQ and of dP; KS of S
  constexpr int RING = 4;                  // fragments requested three fragments ahead
  u32x4 fr[RING];
  u32x2 corr_k = {0u, QFA_BIAS_A(T)};
  f32x4 sk[2];                             // scales of key rows 8aa + 4g + {0..3}: aa % 2
  auto ld_sk = [&](int buf, int mbk, int aa) __attribute__((always_inline)) {
    sk[aa % 2] = ldf(buf + SM::OFF_C + 2 * TILE * 4 + 16 * g + mbk * 128 + aa * 32);
  };
  auto request_head = [&](int buf, int mbk, int kt_prev) __attribute__((always_inline)) {
#pragma unroll
    for (int n = 0; n < RING - 1; ++n) fr[n] = ld(kt_prev + n * 1024);
    corr_k[0] = *reinterpret_cast<const unsigned *>(smem + buf + SM::OFF_C + (2 * lr + g) * 4 + mbk * 256);
    ld_sk(buf, mbk, 0);
  };

  // One step: 32 keys (part mbk of the tile in buffer `buf`) against the wave's queries.  `nbuf`: buffer of the next step.
  auto body = [&](int t, int buf, int nbuf, int kt_prev, auto mbk_tag, auto masked_tag, const u32x4 (&ds_in)[QB][2],
                  u32x4 (&ds_out)[QB][2]) __attribute__((always_inline)) {
    constexpr bool MASKED = decltype(masked_tag)::value;
    constexpr int mbk = decltype(mbk_tag)::value;
    constexpr bool LAST = mbk == NSTEP - 1;
    const int rowb = buf + row_l + mbk * 1024 + SM::OFF_V;
    const int nrow = nbuf + row_l + (LAST ? 0 : (mbk + 1) * 1024) + SM::OFF_K;
    const int j0 = TILE * t + 32 * mbk + 4 * g;

    // MFMA slots: fragments 0 .. NX-2 of dQ, dP, S of the next step, fragment NX-1 of dQ; QB slots per fragment
    constexpr int XA = NX - 1, P0 = XA, S0 = P0 + NP, XZ = S0 + KS, SLOTS = QB * (XZ + 1);
    // ---- the vector work: P in 16 QB half items (even: scaling of a pair of scores, odd: exponentials) over the slots
    // from the third one on, dS in 8 QB dwords over the slots from the third behind dP
    constexpr int P_LO = 2, D_LO = QB * S0 + 2, HALF = 16 * QB, DSW = 8 * QB;
    f32x16 f[QB], dp[QB];
    auto half_item = [&](auto i_tag) __attribute__((always_inline)) {
      constexpr int i = decltype(i_tag)::value, x = i / 2, qb = x / 4 % QB, aa = 2 * (x / (4 * QB)) + x / 2 % 2, v = 4 * aa + 2 * (x % 2);
      if constexpr (i % 2 == 0) {
        f[qb][v] = __builtin_fmaf(a_i[qb], f[qb][v] * sk[aa % 2][2 * (x % 2)], nlse[qb]);
        f[qb][v + 1] = __builtin_fmaf(a_i[qb], f[qb][v + 1] * sk[aa % 2][2 * (x % 2) + 1], nlse[qb]);
      } else {
        f[qb][v] = __builtin_amdgcn_exp2f(f[qb][v]);
        f[qb][v + 1] = __builtin_amdgcn_exp2f(f[qb][v + 1]);
      }
      // the scales of quad aa + 2 replace those of aa behind their last use
      constexpr int last0 = QB == 2 ? 10 : 2, last1 = QB == 2 ? 14 : 6;
      if constexpr (i == last0 + 1) ld_sk(buf, mbk, 2);
      if constexpr (i == last1 + 1) ld_sk(buf, mbk, 3);
    };
    auto ds_dword = [&](auto k_tag) __attribute__((always_inline)) {
      constexpr int k = decltype(k_tag)::value, qb = k / 4 % QB, hh = k / (4 * QB), e = k % 4, v = 8 * hh + 2 * e;
      float x0 = f[qb][v] * dp[qb][v], x1 = f[qb][v + 1] * dp[qb][v + 1];
      if constexpr (MASKED) {   // dS and not P: dP of a masked pair may be anything (V may be infinite there)
        const int j = j0 + 8 * (v / 4) + v % 4;
        x0 = j <= k_hi[qb] ? x0 : 0.f;
        x1 = j + 1 <= k_hi[qb] ? x1 : 0.f;
      }
      ds_out[qb][hh][e] = pack2<T>(x0, x1);
    };
    // the copy's pieces are spread over the slots behind the turn of the tile
    TileDesc td;
    constexpr int CSLOTS = SLOTS - QB * XA;
    auto work = [&](auto slot_tag) __attribute__((always_inline)) {
      constexpr int s = decltype(slot_tag)::value;
      if constexpr (s >= P_LO && s < D_LO) {
        constexpr int n = D_LO - P_LO, i0_ = (s - P_LO) * HALF / n, i1_ = (s - P_LO + 1) * HALF / n;
        static_for<i1_ - i0_>([&](auto k) __attribute__((always_inline)) { half_item(ic<i0_ + decltype(k)::value>{}); });
      }
      if constexpr (s >= D_LO) {
        constexpr int n = SLOTS - D_LO, i0_ = (s - D_LO) * DSW / n, i1_ = (s - D_LO + 1) * DSW / n;
        static_for<i1_ - i0_>([&](auto k) __attribute__((always_inline)) { ds_dword(ic<i0_ + decltype(k)::value>{}); });
      }
      if constexpr (LAST && s >= QB * XA) {
        constexpr int c = s - QB * XA, p0 = c * PIECES / CSLOTS, p1 = (c + 1) * PIECES / CSLOTS;
        static_for<p1 - p0>([&](auto p) __attribute__((always_inline)) { copy_piece(td, p0 + decltype(p)::value); });
      }
    };
    u32x4 fz;   // the last fragment of dQ, requested with the others: its buffer may be refilled behind the barrier
    auto request = [&](auto n_tag) __attribute__((always_inline)) {
      constexpr int n = decltype(n_tag)::value;
      if constexpr (n < P0) fr[n % RING] = ld(kt_prev + n * 1024);
      else if constexpr (n < S0) fr[n % RING] = ld(rowb + (n - P0) * SLAB);
      else if constexpr (n < XZ) fr[n % RING] = ld(nrow + (n - S0) * SLAB);
    };

#pragma unroll
    for (int qb = 0; qb < QB; ++qb) f[qb] = mfma_16b_k8<T>(corr_k, corr_q[qb], __builtin_bit_cast(f32x16, si[qb]));
    // The turn of the tile: the next one has landed, the one after it goes into the buffer of the previous one, whose last
    // fragments have been requested.  It comes before the first request of V: three fragments' products follow whose operands are
    // there (dQ of 16384 x 16384, 16 heads of 128: 2273 -> 2246 us against a turn behind them, 4096 causal 671 -> 666).  With one
    // step per tile (head_dim 256) the last pieces of a copy have 15 products' time until the next turn, and the wave waited for
    // them (42 % of its time): there only the codes and constants of the next tile have to be there, V and Kz^T one turn later.
    // 64 heads of 4096 causal: 818 -> 704 us; the whole backward without a mask 3394 -> 2976 us
    auto turn = [&]() __attribute__((always_inline)) {
      vm_wait<PIECES - FIRST>();
      lds_barrier();
      td = tile_desc(t + 2);
    };
    constexpr int TURN = XA - RING + 1;   // in front of this fragment's products
    static_for<XA>([&](auto n_tag) __attribute__((always_inline)) {     // hh = n / DB, db = n % DB
      constexpr int n = decltype(n_tag)::value;
      if constexpr (LAST && n == TURN) turn();
      static_for<QB>([&](auto qb_tag) __attribute__((always_inline)) {
        constexpr int qb = decltype(qb_tag)::value;
        QFA_FENCE();
        acc_mfma<T, qb * DB + n % DB, ACC>(fr[n % RING], ds_in[qb][n / DB]);
        QFA_FENCE();
        work(ic<QB * n + qb>{});
        if constexpr (qb == 0) {
          request(ic<n + RING - 1>{});
          if constexpr (n == 0) {
            ld_sk(buf, mbk, 1);
            fz = ld(kt_prev + XA * 1024);
          }
        }
      });
    });
    static_for<NP>([&](auto m_tag) __attribute__((always_inline)) {
      constexpr int m = decltype(m_tag)::value, n = P0 + m;
      static_for<QB>([&](auto qb_tag) __attribute__((always_inline)) {
        constexpr int qb = decltype(qb_tag)::value;
        QFA_FENCE();
        dp[qb] = mfma_16b<T>(fr[n % RING], dof[qb][m], m == 0 ? nd[qb] : dp[qb]);
        QFA_FENCE();
        work(ic<QB * n + qb>{});
        if constexpr (qb == 0) request(ic<n + RING - 1>{});
      });
    });
    static_for<KS>([&](auto m_tag) __attribute__((always_inline)) {
      constexpr int m = decltype(m_tag)::value, n = S0 + m;
      static_for<QB>([&](auto qb_tag) __attribute__((always_inline)) {
        constexpr int qb = decltype(qb_tag)::value;
        QFA_FENCE();
        si[qb] = mfma_i8(__builtin_bit_cast(i32x4, fr[n % RING]), qf[qb][m], m == 0 ? bias : si[qb]);
        QFA_FENCE();
        work(ic<QB * n + qb>{});
        if constexpr (qb == 0) request(ic<n + RING - 1>{});
      });
    });
    const int kt = buf + SM::OFF_KT + row_l + mbk * (2 * DB * 1024);
    static_for<QB>([&](auto qb_tag) __attribute__((always_inline)) {
      constexpr int qb = decltype(qb_tag)::value;
      QFA_FENCE();
      acc_mfma<T, qb * DB + XA % DB, ACC>(fz, ds_in[qb][XA / DB]);
      QFA_FENCE();
      if constexpr (qb == 0) request_head(nbuf, LAST ? 0 : mbk + 1, kt);
      work(ic<QB * XZ + qb>{});
    });
    QFA_FENCE();
  };

  dma_wait();
  __syncthreads();
  int t = 0, buf = 0, nbuf = SM::BUF;
  if (wtiles > 0) {
#pragma unroll
    for (int qb = 0; qb < QB; ++qb) {
      si[qb] = bias;
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) si[qb] = mfma_i8(__builtin_bit_cast(i32x4, ld(row_l + SM::OFF_K + ks * SLAB)), qf[qb][ks], si[qb]);
    }
    int kt_prev = SM::OFF_KT + row_l;     // (dS is zero: the product adds nothing)
    request_head(0, 0, kt_prev);
    // full tiles, then masked ones (diagonal, ragged end)
    auto tiles = [&](int t_end, auto masked_tag) __attribute__((always_inline)) {
      for (; t < t_end; ++t) {
        static_for<NSTEP>([&](auto mbk_tag) __attribute__((always_inline)) {
          constexpr int mbk = decltype(mbk_tag)::value;
          body(t, buf, mbk == NSTEP - 1 ? nbuf : buf, kt_prev, mbk_tag, masked_tag, ds[mbk % 2], ds[(mbk + 1) % 2]);
          kt_prev = buf + SM::OFF_KT + row_l + mbk * (2 * DB * 1024);
        });
        if constexpr (NSTEP % 2 == 1) {
#pragma unroll
          for (int qb = 0; qb < QB; ++qb) { ds[0][qb][0] = ds[1][qb][0]; ds[0][qb][1] = ds[1][qb][1]; }
        }
        const int b2 = 3 * SM::BUF - buf - nbuf;
        buf = nbuf;
        nbuf = b2;
      }
    };
    tiles(min(wtiles, min(Nk / TILE, CAUSAL ? (q_first + coff + 1) / TILE : wtiles)), std::false_type{});
    tiles(wtiles, std::true_type{});
    static_for<NX>([&](auto n_tag) __attribute__((always_inline)) {
      constexpr int n = decltype(n_tag)::value;
      const u32x4 tk = ld(kt_prev + n * 1024);
      static_for<QB>([&](auto qb) __attribute__((always_inline)) { acc_mfma<T, decltype(qb)::value * DB + n % DB, ACC>(tk, ds[0][decltype(qb)::value][n / DB]); });
    });
  }
  for (; t < ntiles; ++t) {   // tiles that only other waves see
    dma_wait();
    lds_barrier();
    copy_tile(t + 2);
  }
  // what only the epilogue needs is read and formed here: held in scalar registers through the loop it would push others out,
  // and behind the barrier its latency would be seen
  typedef __attribute__((address_space(4))) const BwdArgs KernArgs;
  KernArgs *ep = (KernArgs *)__builtin_amdgcn_kernarg_segment_ptr();
  int bh_ = bh;
  asm volatile("" : "+s"(ep), "+s"(bh_));
  const int64_t eb = index_div(bh_, ep->H), eh = bh_ - eb * ep->H;
  void *dq = ep->dq;
  int64_t dq_at = eb * ep->sdqb + eh * ep->sdqh + blockIdx.y * ep->split_stride, sdqn = ep->sdqn;
  float sm = ep->sm_scale;
  int f32 = ep->grad_f32;
  asm volatile("" : "+s"(dq), "+s"(dq_at), "+s"(sdqn), "+s"(sm), "+s"(f32));
  acc_settle();
  __syncthreads();   // the tile buffers are done with: the output stages overlay them
  static_assert(4 * 32 * 2 * D <= 3 * SM::BUF, "output staging fits the tile buffers");
  unsigned char *stage = smem + wave * (32 * 2 * D);
  if (f32) {
    float *dq_bh = reinterpret_cast<float *>(dq) + dq_at;
    static_for<QB>([&](auto qb_tag) __attribute__((always_inline)) {
      constexpr int qb = decltype(qb_tag)::value;
      acc_store_rows_f32<D, qb * DB>(sm, dq_bh, sdqn, q_first + 32 * qb, a.Nq, lane);
    });
    return;
  }
  T *dq_bh = reinterpret_cast<T *>(dq) + dq_at;
  static_for<QB>([&](auto qb_tag) __attribute__((always_inline)) {
    constexpr int qb = decltype(qb_tag)::value;
    acc_store_rows<T, D, qb * DB>(sm, stage, dq_bh, sdqn, q_first + 32 * qb, a.Nq, lane);
  });
#endif
}

template <typename T, int D, int QB> static int launch_dq_qb(BwdArgs a, int64_t BH, bool causal, int splits, hipStream_t st) {
  a.nblocks = (a.Nq + 128 * QB - 1) / (128 * QB);
  a.group_log2 = bwd_group_log2(a.Nk, D, true);   // per head the kernel streams Kc, V and Kz^T: 5 bytes per key and d
  const int64_t total = (int64_t)a.nblocks * BH;
  if (total > 0x3fffffffLL) return set_error(QFA_EUNSUPPORTED, "attn_bwd: too many query blocks for one launch");
  a.total_blocks = (int)total;
  a.blocks_per_xcd = (a.total_blocks + 7) / 8;
  const dim3 grid((unsigned)(a.blocks_per_xcd * 8), (unsigned)splits);
  if (causal) bwd_dq_kernel<T, D, QB, true><<<grid, dim3(256), 0, st>>>(a);
  else bwd_dq_kernel<T, D, QB, false><<<grid, dim3(256), 0, st>>>(a);
  return check_launch("qfa_attn_bwd (dq)");
}

template <typename T, int D> int launch_dq(BwdArgs a, int64_t BH, bool causal, int blocks, int splits, hipStream_t st) {
  if constexpr (D == 128) {
    if (blocks == 2) return launch_dq_qb<T, D, 2>(a, BH, causal, splits, st);
  }
  return launch_dq_qb<T, D, 1>(a, BH, causal, splits, st);
}
template int launch_dq<__bf16, 64>(BwdArgs, int64_t, bool, int, int, hipStream_t);
template int launch_dq<__bf16, 128>(BwdArgs, int64_t, bool, int, int, hipStream_t);
template int launch_dq<__bf16, 256>(BwdArgs, int64_t, bool, int, int, hipStream_t);
template int launch_dq<_Float16, 64>(BwdArgs, int64_t, bool, int, int, hipStream_t);
template int launch_dq<_Float16, 128>(BwdArgs, int64_t, bool, int, int, hipStream_t);
template int launch_dq<_Float16, 256>(BwdArgs, int64_t, bool, int, int, hipStream_t);

}  // namespace qfa
