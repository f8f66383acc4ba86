// dK and dV:  S = Qc.Kc^T (INT8 MFMA), P = exp2(.), dP = dO.V^T, dV^T += dO^T.P, dS = P o (dP - delta), dK^T += Qz^T.dS
// with Qz the dequantized Q rounded to 16 bits, for one block of keys over all queries that see them.
//
// Work split.  One workgroup = 4 waves, ONE wave per SIMD (two at head_dim 64); a wave owns 64 keys (or 32, see launch_dkv):
// their codes and V rows are B operands in registers for the whole kernel, their dK^T and dV^T accumulators (up to 256
// registers) live in AccVGPRs by hand (qfa_acc.h), which leaves the other 256 registers to everything else.  Queries stream
// through LDS in tiles of 64 (32 at head_dim 256), three buffers, one barrier per tile.
//
// Why one wave: the A operand of every product comes out of LDS, 1 KB per MFMA, and two waves of 32 keys per SIMD read all
// of it twice; 64 keys per wave use every fragment for two MFMAs.  The version before this one split the work of 32 keys
// over a pair of waves (scores | dP) that met at a workgroup barrier per 32 queries; its matrix pipe was busy 42 % of the
// time.  With one wave nobody fills its waits, so the instruction stream is written out: a step (32 queries) is one
// straight line in which every MFMA is followed by its share of the vector work and of the LDS requests, pinned by
// scheduling fences:
//     dK of the previous step  |  P of this one, first part
//     dP                       |  P, second part
//     dV, S of the next step   |  dS
// so that no product waits for the vector work it depends on.  What bounds it: the instructions one wave can issue (about
// 5 cycles each, 16 + 2 MFMAs' worth of vector work per block against 29 MFMAs of 32 cycles), then power.
// Measured, the whole backward before and after: 16384 x 16384, 16 heads of 128: 6.70 -> 5.81 ms (matrix pipe of this kernel
// busy 42 -> 72 % of the time, at 1.85 GHz); 4096 causal, 128 heads of 128: 1.97 -> 1.79; 64 heads of 256: 2.74 -> 2.31;
// 2048 causal, 256 heads of 64: 0.737 -> 0.68 (there exponentials and vector work take longer than the products).
//
// LDS layout of a tile.  Rows of codes and of dO are cut into slabs of 32 bytes: slab s holds bytes 32s..32s+31 of every
// row, so that fragment s of 32 rows is 1 KB in one piece and all fragments of a tile are one address plus an immediate
// (no XOR per fragment).  Inside a slab the two 16-byte halves of rows 8-15 and 24-31 are swapped, and slabs are 128 bytes
// apart modulo 256: 16 lanes reading 16 rows, and 32 lanes of a transposing read (4 rows x 2 slabs), hit all banks once.
// The transposed Qz tile is staged in the order of its reads (qt_offset).
#include <type_traits>

#include "qfa_acc.h"
#include "qfa_bwd_common.h"

namespace qfa {

template <int D> struct DkvSmem : BwdSlab<D> {
  static constexpr int SLAB = BwdSlab<D>::SLAB;
  static constexpr int OFF_Q = 0, OFF_DO = OFF_Q + D / 32 * SLAB, OFF_QT = OFF_DO + D / 16 * SLAB,
                       OFF_C = OFF_QT + BwdWs<D>::T_BYTES, C_COPY = (BwdWs<D>::CQ_BYTES + 1023) / 1024 * 1024,
                       BUF = OFF_C + C_COPY;
  static_assert(3 * BUF <= 160 * 1024, "three tile buffers");
};

// KB: 32-key blocks per wave
template <typename T, int D, int KB, bool CAUSAL> __global__ __launch_bounds__(256, D == 64 ? 2 : 1) void bwd_dkv_kernel(BwdArgs a) {
#ifdef __HIP_DEVICE_COMPILE__   // (with the body in view the host pass of this compiler emits no launch stub)
  typedef BwdWs<D> WS;
  typedef DkvSmem<D> SM;
  constexpr int TILE = WS::TILE, NSTEP = TILE / 32;   // queries per tile, steps of 32 per tile
  constexpr int KS = D / 32, DB = D / 32, KD = D / 16, SLAB = SM::SLAB;
  constexpr int KEYS = 32 * KB;   // keys per wave
  __shared__ __attribute__((aligned(256))) unsigned char smem[3 * SM::BUF];

  const int L = blockIdx.x;
  const int vid = (L % 8) * a.blocks_per_xcd + (L / 8);
  if (vid >= a.total_blocks) return;
  int bh = vid / a.nblocks;
  int nbk = vid % a.nblocks;   // causal: early key blocks see the most queries and come first
  if (CAUSAL && a.group_log2 > 0) {
    // key blocks of 2^group_log2 heads dispatched together, from the longest down; the launcher allows it only while the
    // query-side tiles of the group fit an XCD's L2
    const int GL = a.group_log2;
    const int pb = bh >> GL << GL;
    if (pb + (1 << GL) <= a.total_blocks / a.nblocks) {
      const int idx = (bh - pb) * a.nblocks + nbk;
      bh = pb + (idx & ((1 << GL) - 1));
      nbk = idx >> GL;
    }
  }
  const int64_t b = index_div(bh, a.H), h = bh - b * a.H;
  // this workgroup's queries: q0 .. q0 + Nq - 1, a sequence of its own whose mask is shifted (late ones first: causal, they see
  // the most keys)
  const int q0 = a.last_part - (int)blockIdx.y * a.per_split, Nq = min(a.per_split, a.Nq - q0);
  const int n0 = nbk * 4 * KEYS;
  const int tid = threadIdx.x, lane = tid % 64, lr = lane % 32, g = lane / 32;
  const int wave = __builtin_amdgcn_readfirstlane(tid / 64);
  const int k_first = n0 + wave * KEYS;

  const unsigned char *qc_bh = reinterpret_cast<const unsigned char *>(a.qc + b * a.sqb + h * a.sqh + q0 * a.sqn);
  const int8_t *kc_bh = a.kc + b * a.skb + h * a.skh;
  const T *v_bh = reinterpret_cast<const T *>(a.v) + b * a.svb + h * a.svh;
  const unsigned char *do_bh = reinterpret_cast<const unsigned char *>(reinterpret_cast<const T *>(a.dout) + b * a.sdob + h * a.sdoh + q0 * a.sdon);
  const unsigned char *wsk_bh = a.ws_k + (int64_t)bh * a.tiles_k * WS::K_BLOB;
  const unsigned char *wsq_bh = a.ws_q + ((int64_t)bh * a.tiles_q + q0 / TILE) * WS::Q_BLOB;

  const int coff = CAUSAL ? a.Nk - a.Nq + q0 : 0;   // causal: key j is seen by the queries i >= j - coff
  const int it0 = CAUSAL ? max(n0 - coff, 0) / TILE : 0;
  const int ntiles = (Nq + TILE - 1) / TILE;

  // ---- tile copies (direct to LDS)
  typedef SlabCopy<TILE, KS> CopyQ;
  typedef SlabCopy<TILE, KD> CopyDo;
  typedef BlobCopy<WS::T_BYTES, SM::C_COPY> CopyB;
  const CopyQ cp_q(lane, (unsigned)a.sqn);
  const CopyDo cp_do(lane, (unsigned)a.sdon * 2u);
  // pieces of a tile; at head_dim 256 without a mask the FIRST of them, the codes and the constants, are what the turn of the tile waits for
  constexpr bool EARLY = NSTEP == 1 && !CAUSAL;
  constexpr int PIECES = CopyQ::N + CopyDo::N + CopyB::N, FIRST = EARLY ? CopyQ::N + 1 : PIECES;
  struct TileDesc { rsrc_t q, g, b; unsigned char *dst; };
  auto tile_desc = [&](int t) __attribute__((always_inline)) -> TileDesc {
    const int rows = min(TILE, Nq - TILE * t);
    return {cp_q.desc(qc_bh + (int64_t)t * TILE * a.sqn, rows), cp_do.desc(do_bh + (int64_t)t * TILE * a.sdon * 2, rows),
            make_rsrc(wsq_bh + (int64_t)t * WS::Q_BLOB, rows > 0 ? (unsigned)WS::Q_BLOB : 0u), smem + (t - it0) % 3 * SM::BUF};
  };
  auto copy_piece = [&](const TileDesc &d, int i) __attribute__((always_inline)) {   // i: a compile-time constant everywhere
    if constexpr (EARLY) {
      if (i < FIRST - 1) cp_q.piece(i, d.q, d.dst + SM::OFF_Q, wave);
      else if (i == FIRST - 1) CopyB::piece(CopyB::N - 1, d.b, d.dst + SM::OFF_QT, d.dst + SM::OFF_C, wave, lane);
      else if (i < FIRST + CopyDo::N) cp_do.piece(i - FIRST, d.g, d.dst + SM::OFF_DO, wave);
      else CopyB::piece(i - FIRST - CopyDo::N, d.b, d.dst + SM::OFF_QT, d.dst + SM::OFF_C, wave, lane);
      return;
    }
    if (i < CopyDo::N) cp_do.piece(i, d.g, d.dst + SM::OFF_DO, wave);
    else if (i < CopyDo::N + CopyQ::N) cp_q.piece(i - CopyDo::N, d.q, d.dst + SM::OFF_Q, wave);
    else CopyB::piece(i - CopyDo::N - CopyQ::N, d.b, d.dst + SM::OFF_QT, d.dst + SM::OFF_C, wave, lane);
  };
  auto copy_tile = [&](int t) __attribute__((always_inline)) {
    const TileDesc d = tile_desc(t);
#pragma unroll
    for (int i = 0; i < PIECES; ++i) copy_piece(d, i);
  };
  copy_tile(it0);
  copy_tile(it0 + 1);

  // ---- this lane's keys: codes and V rows as B operands for the whole kernel, correction digits, scale
  i32x4 kf[KB][KS];
  u32x4 vf[KB][KD];
  u32x2 corr_k[KB];
  float sk[KB];
  int q_lo[KB];   // first query that sees the lane's key (none for a key past the end)
#pragma unroll
  for (int kb = 0; kb < KB; ++kb) {
    const int kj = k_first + 32 * kb + lr, kc = min(kj, a.Nk - 1);
    q_lo[kb] = kj >= a.Nk ? 0x7fffffff : CAUSAL ? kj - coff : 0;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
      kf[kb][ks] = *reinterpret_cast<const i32x4 *>(kc_bh + (int64_t)kc * a.skn + ks * 32 + g * 16);
#pragma unroll
    for (int kd = 0; kd < KD; ++kd)
      vf[kb][kd] = *reinterpret_cast<const u32x4 *>(v_bh + (int64_t)kc * a.svn + kd * 16 + g * 8);
    const unsigned *ck = reinterpret_cast<const unsigned *>(wsk_bh + (int64_t)(kc / TILE) * WS::K_BLOB + WS::T_BYTES);
    const int kl = kc % TILE;
    corr_k[kb] = u32x2{ck[2 * kl + g], g ? 0u : QFA_BIAS_B(T)};
    sk[kb] = __builtin_bit_cast(float, ck[2 * TILE + kl]);
  }

  // ---- per-lane read offsets: rows (lane = row lr, k-group g), transposing reads (rows 4g + {0..3} of slabs u; those + 8
  // with the halves swapped)
  const int row_l = slab_row(lr, g);
  const int s16 = lane % 16, u16 = (lane / 16) % 2;
  const int tr_l = u16 * SLAB + (4 * g + s16 / 4) * 32 + ((s16 % 4) / 2) * 16 + (s16 % 2) * 8;
  const unsigned lds0 = lds_addr(smem);

  // accumulators: dK^T of (key block kb, columns 32db) in tile kb * DB + db, dV^T behind them
  constexpr int DV0 = KB * DB, ACC = 2 * KB * DB;
  acc_zero<ACC>();

  f32x16 f[KB];            // scores of the step in work (biased integers without the zero-point term), later its P
  i32x16 bias;
#pragma unroll
  for (int v = 0; v < 16; ++v) bias[v] = QFA_BIAS_BITS;
  u32x4 pf[KB][2], ds[KB][2];
#pragma unroll
  for (int kb = 0; kb < KB; ++kb)
#pragma unroll
    for (int hh = 0; hh < 2; ++hh) ds[kb][hh] = u32x4{0u, 0u, 0u, 0u};

  auto ld = [&](int off) -> u32x4 { return *reinterpret_cast<const u32x4 *>(smem + off); };
  auto ldf = [&](int off) -> f32x4 { return *reinterpret_cast<const f32x4 *>(smem + off); };
  auto cq_a = [&](int buf, int mbk) { return buf + SM::OFF_C + 2 * TILE * 4 + 16 * g + mbk * 128; };   // a; then -lse*log2e, -delta

  // What a step finds in registers, requested at the end of the previous one: the first fragments of Qz^T of the previous
  // step, the correction operand, and the constants of the first query rows
  constexpr int RING = 4;   // fragments requested three slots ahead
  u32x4 fr[RING];
  u32x2 corr_q = {0u, QFA_BIAS_A(T)};
  f32x4 ca[2], cn[2];   // a and -lse*log2e of query rows 8aa + 4g + {0..3}: aa % 2
  auto request_head = [&](int buf, int mbk, int qt_prev) __attribute__((always_inline)) {
#pragma unroll
    for (int n = 0; n < RING - 1; ++n) fr[n] = ld(qt_prev + n * 1024);
    corr_q[0] = *reinterpret_cast<const unsigned *>(smem + buf + SM::OFF_C + (2 * lr + g) * 4 + mbk * 256);
    ca[0] = ldf(cq_a(buf, mbk));
    cn[0] = ldf(cq_a(buf, mbk) + TILE * 4);
  };

  // One step: 32 queries (part mbk of the tile in buffer `buf`) against the wave's keys.  `nbuf`: buffer of the next step.
  auto body = [&](int t, int buf, int nbuf, int qt_prev, auto mbk_tag, auto masked_tag) __attribute__((always_inline)) {
    constexpr bool MASKED = decltype(masked_tag)::value;
    constexpr int mbk = decltype(mbk_tag)::value;
    constexpr bool LAST = mbk == NSTEP - 1;
    const int rowb = buf + row_l + mbk * 1024;
    const int cb = cq_a(buf, mbk);
    const int i0 = TILE * t + 32 * mbk + 4 * g;
    // dO^T is zero for the key blocks that none of the step's queries sees (a wave's first step may hold such blocks): P is
    // zero there, and dO may be infinite
    constexpr bool UNSEEN = MASKED && CAUSAL && KB > 1;
    unsigned dv_mask[KB];
#pragma unroll
    for (int kb = 0; kb < KB; ++kb) dv_mask[kb] = TILE * t + 32 * mbk + 31 >= k_first + 32 * kb - coff ? ~0u : 0u;

    // ---- the vector work of P, in 16 KB half items dealt to the MFMA slots: scaling of a pair of scores and packing of the
    // pair before it (even), exponentials (odd).  Pairs in an order that lets two quads' constants serve all key blocks:
    // quad aa = 0, 1 of every key block, then aa = 2, 3
    constexpr int HALF = 16 * KB;
    float x0, x1;
    auto pack_pair = [&](auto x_tag) __attribute__((always_inline)) {
      constexpr int x = decltype(x_tag)::value, kb = x / 4 % KB, aa = 2 * (x / (4 * KB)) + x / 2 % 2;
      pf[kb][aa / 2][2 * (aa % 2) + x % 2] = pack2<T>(x0, x1);
    };
    auto half_item = [&](auto i_tag) __attribute__((always_inline)) {
      constexpr int i = decltype(i_tag)::value, x = i / 2, kb = x / 4 % KB, aa = 2 * (x / (4 * KB)) + x / 2 % 2, v = 4 * aa + 2 * (x % 2);
      if constexpr (i % 2 == 0) {
        if constexpr (x > 0) pack_pair(ic<x - 1>{});
        x0 = __builtin_fmaf(ca[aa % 2][2 * (x % 2)], f[kb][v] * sk[kb], cn[aa % 2][2 * (x % 2)]);
        x1 = __builtin_fmaf(ca[aa % 2][2 * (x % 2) + 1], f[kb][v + 1] * sk[kb], cn[aa % 2][2 * (x % 2) + 1]);
      } else {
        x0 = __builtin_amdgcn_exp2f(x0);
        x1 = __builtin_amdgcn_exp2f(x1);
        if constexpr (MASKED) {   // (no short circuit: a branch per element would end the block)
          const int q = i0 + 8 * aa + 2 * (x % 2);
          x0 = ((q >= q_lo[kb]) & (q < Nq)) ? x0 : 0.f;
          x1 = ((q + 1 >= q_lo[kb]) & (q + 1 < Nq)) ? x1 : 0.f;
        }
        f[kb][v] = x0;
        f[kb][v + 1] = x1;
      }
      // the constants of quad aa + 2 replace those of aa behind their last use
      constexpr int last0 = KB == 2 ? 10 : 2, last1 = KB == 2 ? 14 : 6;
      if constexpr (i == last0 + 1) { ca[0] = ldf(cb + 64); cn[0] = ldf(cb + TILE * 4 + 64); }
      if constexpr (i == last1 + 1) { ca[1] = ldf(cb + 96); cn[1] = ldf(cb + TILE * 4 + 96); }
    };
    constexpr int NX = 2 * DB, NP = KD, SLOTS = KB * (NX + NP);   // fragments of dK, of dP; MFMA slots of both
    auto work = [&](auto slot_tag) __attribute__((always_inline)) {   // slot s: the items that fall to it, two slots late
      constexpr int s = decltype(slot_tag)::value - 2;
      if constexpr (s >= 0) {
        constexpr int i0_ = s * HALF / SLOTS, i1_ = (s + 1) * HALF / SLOTS;
        static_for<i1_ - i0_>([&](auto k) __attribute__((always_inline)) { half_item(ic<i0_ + decltype(k)::value>{}); });
      }
    };

    // Turn of the tile: the next one has landed, the one after it goes into the buffer of the previous one, whose last fragments
    // have been requested.  With one step per tile (head_dim 256) the last pieces of a copy have little time until the next turn.
    // Without a mask the turn comes before the first request of dO there, and only the codes and constants of the next tile have to be
    // there, dO and Qz^T one turn later (the whole backward, 64 heads of 4096: 2976 -> 2949 us; with a mask, where waves begin at
    // different tiles: 1726 -> 1734)
    TileDesc td;
    auto turn = [&]() __attribute__((always_inline)) {
      vm_wait<PIECES - FIRST>();
      lds_barrier();
      td = tile_desc(t + 2);
    };
    constexpr int TURN = EARLY ? NX - RING + 1 : NX;   // in front of this fragment's products
    // ---------------- dK of the previous step (Qz^T . dS) under the first part of P
#pragma unroll
    for (int kb = 0; kb < KB; ++kb) f[kb] = mfma_16b_k8<T>(corr_q, corr_k[kb], f[kb]);
    f32x4 nd4[4];
    static_for<NX>([&](auto n_tag) __attribute__((always_inline)) {     // hh = n / DB, db = n % DB
      constexpr int n = decltype(n_tag)::value;
      if constexpr (LAST && n == TURN) turn();
      static_for<KB>([&](auto kb_tag) __attribute__((always_inline)) {
        constexpr int kb = decltype(kb_tag)::value;
        QFA_FENCE();
        acc_mfma<T, kb * DB + n % DB, ACC>(fr[n % RING], ds[kb][n / DB]);
        QFA_FENCE();
        work(ic<KB * n + kb>{});
        if constexpr (kb == 0) {
          if constexpr (n + RING - 1 < NX) fr[(n + RING - 1) % RING] = ld(qt_prev + (n + RING - 1) * 1024);
          else fr[(n + RING - 1) % RING] = ld(rowb + SM::OFF_DO + (n + RING - 1 - NX) * SLAB);
          if constexpr (n == 0) { ca[1] = ldf(cb + 32); cn[1] = ldf(cb + TILE * 4 + 32); }
        }
        if constexpr (kb == KB - 1 && n >= NX - 4) nd4[n - (NX - 4)] = ldf(cb + 2 * TILE * 4 + (n - (NX - 4)) * 32);
      });
    });
    if constexpr (LAST && TURN == NX) turn();
    constexpr int CSLOTS = KB * (NP + 2 * DB);   // the copy's pieces are spread over the slots that are left
    auto copy_slot = [&](auto s_tag) __attribute__((always_inline)) {
      constexpr int s = decltype(s_tag)::value, p0 = s * PIECES / CSLOTS, p1 = (s + 1) * PIECES / CSLOTS;
      if constexpr (LAST) static_for<p1 - p0>([&](auto p) __attribute__((always_inline)) { copy_piece(td, p0 + decltype(p)::value); });
    };
    // ---------------- dP - delta under the second part of P
    f32x16 dp[KB], nd;
#pragma unroll
    for (int v = 0; v < 16; ++v) nd[v] = nd4[v / 4][v % 4];
    const int nrow = nbuf + row_l + (LAST ? 0 : (mbk + 1) * 1024) + SM::OFF_Q;
    u32x4 qa[KS];
    static_for<NP>([&](auto n_tag) __attribute__((always_inline)) {
      constexpr int n = decltype(n_tag)::value;
      static_for<KB>([&](auto kb_tag) __attribute__((always_inline)) {
        constexpr int kb = decltype(kb_tag)::value;
        QFA_FENCE();
        dp[kb] = mfma_16b<T>(fr[(NX + n) % RING], vf[kb][n], n == 0 ? nd : dp[kb]);
        QFA_FENCE();
        work(ic<KB * (NX + n) + kb>{});
        if constexpr (kb == 0 && n + RING - 1 < NP) fr[(NX + n + RING - 1) % RING] = ld(rowb + SM::OFF_DO + (n + RING - 1) * SLAB);
        copy_slot(ic<KB * n + kb>{});
      });
    });
    // ---------------- dV (dO^T . P) and, in between, S of the next step, under the last of P, dS and the conversion of S
    const unsigned trb = lds0 + buf + SM::OFF_DO + tr_l + mbk * 1024, trb1 = trb ^ 16u;
    u32x2 tr[3][2];
    auto tr_read = [&](auto n_tag) __attribute__((always_inline)) {   // hh = n / DB, db = n % DB
      constexpr int n = decltype(n_tag)::value, off = 2 * (n % DB) * SLAB + 16 * (n / DB) * 32;
      tr[n % 3][0] = lds_read_tr16_async<off>(trb);
      tr[n % 3][1] = lds_read_tr16_async<off + 256>(trb1);
    };
    i32x16 si[KB];
    constexpr int DSW = 8 * KB;   // dwords of dS
    auto ds_dword = [&](auto k_tag) __attribute__((always_inline)) {
      constexpr int k = decltype(k_tag)::value, kb = k / 8, hh = k / 4 % 2, e = k % 4, v = 8 * hh + 2 * e;
      // (a masked pair has P = 0, but its dP may be anything: dO may be infinite there)
      const float x0 = MASKED ? mul_zero_wins(f[kb][v], dp[kb][v]) : f[kb][v] * dp[kb][v];
      const float x1 = MASKED ? mul_zero_wins(f[kb][v + 1], dp[kb][v + 1]) : f[kb][v + 1] * dp[kb][v + 1];
      ds[kb][hh][e] = pack2<T>(x0, x1);
    };
    // S comes before the last dV fragment, whose MFMAs cover the time its results take
    constexpr int NV = 2 * DB, V1 = NV - 1;
    constexpr int S1 = KB * V1;   // slots before S
    tr_read(ic<0>{});
    tr_read(ic<1>{});
    auto dv_slot = [&](auto n_tag) __attribute__((always_inline)) {
      constexpr int n = decltype(n_tag)::value;
      if constexpr (n + 2 < NV) tr_read(ic<n + 2>{});
      u32x2(&w)[2] = tr[n % 3];
      if constexpr (n + 2 < NV) lds_wait_for<4>(w);
      else if constexpr (n + 1 < NV) lds_wait_for<2>(w);
      else lds_wait_for<0>(w);
      u32x4 g4 = {w[0][0], w[0][1], w[1][0], w[1][1]};
      static_for<KB>([&](auto kb_tag) __attribute__((always_inline)) {
        constexpr int kb = decltype(kb_tag)::value, m = KB * n + kb;
        if constexpr (UNSEEN && kb == 0 && mbk == 0) {   // (a tile's second step sees it)
          g4 &= dv_mask[0];
          QFA_FENCE();
          asm volatile("s_nop 1");
        }
        // (at head_dim 64 the last pair of P is packed in the slot before the first product that reads it)
        if constexpr (m == 2 && n / DB == 1 && !UNSEEN) asm volatile("s_nop 1");
        QFA_FENCE();
        acc_mfma<T, DV0 + kb * DB + n % DB, ACC>(g4, pf[kb][n / DB]);
        QFA_FENCE();
        if constexpr (UNSEEN && kb == 0) {   // (fewer queries see the second block)
          g4 &= dv_mask[KB - 1];
          QFA_FENCE();
          if constexpr (m >= S1) asm volatile("s_nop 1");
        }
        if constexpr (m < S1) {
          if constexpr (m < 2) work(ic<SLOTS + m>{});
          if constexpr (m == 1) pack_pair(ic<8 * KB - 1>{});
          constexpr int k0 = m <= 1 ? 0 : DSW * (m - 2) / (S1 - 2), k1 = m <= 1 ? 0 : DSW * (m - 1) / (S1 - 2);
          static_for<k1 - k0>([&](auto k) __attribute__((always_inline)) { ds_dword(ic<k0 + decltype(k)::value>{}); });
        }
        copy_slot(ic<KB * NP + m>{});
        if constexpr (m < S1) {   // the codes of S, late in this part
          constexpr int Q1 = S1 > KS ? S1 - KS : 0, y = m - Q1, k0 = y < 0 ? 0 : KS * y / (S1 - Q1), k1 = y < 0 ? 0 : KS * (y + 1) / (S1 - Q1);
          static_for<k1 - k0>([&](auto k) __attribute__((always_inline)) {
            qa[k0 + decltype(k)::value] = ld(nrow + (k0 + decltype(k)::value) * SLAB);
          });
        }
      });
    };
    static_for<V1>([&](auto n) __attribute__((always_inline)) { dv_slot(n); });
#pragma unroll
    for (int kb = 0; kb < KB; ++kb)
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        QFA_FENCE();
        si[kb] = mfma_i8(__builtin_bit_cast(i32x4, qa[ks]), kf[kb][ks], ks == 0 ? bias : si[kb]);
      }
    const int qt = buf + SM::OFF_QT + row_l + mbk * (2 * DB * 1024);
    static_for<NV - V1>([&](auto n) __attribute__((always_inline)) { dv_slot(ic<V1 + decltype(n)::value>{}); });
    QFA_FENCE();
    request_head(nbuf, LAST ? 0 : mbk + 1, qt);
#pragma unroll
    for (int kb = 0; kb < KB; ++kb) f[kb] = __builtin_bit_cast(f32x16, si[kb]);
    QFA_FENCE();
  };

  // ---- first tile this wave sees; with one key block per wave it begins with the first step that the wave sees, so that
  // every block of a step is seen by some query (with two the second block's masks do that)
  int ft = it0;
  const bool late = CAUSAL && KB == 1 && NSTEP == 2 && max(k_first - coff, 0) / 32 % 2 == 1;
  if (CAUSAL) ft = max(ft, max(k_first - coff, 0) / TILE);
  if (k_first >= a.Nk) ft = ntiles;
  ft = min(ft, ntiles);   // (a part of the queries may hold none that sees the wave's keys)
  dma_wait();
  __syncthreads();
  int t = it0;
  for (; t < ft; ++t) {
    dma_wait();
    lds_barrier();
    copy_tile(t + 2);
  }
  if (t < ntiles) {
    int buf = (t - it0) % 3 * SM::BUF, nbuf = (t + 1 - it0) % 3 * SM::BUF;
#pragma unroll
    for (int kb = 0; kb < KB; ++kb) {
      i32x16 si = bias;
#pragma unroll
      for (int ks = 0; ks < KS; ++ks)
        si = mfma_i8(__builtin_bit_cast(i32x4, ld(buf + row_l + (late ? 1024 : 0) + SM::OFF_Q + ks * SLAB)), kf[kb][ks], si);
      f[kb] = __builtin_bit_cast(f32x16, si);
    }
    int qt_prev = buf + SM::OFF_QT + row_l;     // (dS is zero: the product adds nothing)
    request_head(buf, late ? 1 : 0, qt_prev);
    const int k_last = k_first + KEYS - 1;
    // masked tiles (diagonal), full ones, masked ones (ragged end)
    auto tiles = [&](int t_end, auto masked_tag) __attribute__((always_inline)) {
      for (; t < t_end; ++t) {
        static_for<NSTEP>([&](auto mbk_tag) __attribute__((always_inline)) {
          constexpr int mbk = decltype(mbk_tag)::value;
          if constexpr (decltype(masked_tag)::value && CAUSAL && KB == 1 && NSTEP == 2 && mbk == 0) {
            if (late && t == ft) return;
          }
          body(t, buf, mbk == NSTEP - 1 ? nbuf : buf, qt_prev, mbk_tag, masked_tag);
          qt_prev = buf + SM::OFF_QT + row_l + mbk * (2 * DB * 1024);
        });
        const int b2 = 3 * SM::BUF - buf - nbuf;
        buf = nbuf;
        nbuf = b2;
      }
    };
    const int full0 = k_last >= a.Nk ? ntiles : CAUSAL ? max(k_last - coff + TILE - 1, 0) / TILE : 0;
    tiles(min(full0, ntiles), std::true_type{});
    tiles(Nq / TILE, std::false_type{});
    tiles(ntiles, std::true_type{});
    static_for<2 * DB>([&](auto n_tag) __attribute__((always_inline)) {
      constexpr int n = decltype(n_tag)::value;
      const u32x4 tq = ld(qt_prev + n * 1024);
      static_for<KB>([&](auto kb) __attribute__((always_inline)) { acc_mfma<T, decltype(kb)::value * DB + n % DB, ACC>(tq, ds[kb][n / DB]); });
    });
  }
  // what only the epilogue needs is read and formed here: held in scalar registers through the loop it would push others out,
  // and behind the barrier its latency would be seen
  typedef __attribute__((address_space(4))) const BwdArgs KernArgs;
  KernArgs *ep = (KernArgs *)__builtin_amdgcn_kernarg_segment_ptr();
  int bh_ = bh;
  asm volatile("" : "+s"(ep), "+s"(bh_));
  const int64_t eb = index_div(bh_, ep->H), eh = bh_ - eb * ep->H;
  void *dk = ep->dk, *dv = ep->dv;
  int64_t dk_at = eb * ep->sdkb + eh * ep->sdkh + blockIdx.y * ep->split_stride,
          dv_at = eb * ep->sdvb + eh * ep->sdvh + blockIdx.y * ep->split_stride, sdkn = ep->sdkn, sdvn = ep->sdvn;
  float sm = ep->sm_scale;
  int f32 = ep->grad_f32;
  asm volatile("" : "+s"(dk), "+s"(dv), "+s"(dk_at), "+s"(dv_at), "+s"(sdkn), "+s"(sdvn), "+s"(sm), "+s"(f32));
  acc_settle();
  __syncthreads();   // the tile buffers are done with: the output stages overlay them
  static_assert(4 * 32 * 2 * D <= 3 * SM::BUF, "output staging fits the tile buffers");
  unsigned char *stage = smem + wave * (32 * 2 * D);
  if (f32) {
    float *dk_bh = reinterpret_cast<float *>(dk) + dk_at, *dv_bh = reinterpret_cast<float *>(dv) + dv_at;
    static_for<KB>([&](auto kb_tag) __attribute__((always_inline)) {
      constexpr int kb = decltype(kb_tag)::value;
      acc_store_rows_f32<D, kb * DB>(sm, dk_bh, sdkn, k_first + 32 * kb, a.Nk, lane);
      acc_store_rows_f32<D, DV0 + kb * DB>(1.0f, dv_bh, sdvn, k_first + 32 * kb, a.Nk, lane);
    });
    return;
  }
  T *dk_bh = reinterpret_cast<T *>(dk) + dk_at, *dv_bh = reinterpret_cast<T *>(dv) + dv_at;
  static_for<KB>([&](auto kb_tag) __attribute__((always_inline)) {
    constexpr int kb = decltype(kb_tag)::value;
    acc_store_rows<T, D, kb * DB>(sm, stage, dk_bh, sdkn, k_first + 32 * kb, a.Nk, lane);
    acc_store_rows<T, D, DV0 + kb * DB>(1.0f, stage, dv_bh, sdvn, k_first + 32 * kb, a.Nk, lane);
  });
#endif
}

template <typename T, int D, int KB> static int launch_dkv_kb(BwdArgs a, int64_t BH, bool causal, int splits, hipStream_t st) {
  a.nblocks = (a.Nk + 128 * KB - 1) / (128 * KB);
  a.group_log2 = bwd_group_log2(a.Nq, D, false);   // per head the kernel streams Qc, dO and Qz^T: 5 bytes per query and d
  const int64_t total = (int64_t)a.nblocks * BH;
  if (total > 0x3fffffffLL) return set_error(QFA_EUNSUPPORTED, "attn_bwd: too many key blocks for one launch");
  a.total_blocks = (int)total;
  a.blocks_per_xcd = (a.total_blocks + 7) / 8;
  const dim3 grid((unsigned)(a.blocks_per_xcd * 8), (unsigned)splits);
  if (causal) bwd_dkv_kernel<T, D, KB, true><<<grid, dim3(256), 0, st>>>(a);
  else bwd_dkv_kernel<T, D, KB, false><<<grid, dim3(256), 0, st>>>(a);
  return check_launch("qfa_attn_bwd (dk, dv)");
}

template <typename T, int D> int launch_dkv(BwdArgs a, int64_t BH, bool causal, int blocks, int splits, hipStream_t st) {
  if constexpr (D == 128) {
    if (blocks == 2) return launch_dkv_kb<T, D, 2>(a, BH, causal, splits, st);
  }
  // (head_dim 256: the registers hold the operands and accumulators of 32 keys; head_dim 64: of 32 keys in two waves per
  // SIMD, which share the issue slots better than one wave of 64 keys: 3 - 10 % faster, 20 % when the chip is not full)
  return launch_dkv_kb<T, D, 1>(a, BH, causal, splits, st);
}
template int launch_dkv<__bf16, 64>(BwdArgs, int64_t, bool, int, int, hipStream_t);
template int launch_dkv<__bf16, 128>(BwdArgs, int64_t, bool, int, int, hipStream_t);
template int launch_dkv<__bf16, 256>(BwdArgs, int64_t, bool, int, int, hipStream_t);
template int launch_dkv<_Float16, 64>(BwdArgs, int64_t, bool, int, int, hipStream_t);
template int launch_dkv<_Float16, 128>(BwdArgs, int64_t, bool, int, int, hipStream_t);
template int launch_dkv<_Float16, 256>(BwdArgs, int64_t, bool, int, int, hipStream_t);

}  // namespace qfa
