// Backward of the shared-KV attention for query blocks that the fused one-pass kernel (qfa_skv_bwd.hip) does not take, as a dQ
// kernel and a dKV kernel.  Same mathematics (quant_flash_attn.py:104-166):
//     P = exp(sm_scale * Q KV^T - LSE),   dP = dO KV^T,   dS = sm_scale * P o (dP - delta),
//     dQ = dS KV,   dKV = P^T dO + dS^T Q,   delta = rowsum(O o dO)
//
// dQ    skv_dq_kernel here where there is little to do: one workgroup per block of 16 queries, built like the forward of
//       qfa_skv.hip (the 32-key tiles are dealt to the four waves, streamed through private LDS rings, S^T and dP^T share the
//       expanded code operands, dS * scale_j is the operand of dQ^T += C^T (dS*scale)^T, the four partial dQ are summed at the
//       end).  Its tiles start at once; with more work skv_tile_dq_kernel (qfa_skv_tile.hip) takes over (skv_tile_dq_plan).
// dKV   skv_dkv_kernel (qfa_skv_dkv.hip) up to head_dim 128.  At 256 the accumulators of a tile do not fit one of two waves per
//       SIMD: in skv_dkv256_kernel two waves share a tile of 32 keys, each keeping 128 of the 256 columns (both compute S and
//       dP), a workgroup covers 64 keys and walks over the query blocks of 32, whose Q / dO rows arrive in LDS by direct loads.
//       (skv_dkv_kernel with one wave per SIMD takes 1.25 instead of 1.07 ms for the backward of 1584 heads, 97 queries, 689
//       keys.)
// All of them compute delta from O and dO; S and dP are computed for dQ and for dKV.
#include <type_traits>

#include "qfa_host.h"
#include "qfa_skv_common.h"

namespace qfa {

struct SkvBwdLongArgs {
  const _Float16 *q, *o, *dout;
  const int8_t *codes; const void *scale; const int8_t *zp;
  const float *lse;
  _Float16 *dq, *dkv;          // 16-bit outputs: binary16, or bfloat16 when grad_bf16 is set
  const float *grad_scale;     // nullable device scalar: dq and dkv are multiplied by it before rounding
  int grad_bf16;
  int direct, q_bf16, do_bf16;   // dQ, up to head_dim 128: q, o and dO as the caller has them, dO scaled here (no grad_scale)
  int64_t H;
  int Nq, Nk, BH, qblocks, kchunks, cpw;   // cpw: key chunks per workgroup of the dKV kernel
  int64_t sqb, sqh, sqn, scb, sch, scn, sob, soh, son, sdob, sdoh, sdon, sdqb, sdqh, sdqn, sdkb, sdkh, sdkn;
  float sm_scale, sm_scale_log2;
};

// ------------------------------------------------------------------------------------------ dQ

template <typename S, int D> __global__ __launch_bounds__(256, 2) void skv_dq_kernel(SkvBwdLongArgs a) {
  typedef SwzSkv<D> KSW;
  typedef TileCopy<D, SKV_TILE, 64, KSW> Copy;
  constexpr int KS = D / 32, DB = D / 16, OPS = Copy::N + 2;
  constexpr int SKVQ_NBUF = D == 256 ? 2 : 3;   // ring depth per wave (8 KB tiles at D = 256)
  constexpr int K_BYTES = SKV_TILE * D, SLOT = K_BYTES + 2 * SKV_TILE * 4, WAVE = SKVQ_NBUF * SLOT;
  constexpr int MG = 16 * D;   // floats of one partial dQ^T [D][16]
  static_assert(3 * MG * 4 <= 4 * WAVE, "the merge area overlays the rings");
  // (One array: with the maxima of a direct call in a second one, the compiler waits for all LDS loads in
  // front of a tile's scales: 48 heads, 33 x 12000, 82 us against 75.)
  __shared__ __attribute__((aligned(16))) unsigned char smem[4 * WAVE + (D <= 128 ? 48 : 0)];

  const XcdBlock id(a.BH, a.qblocks);
  if (!id.live) return;
  const int bh = id.bh, qb = id.sub;
  const int64_t b = index_div(bh, a.H), h = bh - b * a.H;
  const int tid = threadIdx.x, lane = tid % 64, q16 = lane % 16, G = lane / 16;
  const int wave = __builtin_amdgcn_readfirstlane(tid / 64);
  const int wave_off = wave * WAVE;

  const unsigned char *codes_bh = reinterpret_cast<const unsigned char *>(a.codes + b * a.scb + h * a.sch);
  const int64_t tk0 = (int64_t)bh * a.Nk, tq0 = (int64_t)bh * a.Nq;
  const int ntiles = (a.Nk + SKV_TILE - 1) / SKV_TILE;
  const int my_tiles = ntiles > wave ? (ntiles - wave + 3) / 4 : 0;

  Copy cp;
  cp.init((unsigned)a.scn, lane);
  auto issue = [&](int i, int slot_idx) {
    skv_issue_tile<S, D>(cp, smem + wave_off + slot_idx * SLOT, codes_bh, a.scale, a.zp, tk0, wave + 4 * i, a.Nk, a.scn, lane);
  };
  auto scale_of = [](unsigned w) -> float {
    return scale_to_f32<S>(w);
  };
  float osc = a.grad_scale ? *a.grad_scale : 1.0f;
  auto pack_out = [&](float x, float y) -> unsigned {
    return a.grad_bf16 ? pack2<__bf16>(x * osc, y * osc) : pack2<_Float16>(x * osc, y * osc);
  };
#pragma unroll
  for (int i = 0; i < SKVQ_NBUF - 1; ++i)
    if (i < my_tiles) issue(i, i);

  // ---- this lane's query and dO row as B operands (k-step m, k-group G: d = 64(m/2) + 16G + 8(m%2) + {0..7}),
  //      their sums, delta and LSE
  const int qi = 16 * qb + q16;
  const bool q_ok = qi < a.Nq;
  const int qi_c = q_ok ? qi : a.Nq - 1;
  const _Float16 *qrow = a.q + b * a.sqb + h * a.sqh + (int64_t)qi_c * a.sqn;
  const _Float16 *orow = a.o + b * a.sob + h * a.soh + (int64_t)qi_c * a.son;
  const _Float16 *drow = a.dout + b * a.sdob + h * a.sdoh + (int64_t)qi_c * a.sdon;
  u32x4 qf[KS], dof[KS], of[KS];
  const KeyScaleMax scales(a.scale, sizeof(S) == 4 ? QFA_F32 : QFA_F16, tk0, a.direct ? a.Nk : 1, tid);
  float rq = 0.f, rd = 0.f, delta = 0.f;
#pragma unroll
  for (int m = 0; m < KS; ++m) {
    const int d0 = 64 * (m / 2) + 16 * G + 8 * (m % 2);
    qf[m] = *reinterpret_cast<const u32x4 *>(qrow + d0);
    dof[m] = *reinterpret_cast<const u32x4 *>(drow + d0);
    of[m] = *reinterpret_cast<const u32x4 *>(orow + d0);
  }
  if (D <= 128 && a.direct) {   // a power of two of the workgroup's own queries and of all its head's keys, which bound delta
    const int k = block_dout_exponent(max_abs_dout(dof, a.do_bf16), scales.get(), 0.f, reinterpret_cast<float *>(smem + 4 * WAVE));
    osc = exp2_neg(k);
    scale_dout(dof, a.do_bf16, k);
    if (a.q_bf16) {
#pragma unroll
      for (int m = 0; m < KS; ++m) qf[m] = half_of_bf16(qf[m]), of[m] = half_of_bf16(of[m]);
    }
  }
#pragma unroll
  for (int m = 0; m < KS; ++m) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const unsigned qw = qf[m][e], dw = dof[m][e], ow = of[m][e];
      const float d0f = lo_to_f32<_Float16>(dw), d1f = hi_to_f32<_Float16>(dw);
      rq += lo_to_f32<_Float16>(qw) + hi_to_f32<_Float16>(qw);
      rd += d0f + d1f;
      delta += lo_to_f32<_Float16>(ow) * d0f + hi_to_f32<_Float16>(ow) * d1f;
    }
  }
#pragma unroll
  for (int m = 16; m < 64; m *= 2) {
    rq += __shfl_xor(rq, m, 64);
    rd += __shfl_xor(rd, m, 64);
    delta += __shfl_xor(delta, m, 64);
  }
  const bool big = offset_needs_x32(fmaxf(fabsf(rq), fabsf(rd)));
  u32x4 corr_q = {0u, 0u, 0u, 0u}, corr_do = {0u, 0u, 0u, 0u};
  if (G == 0) {
    const u32x2 cq2 = offset_query_operand(rq, big), cd2 = offset_query_operand(rd, big);
    corr_q[0] = cq2[0];
    corr_q[1] = cq2[1];
    corr_do[0] = cd2[0];
    corr_do[1] = cd2[1];
  }
  const float a_s = a.sm_scale_log2;
  const float nlse2 = q_ok ? -a.lse[tq0 + qi] * kLog2e : -INFINITY;   // padding rows: p = 0

  int k_off[2];
#pragma unroll
  for (int rb = 0; rb < 2; ++rb) k_off[rb] = (16 * rb + q16) * D + ((G ^ KSW::swz(16 * rb + q16)) << 4);
  int vt_off;
  {
    const int s = lane % 16, j = s / 2;
    const int key = 16 * (j / 4) + 4 * G + j % 4;
    vt_off = key * D + (KSW::swz(key) << 4) + 8 * (s % 2);
  }
  const unsigned lds0 = lds_addr(smem);

  f32x4 acc[DB];
#pragma unroll
  for (int db = 0; db < DB; ++db) acc[db] = f32x4{0.f, 0.f, 0.f, 0.f};
  float w_run = 0.f;

  auto tile = [&](int i, int slot_idx) {
    const int slot_off = wave_off + slot_idx * SLOT;
    const unsigned char *slot = smem + slot_off;
    const unsigned *skp = reinterpret_cast<const unsigned *>(slot + K_BYTES);
    const unsigned *zpp = skp + SKV_TILE;
    const int krem = a.Nk - (wave + 4 * i) * SKV_TILE;   // keys of this tile that exist (>= 32: all)
    const unsigned z_a[2] = {zpp[q16], zpp[16 + q16]};
    // (per-block read addresses are re-formed from these every tile: one XOR each instead of registers
    // held across the loop)
    int vt = vt_off, ko[2] = {k_off[0], k_off[1]};
    asm volatile("" : "+v"(vt), "+v"(ko[0]), "+v"(ko[1]));
    constexpr int VG = DB < 8 ? DB : 8;   // transposed fragments in groups of 8 blocks, the first one now
    u32x2 vr[VG];
#pragma unroll
    for (int db = 0; db < VG; ++db) vr[db] = lds_read_tr8_async(lds0 + slot_off + (vt ^ (db << 4)));
    // ---- S^T and dP^T from the same expanded code operands
    f32x4 f[2], gq[2];
#pragma unroll
    for (int rb = 0; rb < 2; ++rb) {
      f[rb] = f32x4{0.f, 0.f, 0.f, 0.f};
      gq[rb] = f32x4{0.f, 0.f, 0.f, 0.f};
      u32x4 kw[(KS + 1) / 2];
#pragma unroll
      for (int mm = 0; mm < (KS + 1) / 2; ++mm)
        kw[mm] = *reinterpret_cast<const u32x4 *>(slot + (ko[rb] ^ ((4 * mm) << 4)));
#pragma unroll
      for (int m = 0; m < KS; ++m) {
        const u32x4 ca = expand_codes(kw[m / 2][2 * (m % 2)], kw[m / 2][2 * (m % 2) + 1]);
        f[rb] = mfma_h16(ca, qf[m], f[rb]);
        gq[rb] = mfma_h16(ca, dof[m], gq[rb]);
      }
      u32x4 corr_k = {0u, 0u, 0u, 0u};
      if (G == 0) {
        const u32x2 ck2 = offset_key_operand(z_a[rb], big);
        corr_k[0] = ck2[0];
        corr_k[1] = ck2[1];
      }
      f[rb] = mfma_h16(corr_k, corr_q, f[rb]);
      gq[rb] = mfma_h16(corr_k, corr_do, gq[rb]);
    }
    // ---- p, ds, x = ds * scale_j as binary16 (keys 16rb + 4G + v), offset term
    u32x4 xf;
#pragma unroll
    for (int rb = 0; rb < 2; ++rb) {
      const u32x4 sk4 = *reinterpret_cast<const u32x4 *>(skp + 16 * rb + 4 * G);
      const u32x4 zk4 = *reinterpret_cast<const u32x4 *>(zpp + 16 * rb + 4 * G);
      float x[4];
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const float sk = scale_of(sk4[v]);
        float p = __builtin_amdgcn_exp2f(__builtin_fmaf(a_s * sk, f[rb][v], nlse2));
        if (16 * rb + 4 * G + v >= krem) p = 0.f;
        x[v] = a.sm_scale * p * (gq[rb][v] * sk - delta) * sk;
      }
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        const unsigned xx = pack_h2(x[2 * e], x[2 * e + 1]);
        xf[2 * rb + e] = xx;
        const unsigned cpair = magic_zp_pair(zk4[2 * e], zk4[2 * e + 1]);
        w_run = __builtin_amdgcn_fdot2(__builtin_bit_cast(f16x2, xx), __builtin_bit_cast(f16x2, cpair), w_run, false);
      }
    }
    // ---- dQ^T += (1152 + codes)^T . x^T
#pragma unroll
    for (int g0 = 0; g0 < DB; g0 += VG) {
      lds_wait_all();
      u32x2 now[VG];
#pragma unroll
      for (int db = 0; db < VG; ++db) now[db] = tie(vr[db]);
      if (g0 + VG < DB) {
#pragma unroll
        for (int db = 0; db < VG; ++db) vr[db] = lds_read_tr8_async(lds0 + slot_off + (vt ^ ((g0 + VG + db) << 4)));
      }
#pragma unroll
      for (int db = 0; db < VG; ++db) acc[g0 + db] = mfma_h16(expand_codes(now[db][0], now[db][1]), xf, acc[g0 + db]);
    }
  };

  int cur = 0, nxt = SKVQ_NBUF - 1;
  for (int i = 0; i < my_tiles; ++i) {
    if (i + SKVQ_NBUF - 1 < my_tiles) {
      issue(i + SKVQ_NBUF - 1, nxt);
      asm volatile("s_waitcnt vmcnt(%0)" ::"n"((SKVQ_NBUF - 1) * OPS) : "memory");
    } else {
      dma_wait();
    }
    tile(i, cur);
    cur = cur + 1 == SKVQ_NBUF ? 0 : cur + 1;
    nxt = nxt + 1 == SKVQ_NBUF ? 0 : nxt + 1;
  }

  float w_tot = w_run + __shfl_xor(w_run, 16, 64);
  w_tot += __shfl_xor(w_tot, 32, 64);
  __syncthreads();
  float *mg = reinterpret_cast<float *>(smem);
  if (wave > 0) {
    float *dst = mg + (wave - 1) * MG;
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
      for (int v = 0; v < 4; ++v) dst[(16 * db + 4 * G + v) * 16 + q16] = acc[db][v] - w_tot;
  }
  __syncthreads();
  if (wave == 0 && q_ok) {
    _Float16 *out = a.dq + b * a.sdqb + h * a.sdqh + (int64_t)qi * a.sdqn;
#pragma unroll
    for (int db = 0; db < DB; ++db) {
      float r[4];
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int d = 16 * db + 4 * G + v;
        r[v] = acc[db][v] - w_tot + mg[d * 16 + q16] + mg[MG + d * 16 + q16] + mg[2 * MG + d * 16 + q16];
      }
      u32x2 o2;
      o2[0] = pack_out(r[0], r[1]);
      o2[1] = pack_out(r[2], r[3]);
      *reinterpret_cast<u32x2 *>(out + 16 * db + 4 * G) = o2;
    }
  }
}

// ------------------------------------------------------------------------------------------ dKV
// Chunk swizzle of the binary16 Q / dO / O rows in LDS (see row_swizzle in qfa_skv_bwd.hip): distinct for 16
// consecutive rows at one chunk index, whole 32-byte pairs apart for 4 consecutive rows.
template <int D> struct RowSwz {
  static constexpr int CPR = D / 8;
  static __device__ __forceinline__ int swz(int i) { return (2 * (i % 4) + (i / 4) % 2 + 8 * ((i / 8) % 2)) % CPR; }
};

struct SkvDkvSmem {
  static constexpr int D = 256, DS = 2;                          // waves sharing one tile (each keeps D / DS columns of dKV)
  static constexpr int SLOT = SKV_TILE * D + 2 * SKV_TILE * 4;   // one tile copy per wave
  static constexpr int ROWS = 32 * D * 2;                        // one block of 32 binary16 rows
  static constexpr int BUF = 2 * ROWS;                           // Q, dO of one query block
  static constexpr int OFF_SLOT = BUF;                           // tile copies behind the rows: both are copied at once in the prologue
  static constexpr int OFF_STAT = OFF_SLOT + 4 * SLOT;
  static constexpr int STAGE = 32 * 128;                         // per wave: 64 columns of its tile's dKV rows on their way out
  static constexpr int TOTAL = OFF_STAT + 4 * 32 * 4;            // statistics: lse (log2), delta, rowsum(Q), rowsum(dO)
  static_assert(4 * STAGE <= BUF && STAGE <= SLOT, "the output stage overlays the rows or the slot");
  static_assert(2 * BUF <= OFF_STAT, "the tile copies leave room for a second block of rows");
  static_assert(ROWS % 256 == 0, "row offsets are XOR-ed with block offsets");
  static_assert(2 * TOTAL <= 160 * 1024, "two workgroups per CU");
};

// KEEP: at most 32 queries.  They are copied once, their statistics are computed once, and the workgroup then walks over `cpw`
// consecutive 64-key chunks of its (batch, head) with no barrier at all.  Otherwise one workgroup per chunk, two barriers per
// block of rows.
template <typename S, bool KEEP> __global__ __launch_bounds__(256, 2) void skv_dkv256_kernel(SkvBwdLongArgs a) {
  typedef SkvDkvSmem SM;
  constexpr int D = SM::D, DS = SM::DS;
  typedef Swz<D> KSW;
  typedef TileCopy<D, SKV_TILE, 64, KSW> Copy;
  // 32 rows by 256 threads: a thread's chunks lie 8 rows apart and their swizzle repeats after 16, so two offsets serve all four
  struct RowCopy {
    unsigned off[2], step;
    __device__ __forceinline__ void init(unsigned stride, int tid) {
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const int row = tid / 32 + 8 * i;
        off[i] = (unsigned)row * stride + (unsigned)((tid % 32 ^ RowSwz<D>::swz(row)) << 4);
      }
      step = 16 * stride;
    }
    __device__ __forceinline__ void issue_one(rsrc_t rs, unsigned char *lds, int wave, int i) const {
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (lptr_t)(lds + (wave * 64 + 256 * i) * 16), 16, (int)off[i % 2], (int)(step * (unsigned)(i / 2)), 0, 0);
    }
  };
  constexpr int DB = D / 32, DBW = DB / DS, CPR = D / 8, KD = D / 16;
  __shared__ __attribute__((aligned(256))) unsigned char smem[SM::TOTAL];

  const int wgs_per_bh = (a.kchunks + a.cpw - 1) / a.cpw;
  const int bh = blockIdx.x / wgs_per_bh;
  const int c_begin = (blockIdx.x % wgs_per_bh) * a.cpw, c_end = min(a.kchunks, c_begin + a.cpw);
  const int64_t b = index_div(bh, a.H), h = bh - b * a.H;
  const int tid = threadIdx.x, lane = tid % 64, lr = lane % 32, g = lane / 32;
  const int wave = __builtin_amdgcn_readfirstlane(tid / 64);
  const int ntiles = (a.Nk + SKV_TILE - 1) / SKV_TILE;
  const int db0 = (wave % DS) * DBW;              // first of this wave's 32-column blocks of dKV
  unsigned char *slot = smem + SM::OFF_SLOT + wave * SM::SLOT;
  const unsigned char *codes_bh = reinterpret_cast<const unsigned char *>(a.codes + b * a.scb + h * a.sch);
  const int64_t tk0 = (int64_t)bh * a.Nk, tq0 = (int64_t)bh * a.Nq;
  const int nqb = (a.Nq + 31) / 32;
  auto tile_of = [&](int chunk) { return (4 / DS) * chunk + wave / DS; };   // this wave's tile in a chunk
  const float osc = a.grad_scale ? *a.grad_scale : 1.0f;
  auto pack_out = [&](float x, float y) -> unsigned {
    return a.grad_bf16 ? pack2<__bf16>(x * osc, y * osc) : pack2<_Float16>(x * osc, y * osc);
  };

  // ---- row copies of a query block: Q, dO (direct loads)
  RowCopy cq, cd;
  cq.init((unsigned)(a.sqn * 2), tid);
  cd.init((unsigned)(a.sdon * 2), tid);
  const _Float16 *q_bh = a.q + b * a.sqb + h * a.sqh, *d_bh = a.dout + b * a.sdob + h * a.sdoh, *o_bh = a.o + b * a.sob + h * a.soh;
  auto issue_rows = [&](int qb, unsigned char *buf) {
    const int rows = min(32, a.Nq - 32 * qb);
    // rows past Nq read as zeros (exact bounds; rows 16 on are in the scalar offset: see make_rsrc)
    const rsrc_t rq = make_rsrc(q_bh + (int64_t)32 * qb * a.sqn, (unsigned)(((rows - 1) * (int)a.sqn + D) * 2));
    const rsrc_t rd = make_rsrc(d_bh + (int64_t)32 * qb * a.sdon, (unsigned)(((rows - 1) * (int)a.sdon + D) * 2));
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      cq.issue_one(rq, buf, wave, c);
      cd.issue_one(rd, buf + SM::ROWS, wave, c);
    }
  };
  // delta, row sums, LSE of block qb from its rows (thread = row tid/8, chunks tid%8 + 8k); `og` holds this thread's chunks
  // of O, which does not pass through LDS
  auto block_stats = [&](int qb, const u32x4 *og, float lse, const unsigned char *buf) {
    float *stat = reinterpret_cast<float *>(smem + SM::OFF_STAT);
    const int pi = tid / 8, part = tid % 8;
    float dsum = 0.f, rq = 0.f, rd = 0.f;
#pragma unroll
    for (int c = part; c < CPR; c += 8) {
      const int off = pi * (D * 2) + ((c ^ RowSwz<D>::swz(pi)) << 4);
      const u32x4 qv = *reinterpret_cast<const u32x4 *>(buf + off);
      const u32x4 dv = *reinterpret_cast<const u32x4 *>(buf + SM::ROWS + off);
      const u32x4 ov = og[c / 8];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const unsigned qw = qv[e], dw = dv[e], ow = ov[e];
        const float d0 = lo_to_f32<_Float16>(dw), d1 = hi_to_f32<_Float16>(dw);
        rq += lo_to_f32<_Float16>(qw) + hi_to_f32<_Float16>(qw);
        rd += d0 + d1;
        dsum += lo_to_f32<_Float16>(ow) * d0 + hi_to_f32<_Float16>(ow) * d1;
      }
    }
#pragma unroll
    for (int m = 1; m < 8; m *= 2) {
      dsum += __shfl_xor(dsum, m, 64);
      rq += __shfl_xor(rq, m, 64);
      rd += __shfl_xor(rd, m, 64);
    }
    if (part == 0) {
      const int qi = 32 * qb + pi;
      stat[pi] = qi < a.Nq ? lse * kLog2e : INFINITY;
      stat[32 + pi] = dsum;
      stat[64 + pi] = rq;
      stat[96 + pi] = rd;
    }
  };
  auto load_o = [&](int qb, u32x4 *og, float &lse) {
    lse = a.lse[tq0 + min(32 * qb + tid / 8, a.Nq - 1)];
    const int pi = tid / 8, part = tid % 8;
    const bool live = 32 * qb + pi < a.Nq;
#pragma unroll
    for (int k = 0; k < (CPR + 7) / 8; ++k)
      og[k] = live ? *reinterpret_cast<const u32x4 *>(o_bh + (int64_t)(32 * qb + pi) * a.son + (part + 8 * k) * 8)
                   : u32x4{0u, 0u, 0u, 0u};
  };

  Copy cp;
  cp.init((unsigned)a.scn, lane);
  auto issue_tile = [&](int t) {
    skv_issue_tile<S, D>(cp, slot, codes_bh, a.scale, a.zp, tk0, t, a.Nk, a.scn, lane);
  };

  // ---- per-lane LDS offsets inside a row block (as in the fused kernel)
  const int row_off = lr * (D * 2), row_swz = RowSwz<D>::swz(lr);
  const int s16 = lane % 16, G = lane / 16;
  unsigned qt_off[2][2];
#pragma unroll
  for (int hh = 0; hh < 2; ++hh)
#pragma unroll
    for (int r = 0; r < 2; ++r) {
      const int i = 16 * hh + 8 * r + 4 * g + s16 / 4;
      const int chk = 2 * (G % 2) + (s16 % 4) / 2;
      qt_off[hh][r] = i * (D * 2) + ((chk ^ RowSwz<D>::swz(i)) << 4) + 8 * (s16 % 2);
    }

  // ---- this wave's tile in registers: code operands (B operands: column = key lr), scale, offset operand
  u32x4 cb[KD];
  float sk = 0.f;
  unsigned zw = 0u;   // this lane's zero point (low byte)
  auto expand_tile = [&]() {
    const int k_swz = KSW::swz(lr);
#pragma unroll
    for (int jj = 0; jj < D / 32; ++jj) {
      const u32x4 kw = *reinterpret_cast<const u32x4 *>(slot + lr * D + (((2 * jj + g) ^ k_swz) << 4));
      cb[2 * jj] = expand_codes(kw[0], kw[1]);
      cb[2 * jj + 1] = expand_codes(kw[2], kw[3]);
    }
    const unsigned *skp = reinterpret_cast<const unsigned *>(slot + SKV_TILE * D);
    const unsigned skw = skp[lr];
    zw = skp[SKV_TILE + lr];
    sk = scale_to_f32<S>(skw);
  };

  f32x16 dkv[DBW];
  // dKV^T of this wave's tile += contributions of query block qb (its rows and statistics are in LDS)
  auto add_block = [&](bool key_ok, const unsigned char *buf) {
    const float *stat = reinterpret_cast<const float *>(smem + SM::OFF_STAT);
    const float a_sk = key_ok ? a.sm_scale_log2 * sk : 0.f;
    const float sm_k = key_ok ? a.sm_scale : 0.f;
    // operands of the rank-1 offset removal: one scaling for the whole query block
    const float rs_q = stat[64 + lr], rs_do = stat[96 + lr];
    const bool big = offset_needs_x32(fmaxf(fabsf(rs_q), fabsf(rs_do)));
    u32x4 corr_q = {0u, 0u, 0u, 0u}, corr_do = {0u, 0u, 0u, 0u}, corr_k = {0u, 0u, 0u, 0u};
    if (g == 0) {
      const u32x2 cq2 = offset_query_operand(rs_q, big), cd2 = offset_query_operand(rs_do, big);
      const u32x2 ck2 = offset_key_operand(zw, big);
      corr_q[0] = cq2[0];
      corr_q[1] = cq2[1];
      corr_do[0] = cd2[0];
      corr_do[1] = cd2[1];
      corr_k[0] = ck2[0];
      corr_k[1] = ck2[1];
    }
    // S = Q C^T, dP = dO C^T (rows = queries, columns = keys), rank-1 offset removal
    f32x16 sacc, pacc;
#pragma unroll
    for (int v = 0; v < 16; ++v) sacc[v] = 0.f, pacc[v] = 0.f;
#pragma unroll
    for (int m = 0; m < KD; ++m) {
      const int off = row_off + (((4 * (m / 2) + 2 * g + m % 2) ^ row_swz) << 4);
      const u32x4 qa = *reinterpret_cast<const u32x4 *>(buf + off);
      const u32x4 da = *reinterpret_cast<const u32x4 *>(buf + SM::ROWS + off);
      sacc = mfma_h(qa, cb[m], sacc);
      pacc = mfma_h(da, cb[m], pacc);
    }
    sacc = mfma_h(corr_q, corr_k, sacc);
    pacc = mfma_h(corr_do, corr_k, pacc);
    u32x2 fr[2][2][2];   // [matrix: dO, Q][hh][r], requested when needed: the registers are full
    auto request = [&](int db) __attribute__((always_inline)) {
#pragma unroll
      for (int hh = 0; hh < 2; ++hh)
#pragma unroll
        for (int r = 0; r < 2; ++r) {
          const unsigned ad = lds_addr(buf) + (qt_off[hh][r] ^ ((4 * (db0 + db)) << 4));
          fr[0][hh][r] = lds_read_tr16_async<SM::ROWS>(ad);
          fr[1][hh][r] = lds_read_tr16_async<0>(ad);
        }
    };
    // p and ds for this lane's key; registers run over the queries 8aa + 4g + bb
    u32x4 pf[2], df[2];
#pragma unroll
    for (int aa = 0; aa < 4; ++aa) {
      const f32x4 l4 = *reinterpret_cast<const f32x4 *>(stat + 8 * aa + 4 * g);
      const f32x4 d4 = *reinterpret_cast<const f32x4 *>(stat + 32 + 8 * aa + 4 * g);
      float p[4], ds[4];
#pragma unroll
      for (int bb = 0; bb < 4; ++bb) {
        const int v = 4 * aa + bb;
        p[bb] = key_ok ? __builtin_amdgcn_exp2f(__builtin_fmaf(a_sk, sacc[v], -l4[bb])) : 0.f;
        ds[bb] = sm_k * p[bb] * (pacc[v] * sk - d4[bb]);
      }
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        pf[aa / 2][2 * (aa % 2) + e] = pack_h2(p[2 * e], p[2 * e + 1]);
        df[aa / 2][2 * (aa % 2) + e] = pack_h2(ds[2 * e], ds[2 * e + 1]);
      }
    }
    // dKV^T += dO^T P + Q^T dS
#pragma unroll
    for (int db = 0; db < DBW; ++db) {
      request(db);
      lds_wait_all();
      u32x2 now[2][2][2];
#pragma unroll
      for (int x = 0; x < 8; ++x) now[x / 4][x / 2 % 2][x % 2] = tie(fr[x / 4][x / 2 % 2][x % 2]);
#pragma unroll
      for (int hh = 0; hh < 2; ++hh) {
        const u32x2(&d)[2] = now[0][hh], (&q)[2] = now[1][hh];
        dkv[db] = mfma_h(u32x4{d[0][0], d[0][1], d[1][0], d[1][1]}, pf[hh], dkv[db]);
        dkv[db] = mfma_h(u32x4{q[0][0], q[0][1], q[1][0], q[1][1]}, df[hh], dkv[db]);
      }
    }
  };
  // the tile's dKV rows leave through a 4 KB LDS stage as whole 128-byte lines (two 32-column blocks a time)
  auto write_out = [&](unsigned char *stage, int j0) {
    _Float16 *dkv_bh = a.dkv + b * a.sdkb + h * a.sdkh;
    const int st_w = lr * 128 + 8 * g, st_wswz = lr % 8;
    const int st_r = (lane / 8) * 128 + (((lane % 8) ^ (lane / 8)) << 4);
#pragma unroll
    for (int db = 0; db < DBW; ++db) {
#pragma unroll
      for (int aa = 0; aa < 4; ++aa) {
        u32x2 o2;
        o2[0] = pack_out(dkv[db][4 * aa], dkv[db][4 * aa + 1]);
        o2[1] = pack_out(dkv[db][4 * aa + 2], dkv[db][4 * aa + 3]);
        *reinterpret_cast<u32x2 *>(stage + st_w + (((4 * (db % 2) + aa) ^ st_wswz) << 4)) = o2;
      }
      if (db % 2 == 1) {
#pragma unroll
        for (int it = 0; it < 4; ++it) {
          const u32x4 row16 = *reinterpret_cast<const u32x4 *>(stage + st_r + it * 1024);
          const int j = j0 + 8 * it + lane / 8;
          if (j < a.Nk) *reinterpret_cast<u32x4 *>(dkv_bh + (int64_t)j * a.sdkn + 32 * (db0 + db - 1) + 8 * (lane % 8)) = row16;
        }
      }
    }
  };
  auto clear_dkv = [&]() {
#pragma unroll
    for (int db = 0; db < DBW; ++db)
#pragma unroll
      for (int v = 0; v < 16; ++v) dkv[db][v] = 0.f;
  };

  u32x4 og[(CPR + 7) / 8];
  float lse;
  if (KEEP) {
    // ---- the rows and the first tile, copied together; statistics once
    if (tile_of(c_begin) < ntiles) issue_tile(tile_of(c_begin));
    issue_rows(0, smem);
    load_o(0, og, lse);
    dma_wait();
    __syncthreads();
    block_stats(0, og, lse, smem);
    __syncthreads();
    // The output stage is the wave's tile slot once its operands are in registers, so the next tile's copy goes out after the
    // stores, and the wait at the top of the next round covers both.
    for (int c = c_begin; c < c_end; ++c) {
      const int t = tile_of(c);
      if (t >= ntiles) break;   // (tiles of a wave grow with c)
      dma_wait();
      expand_tile();
      const int tn = tile_of(c + 1);
      clear_dkv();
      const int j0 = t * SKV_TILE;
      add_block(j0 + lr < a.Nk, smem);
      write_out(slot, j0);
      if (c + 1 < c_end && tn < ntiles) {
        lds_wait_all();
        issue_tile(tn);
      }
    }
    return;
  }

  // ---- one chunk per workgroup
  const int t = tile_of(c_begin);
  const bool t_ok = t < ntiles;                   // (a wave without a tile still takes part in copies and barriers)
  const int j0 = t * SKV_TILE;
  if (t_ok) issue_tile(t);
  issue_rows(0, smem);   // together with the tile: one memory latency for both
  load_o(0, og, lse);
  dma_wait();
  if (t_ok) expand_tile();
  clear_dkv();
  // Every tile is in registers: the next block's rows land where the copies were, and its O and LSE are on their way, while this one
  // is worked on (one block after the other waited for memory: whole backward, 1584 heads, 97 x 689: 1148 -> 1090 us; 256 heads, 512 x
  // 4096: 3246 -> 3134)
  __syncthreads();
  for (int qb = 0; qb < nqb; ++qb) {
    unsigned char *buf = smem + qb % 2 * SM::BUF;
    if (qb + 1 < nqb) issue_rows(qb + 1, smem + (qb + 1) % 2 * SM::BUF);
    block_stats(qb, og, lse, buf);
    if (qb + 1 < nqb) load_o(qb + 1, og, lse);
    lds_barrier();
    if (t_ok) add_block(j0 + lr < a.Nk, buf);
    dma_wait();          // this thread's share of the next block has landed ...
    lds_barrier();       // ... and everybody's, and everybody is done with this one
  }
  __syncthreads();   // the rows are done with: the stages overlay them
  if (t_ok) write_out(smem + wave * SM::STAGE, j0);
}

template <typename S, int D> static int launch_skv_bwd_long_sd(const SkvAttnArgs &x, hipStream_t st) {
  SkvBwdLongArgs a;
  a.q = static_cast<const _Float16 *>(x.q); a.o = static_cast<const _Float16 *>(x.o);
  a.dout = static_cast<const _Float16 *>(x.dout);
  a.codes = x.codes; a.scale = x.scale; a.zp = x.zp; a.lse = x.lse;
  a.dq = static_cast<_Float16 *>(x.dq); a.dkv = static_cast<_Float16 *>(x.dkv);
  a.grad_scale = x.grad_scale; a.grad_bf16 = x.grad_dtype == QFA_BF16;
  a.direct = x.direct; a.q_bf16 = x.io_dtype == QFA_BF16; a.do_bf16 = x.dout_dtype == QFA_BF16;
  a.H = x.H; a.Nq = (int)x.Nq; a.Nk = (int)x.Nk;
  a.sqb = x.sqb; a.sqh = x.sqh; a.sqn = x.sqn; a.scb = x.scb; a.sch = x.sch; a.scn = x.scn;
  a.sob = x.sob; a.soh = x.soh; a.son = x.son; a.sdob = x.sdob; a.sdoh = x.sdoh; a.sdon = x.sdon;
  a.sdqb = x.sdqb; a.sdqh = x.sdqh; a.sdqn = x.sdqn; a.sdkb = x.sdkb; a.sdkh = x.sdkh; a.sdkn = x.sdkn;
  a.sm_scale = x.sm_scale;
  a.sm_scale_log2 = x.sm_scale * kLog2e;
  if (x.B * x.H > 0x7fffffffLL) return set_error(QFA_EUNSUPPORTED, "attn_bwd_shared_kv: too many (batch, head) pairs");
  a.BH = (int)(x.B * x.H);
  a.qblocks = (int)((x.Nq + 15) / 16);
  const int64_t total_q = xcd_grid(a.BH, a.qblocks);
  if (total_q > 0x7fffffffLL) return set_error(QFA_EUNSUPPORTED, "attn_bwd_shared_kv: too many blocks for one launch");
  const SkvTilePlan p = skv_tile_dq_plan(x.B * x.H, x.Nq, x.Nk, D);
  if (p.qw && (p.splits == 1 || x.workspace)) {
    if (int e = launch_skv_tile_dq(x, p, st)) return e;
  } else {
    skv_dq_kernel<S, D><<<dim3((unsigned)total_q), dim3(256), 0, st>>>(a);
    if (int e = check_launch("qfa_attn_bwd_shared_kv (dQ)")) return e;
  }
  if constexpr (D < 256) {
    return launch_skv_dkv(x, st);
  } else {
    const int keys_per_wg = 4 * SKV_TILE / SkvDkvSmem::DS;
    a.kchunks = (int)((x.Nk + keys_per_wg - 1) / keys_per_wg);
    // a query block that stays resident: a workgroup walks over as many chunks as leave about 2048 workgroups (four rounds of
    // two per CU)
    const bool keep = x.Nq <= 32;
    a.cpw = 1;
    if (keep) {
      const int64_t want = ((int64_t)a.kchunks * a.BH + 2047) / 2048;
      a.cpw = (int)(want < 1 ? 1 : want > a.kchunks ? a.kchunks : want);
    }
    const int64_t total_k = (int64_t)((a.kchunks + a.cpw - 1) / a.cpw) * a.BH;
    if (total_k > 0x7fffffffLL) return set_error(QFA_EUNSUPPORTED, "attn_bwd_shared_kv: too many blocks for one launch");
    if (keep) skv_dkv256_kernel<S, true><<<dim3((unsigned)total_k), dim3(256), 0, st>>>(a);
    else skv_dkv256_kernel<S, false><<<dim3((unsigned)total_k), dim3(256), 0, st>>>(a);
    return check_launch("qfa_attn_bwd_shared_kv (dKV)");
  }
}

int launch_skv_bwd_long(const SkvAttnArgs &x, hipStream_t st) {
  const bool pass = x.workspace ? skv_pass_takes(x.B * x.H, x.Nq, x.Nk, x.D) : skv_pass_takes_unsplit(x.B * x.H, x.Nq, x.Nk, x.D);
  if (pass && skv_pass_fits(x.Nk, x.scn, x.sdqn, x.sdkn)) return launch_skv_pass(x, st);
  const bool s32 = x.scale_dtype == QFA_F32;
  if (x.D == 256) return s32 ? launch_skv_bwd_long_sd<float, 256>(x, st) : launch_skv_bwd_long_sd<_Float16, 256>(x, st);
  if (x.D == 128) return s32 ? launch_skv_bwd_long_sd<float, 128>(x, st) : launch_skv_bwd_long_sd<_Float16, 128>(x, st);
  if (x.D == 64) return s32 ? launch_skv_bwd_long_sd<float, 64>(x, st) : launch_skv_bwd_long_sd<_Float16, 64>(x, st);
  return set_error(QFA_EUNSUPPORTED, "attn_bwd_shared_kv: head_dim must be 64, 128 or 256");
}

}  // namespace qfa
