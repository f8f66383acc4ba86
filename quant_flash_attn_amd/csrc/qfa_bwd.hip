// Backward for gfx950: the staging passes here, then one launch of two kinds of workgroups (qfa_bwd_pair.h) that recompute
// P = exp(S - LSE) from the INT8 codes exactly as the forward does.
//
//   prep_q       per 64-query tile: delta = rowsum(O o dO) in fp32; Qz^T = ((Qc - zq) * sq)^T as a
//                16-bit tile [d][query] in the key order the MFMA layouts want; per-query constants
//   prep_k       per 64-key tile: Kz^T = ((Kc - zk) * sk)^T likewise; per-key constants
//                (both write into the caller's workspace; every tile is converted and transposed
//                once instead of once per consuming workgroup)
//   dK / dV      qfa_bwd_dkv.inc: a workgroup owns keys and streams query tiles
//   dQ           qfa_bwd_dq.inc: a workgroup owns queries and streams key tiles
// In both, the wave's own operand (queries resp. keys) stays in registers as the MFMA B operand
// for the whole loop and the streamed operand comes from LDS as the A operand.  The 32x32
// accumulator layout then leaves P / dS in registers exactly in the B-operand layout of the next
// product; the transposed tiles (Kz^T, Qz^T) are written in the matching permuted order.
// dQ is produced by workgroups of its own instead of atomics, so results are deterministic.
// The scales of the streamed operand are folded into its transposed 16-bit tile (Kz^T, Qz^T) by the staging
// pass, so dS is used as it comes: the tiles then hold the dequantized K and Q rounded to the 16-bit type, the
// operands an unquantized backward would use.
#include <type_traits>

#include "qfa_bwd_common.h"

namespace qfa {

// ------------------------------------------------------------------------------------------ delta
struct DeltaArgs {
  const void *o; const void *dout; float *delta;
  int64_t N, H;
  int64_t sob, soh, son, sdb, sdh, sdn;
  int chunks_per_bh;
};

template <typename T, int D> __global__ __launch_bounds__(256) void delta_kernel(DeltaArgs a) {
  constexpr int LPT = D / 8;
  constexpr int TPP = 256 / LPT;
  const int tid = threadIdx.x, sub = tid % LPT;
  const int64_t bh = blockIdx.x / a.chunks_per_bh, chunk = blockIdx.x % a.chunks_per_bh;
  const int64_t b = index_div(bh, a.H), h = bh - b * a.H;
  const int64_t n = chunk * (int64_t)TPP + tid / LPT;
  const int64_t nn = n < a.N ? n : a.N - 1;
  const u32x4 ow = *reinterpret_cast<const u32x4 *>(reinterpret_cast<const T *>(a.o) + b * a.sob + h * a.soh +
                                                     nn * a.son + sub * 8);
  const u32x4 gw = *reinterpret_cast<const u32x4 *>(reinterpret_cast<const T *>(a.dout) + b * a.sdb + h * a.sdh +
                                                     nn * a.sdn + sub * 8);
  float s = 0.f;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    s = __builtin_fmaf(lo_to_f32<T>(ow[e]), lo_to_f32<T>(gw[e]), s);
    s = __builtin_fmaf(hi_to_f32<T>(ow[e]), hi_to_f32<T>(gw[e]), s);
  }
  s += dpp_f<0xB1>(s);
  s += dpp_f<0x4E>(s);
  s += dpp_f<0x141>(s);
  if (LPT >= 16) s += dpp_f<0x140>(s);
  if (LPT >= 32) s += __shfl_xor(s, 16);
  if (n < a.N && sub == 0) a.delta[bh * a.N + n] = s;
}

// out = a + b for two 16-bit tensors of the same dense shape, added in fp32 and rounded once: dKV = dK + dV of the
// shared K = V contract (quant_flash_attn.py:161) when the two gradients come from the INT8-score kernels.
template <typename T> __global__ __launch_bounds__(256) void sum16_kernel(const T *a, const T *b, T *out, int64_t n8) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= n8) return;
  const u32x4 x = reinterpret_cast<const u32x4 *>(a)[i], y = reinterpret_cast<const u32x4 *>(b)[i];
  u32x4 r;
#pragma unroll
  for (int e = 0; e < 4; ++e)
    r[e] = pack2<T>(lo_to_f32<T>(x[e]) + lo_to_f32<T>(y[e]), hi_to_f32<T>(x[e]) + hi_to_f32<T>(y[e]));
  reinterpret_cast<u32x4 *>(out)[i] = r;
}
int launch_sum16(const void *a, const void *b, void *out, int dtype, int64_t n, hipStream_t st) {
  const int64_t n8 = n / 8, blocks = (n8 + 255) / 256;
  if (blocks > 0x7fffffffLL) return set_error(QFA_EUNSUPPORTED, "sum_grads: too many elements for one launch");
  if (dtype == QFA_BF16)
    sum16_kernel<__bf16><<<dim3((unsigned)blocks), dim3(256), 0, st>>>((const __bf16 *)a, (const __bf16 *)b, (__bf16 *)out, n8);
  else
    sum16_kernel<_Float16><<<dim3((unsigned)blocks), dim3(256), 0, st>>>((const _Float16 *)a, (const _Float16 *)b, (_Float16 *)out, n8);
  return check_launch("qfa_sum_grads");
}

int launch_delta(const void *o, const void *dout, float *delta, int io_dtype, int64_t B, int64_t H, int64_t N, int D,
                 int64_t sob, int64_t soh, int64_t son, int64_t sdb, int64_t sdh, int64_t sdn, hipStream_t st) {
  DeltaArgs a;
  a.o = o; a.dout = dout; a.delta = delta; a.N = N; a.H = H;
  a.sob = sob; a.soh = soh; a.son = son; a.sdb = sdb; a.sdh = sdh; a.sdn = sdn;
  const int tpp = 256 / (D / 8);
  const int64_t chunks = (N + tpp - 1) / tpp;
  if (chunks * B * H > 0x7fffffffLL) return set_error(QFA_EUNSUPPORTED, "bwd_delta: too many tokens for one launch");
  a.chunks_per_bh = (int)chunks;
  const dim3 grid((unsigned)(chunks * B * H)), block(256);
  if (io_dtype == QFA_BF16) {
    if (D == 256) delta_kernel<__bf16, 256><<<grid, block, 0, st>>>(a);
    else if (D == 128) delta_kernel<__bf16, 128><<<grid, block, 0, st>>>(a);
    else delta_kernel<__bf16, 64><<<grid, block, 0, st>>>(a);
  } else {
    if (D == 256) delta_kernel<_Float16, 256><<<grid, block, 0, st>>>(a);
    else if (D == 128) delta_kernel<_Float16, 128><<<grid, block, 0, st>>>(a);
    else delta_kernel<_Float16, 64><<<grid, block, 0, st>>>(a);
  }
  return check_launch("qfa_bwd_delta");
}

int64_t bwd_workspace_bytes(int64_t B, int64_t H, int64_t Nq, int64_t Nk, int D) {
  const int64_t tile = D == 256 ? BwdWs<256>::TILE : 64;
  const int64_t tq = (Nq + tile - 1) / tile, tk = (Nk + tile - 1) / tile;
  const int64_t qb = D == 256 ? BwdWs<256>::Q_BLOB : D == 128 ? BwdWs<128>::Q_BLOB : BwdWs<64>::Q_BLOB;
  const int64_t kb = D == 256 ? BwdWs<256>::K_BLOB : D == 128 ? BwdWs<128>::K_BLOB : BwdWs<64>::K_BLOB;
  return B * H * (tq * qb + tk * kb);
}

// (code - zp) * scale for the 8 codes in two dwords of 4 rows, rounded to 16 bits, transposed: for each of the 8 columns
// the 4 rows as 8 bytes at dst(column)
template <typename T, typename F>
__device__ __forceinline__ void store_codes_transposed(const u32x2 (&c)[4], const float (&zp)[4], const float (&sc)[4], F dst) {
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    float f[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) f[r] = ((float)(int)(int8_t)((c[r][e / 4] >> (8 * (e % 4))) & 0xff) - zp[r]) * sc[r];
    u32x2 o;
    o[0] = pack2<T>(f[0], f[1]);
    o[1] = pack2<T>(f[2], f[3]);
    *reinterpret_cast<u32x2 *>(dst(e)) = o;
  }
}
// integer n -> (2^SH * floor(n / 2^SH), n mod 2^SH) resp. their negatives, as a packed pair of 16-bit floats
template <typename T, int SH = 7> __device__ __forceinline__ unsigned base128_pair(int n, float sign) {
  const int hi = n >> SH, lo = n & ((1 << SH) - 1);
  return pack2<T>(sign * (float)(hi * (1 << SH)), sign * (float)lo);
}

// ------------------------------------------------------------------------------------------ prep
// Staging passes: one workgroup per (b,h, 64-query tile), then one per (b,h, 64-key tile), in one launch.  Bound by memory:
// a thread takes 8 columns of 4 rows with the columns of a row on neighbouring lanes (whole rows are read), and the
// transposed tile goes through LDS so that it leaves in 16-byte pieces in a row.  128 heads of 4096 x 128: 671 MB in 109 us
// (6.2 TB/s), against 166 us for two launches that wrote the tiles in 8-byte pieces straight from registers.
template <int D> struct PrepSmem {
  __attribute__((aligned(16))) unsigned char tile[BwdWs<D>::T_BYTES];
  float red[D / 8][BwdWs<D>::TILE + 1];
};
// where byte `off` of a transposed tile is staged: 32-byte pieces of columns 8 apart lie in different banks
__device__ __forceinline__ int prep_stage(int off) { return off ^ ((off >> 8 & 7) << 5); }
template <int D> __device__ __forceinline__ void prep_store_tile(const unsigned char *tile, unsigned char *blob, int tid) {
#pragma unroll
  for (int o = 0; o < BwdWs<D>::T_BYTES; o += 4096)
    *reinterpret_cast<u32x4 *>(blob + o + tid * 16) = *reinterpret_cast<const u32x4 *>(tile + prep_stage(o + tid * 16));
}

// delta, Qz^T and the per-query constants
template <typename T, int D> __device__ __forceinline__ void prep_q(const BwdArgs &a, int blk, PrepSmem<D> &sm) {
  typedef BwdWs<D> WS;
  constexpr int BWD_TILE = WS::TILE;
  const int tid = threadIdx.x;
  const int bh = blk / a.tiles_q, tile = blk % a.tiles_q;
  const int64_t b = index_div(bh, a.H), h = bh - b * a.H;
  const int i0 = tile * BWD_TILE;
  const int64_t tq0 = (int64_t)bh * a.Nq;
  unsigned char *blob = a.ws_q + ((int64_t)bh * a.tiles_q + tile) * WS::Q_BLOB;
  const int dc = tid % (D / 8), r4 = tid / (D / 8);
  if (r4 < BWD_TILE / 4) {
    const int8_t *qc_bh = a.qc + b * a.sqb + h * a.sqh;
    const T *do_bh = reinterpret_cast<const T *>(a.dout) + b * a.sdob + h * a.sdoh;
    const T *o_bh = reinterpret_cast<const T *>(a.o) + b * a.sob + h * a.soh;
    u32x2 creg[4];
    u32x4 greg[4];
    float zreg[4], sreg[4];
    if (a.dout32) {   // (outside the loop below, whose loads go out together)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int i = min(i0 + 4 * r4 + r, a.Nq - 1);
        const f32x4 *g32 = reinterpret_cast<const f32x4 *>(a.dout32 + b * a.sd32b + h * a.sd32h + (int64_t)i * a.sd32n + dc * 8);
        const f32x4 x = g32[0], y = g32[1];
        greg[r] = u32x4{pack2<T>(x[0], x[1]), pack2<T>(x[2], x[3]), pack2<T>(y[0], y[1]), pack2<T>(y[2], y[3])};
        if (i0 + 4 * r4 + r < a.Nq) *reinterpret_cast<u32x4 *>(reinterpret_cast<T *>(a.do16) + (tq0 + i) * D + dc * 8) = greg[r];
      }
    } else {
#pragma unroll
      for (int r = 0; r < 4; ++r)
        greg[r] = *reinterpret_cast<const u32x4 *>(do_bh + (int64_t)min(i0 + 4 * r4 + r, a.Nq - 1) * a.sdon + dc * 8);
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int i = min(i0 + 4 * r4 + r, a.Nq - 1);
      creg[r] = *reinterpret_cast<const u32x2 *>(qc_bh + (int64_t)i * a.sqn + dc * 8);
      const u32x4 gw = greg[r];
      const u32x4 ow = *reinterpret_cast<const u32x4 *>(o_bh + (int64_t)i * a.son + dc * 8);
      zreg[r] = (float)a.zq[tq0 + i];
      sreg[r] = a.sq[tq0 + i];
      float s = 0.f;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        s = __builtin_fmaf(lo_to_f32<T>(ow[e]), lo_to_f32<T>(gw[e]), s);
        s = __builtin_fmaf(hi_to_f32<T>(ow[e]), hi_to_f32<T>(gw[e]), s);
      }
      sm.red[dc][4 * r4 + r] = s;
    }
    const int pos = perm_pos4(r4);
    // the dequantized Q itself, rounded to the 16-bit type (what dK = sm * dS^T Q^ contracts with)
    store_codes_transposed<T>(creg, zreg, sreg, [&](int e) { return sm.tile + prep_stage(qt_offset<D>(dc * 8 + e, pos)); });
  }
  __syncthreads();
  prep_store_tile<D>(sm.tile, blob, tid);
  if (tid < BWD_TILE) {
    const int i = min(i0 + tid, a.Nq - 1);
    float delta = 0.f;
#pragma unroll
    for (int x = 0; x < D / 8; ++x) delta += sm.red[x][tid];
    const int zq = (int)a.zq[tq0 + i];
    const int c = a.rq[tq0 + i] - D * zq;
    unsigned *cq = reinterpret_cast<unsigned *>(blob + WS::T_BYTES);
    u32x2 dg;
    dg[0] = pack2<T>((float)(-zq), (float)(-zq));      // k-group 0: times the two digits of rk
    dg[1] = base128_pair<T, WS::CSH>(c, -1.0f);        // k-group 1: minus the digits of rq - D*zq, times zk
    reinterpret_cast<u32x2 *>(cq)[tid] = dg;
    reinterpret_cast<float *>(cq)[2 * BWD_TILE + tid] = a.sq[tq0 + i] * a.sm_scale_log2;
    reinterpret_cast<float *>(cq)[3 * BWD_TILE + tid] = -a.lse[tq0 + i] * kLog2e;
    reinterpret_cast<float *>(cq)[4 * BWD_TILE + tid] = -delta;   // the dP accumulators start from it
  }
}

// Kz^T and the per-key constants
template <typename T, int D> __device__ __forceinline__ void prep_k(const BwdArgs &a, int blk, PrepSmem<D> &sm) {
  typedef BwdWs<D> WS;
  constexpr int BWD_TILE = WS::TILE;
  const int tid = threadIdx.x;
  const int bh = blk / a.tiles_k, tile = blk % a.tiles_k;
  const int64_t b = index_div(bh, a.H), h = bh - b * a.H;
  const int j0 = tile * BWD_TILE;
  const int64_t tk0 = (int64_t)bh * a.Nk;
  unsigned char *blob = a.ws_k + ((int64_t)bh * a.tiles_k + tile) * WS::K_BLOB;
  const int dc = tid % (D / 8), r4 = tid / (D / 8);
  if (r4 < BWD_TILE / 4) {
    const int8_t *kc_bh = a.kc + b * a.skb + h * a.skh;
    u32x2 creg[4];
    float zreg[4], sreg[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int j = min(j0 + 4 * r4 + r, a.Nk - 1);
      creg[r] = *reinterpret_cast<const u32x2 *>(kc_bh + (int64_t)j * a.skn + dc * 8);
      zreg[r] = (float)a.zk[tk0 + j];
      sreg[r] = a.sk[tk0 + j];
    }
    // the dequantized K, rounded to the 16-bit type (what dQ = sm * dS K^ contracts with)
    const int pos = perm_pos4(r4);
    store_codes_transposed<T>(creg, zreg, sreg, [&](int e) { return sm.tile + prep_stage(qt_offset<D>(dc * 8 + e, pos)); });
  }
  __syncthreads();
  prep_store_tile<D>(sm.tile, blob, tid);
  if (tid < BWD_TILE) {
    const int j = min(j0 + tid, a.Nk - 1);
    const int zk = (int)a.zk[tk0 + j];
    unsigned *ck = reinterpret_cast<unsigned *>(blob + WS::T_BYTES);
    u32x2 dg;
    dg[0] = base128_pair<T>(a.rk[tk0 + j], 1.0f);      // k-group 0: digits of rk
    dg[1] = pack2<T>((float)zk, (float)zk);            // k-group 1: zk, zk
    reinterpret_cast<u32x2 *>(ck)[tid] = dg;
    reinterpret_cast<float *>(ck)[2 * BWD_TILE + tid] = a.sk[tk0 + j];
  }
}

template <typename T, int D> __global__ __launch_bounds__(256) void bwd_prep_kernel(BwdArgs a, int blocks_q) {
  static_assert((BwdWs<D>::TILE / 4) * (D / 8) <= 256, "one thread per 4 rows x 8 columns");
  __shared__ PrepSmem<D> sm;
  const int blk = blockIdx.x;
  if (blk < blocks_q) prep_q<T, D>(a, blk, sm);
  else prep_k<T, D>(a, blk - blocks_q, sm);
}

// ------------------------------------------------------------------------------------------ sum of parts
// Gradients whose streamed rows were split: up to three tensors, each [B*H][splits][N][D] in fp32, added in the order of the
// parts and rounded once.  Bound by memory.
struct BwdSumArgs {
  struct One { const float *part; void *out; int64_t sb, sh, sn, rows; int N, splits, first_block; } t[3];
  int64_t H;
  int count, out_f32;
};
template <typename T, int D> __global__ __launch_bounds__(256) void bwd_sum_kernel(BwdSumArgs a) {
  constexpr int CL = D / 4, RPW = 256 / CL;   // four columns of a row per thread
  int i = 0;
  while (i + 1 < a.count && (int)blockIdx.x >= a.t[i + 1].first_block) ++i;
  const BwdSumArgs::One &x = a.t[i];
  const int64_t row = (int64_t)((int)blockIdx.x - x.first_block) * RPW + threadIdx.x / CL;   // of B*H*N
  const int d = 4 * (threadIdx.x % CL);
  if (row >= x.rows) return;
  const int64_t bh = index_div(row, x.N), n = row - bh * x.N, step = (int64_t)x.N * D, b = index_div(bh, a.H), h = bh - b * a.H;
  const float *p = x.part + bh * x.splits * step + n * D + d;
  f32x4 acc = *reinterpret_cast<const f32x4 *>(p);
#pragma unroll 4
  for (int s = 1; s < x.splits; ++s) {
    const f32x4 y = *reinterpret_cast<const f32x4 *>(p + s * step);
#pragma unroll
    for (int e = 0; e < 4; ++e) acc[e] += y[e];
  }
  const int64_t at = b * x.sb + h * x.sh + n * x.sn + d;
  if (a.out_f32) *reinterpret_cast<f32x4 *>(static_cast<float *>(x.out) + at) = acc;
  else *reinterpret_cast<u32x2 *>(static_cast<T *>(x.out) + at) = u32x2{pack2<T>(acc[0], acc[1]), pack2<T>(acc[2], acc[3])};
}

template <typename T, int D> static int launch_bwd_td(const AttnArgs &x, hipStream_t st) {
  typedef BwdWs<D> WS;
  BwdArgs a;
  a.qc = x.qc; a.sq = x.sq; a.zq = x.zq; a.rq = x.rq; a.kc = x.kc; a.sk = x.sk; a.zk = x.zk; a.rk = x.rk;
  a.v = x.v; a.o = x.o; a.dout = x.dout; a.lse = x.lse; a.dq = x.dq; a.dk = x.dk; a.dv = x.dv;
  a.H = x.H; a.Nq = (int)x.Nq; a.Nk = (int)x.Nk;
  a.tiles_q = (int)((x.Nq + WS::TILE - 1) / WS::TILE);
  a.tiles_k = (int)((x.Nk + WS::TILE - 1) / WS::TILE);
  a.ws_q = reinterpret_cast<unsigned char *>(x.workspace);
  a.ws_k = a.ws_q + x.B * x.H * (int64_t)a.tiles_q * WS::Q_BLOB;
  a.sqb = x.sqb; a.sqh = x.sqh; a.sqn = x.sqn; a.skb = x.skb; a.skh = x.skh; a.skn = x.skn;
  a.svb = x.svb; a.svh = x.svh; a.svn = x.svn; a.sob = x.sob; a.soh = x.soh; a.son = x.son;
  a.sdob = x.sdob; a.sdoh = x.sdoh; a.sdon = x.sdon; a.sdqb = x.sdqb; a.sdqh = x.sdqh; a.sdqn = x.sdqn;
  a.sdkb = x.sdkb; a.sdkh = x.sdkh; a.sdkn = x.sdkn; a.sdvb = x.sdvb; a.sdvh = x.sdvh; a.sdvn = x.sdvn;
  a.sm_scale = x.sm_scale; a.sm_scale_log2 = x.sm_scale * kLog2e;
  a.nblocks = 0; a.total_blocks = 0; a.blocks_per_xcd = 0; a.group_log2 = 0;
  const int64_t BH = x.B * x.H;
  a.dout32 = nullptr; a.do16 = nullptr; a.sd32b = a.sd32h = a.sd32n = 0;
  a.grad_f32 = x.f32;
  if (x.f32) {   // dO and the gradients in fp32: the 16-bit dO lies behind the staged tiles
    a.dout32 = static_cast<const float *>(x.dout);
    a.sd32b = x.sdob; a.sd32h = x.sdoh; a.sd32n = x.sdon;
    a.dout = a.do16 = a.ws_k + BH * (int64_t)a.tiles_k * WS::K_BLOB;
    a.sdob = x.H * x.Nq * D; a.sdoh = x.Nq * D; a.sdon = D;
  }
  if (BH * (a.tiles_q + a.tiles_k) > 0x7fffffffLL)
    return set_error(QFA_EUNSUPPORTED, "attn_bwd: too many tiles for one launch");
  bwd_prep_kernel<T, D><<<dim3((unsigned)(BH * (a.tiles_q + a.tiles_k))), dim3(256), 0, st>>>(a, (int)(BH * a.tiles_q));
  if (int e = check_launch("qfa_attn_bwd (staging)")) return e;
  const BwdPlan &plan = x.bwd;
  float *const parts = reinterpret_cast<float *>(a.ws_q + (x.f32 ? bwd_f32_workspace_bytes(x.B, x.H, x.Nq, x.Nk, D)
                                                         : bwd_workspace_bytes(x.B, x.H, x.Nq, x.Nk, D)));
  float *part = parts;
  BwdSumArgs sum;
  sum.count = 0; sum.H = x.H; sum.out_f32 = x.f32;
  int64_t blocks = 0;
  // the split gradient of N rows: where its parts go, and what adds them
  auto split = [&](void *&out, int64_t &sb, int64_t &sh, int64_t &sn, int64_t N, int splits) {
    sum.t[sum.count++] = {part, out, sb, sh, sn, BH * N, (int)N, splits, (int)blocks};
    blocks += (BH * N + 1024 / D - 1) / (1024 / D);
    out = part;
    sn = D; sh = splits * N * D; sb = x.H * sh;
    part += BH * splits * N * D;
  };
  BwdArgs k = a;   // dK, dV
  k.per_split = plan.queries_per_split;
  k.last_part = (plan.splits_dkv - 1) * plan.queries_per_split;
  k.split_stride = 0;
  if (plan.splits_dkv > 1) {
    split(k.dk, k.sdkb, k.sdkh, k.sdkn, x.Nk, plan.splits_dkv);
    split(k.dv, k.sdvb, k.sdvh, k.sdvn, x.Nk, plan.splits_dkv);
    k.split_stride = x.Nk * D;
    k.grad_f32 = 1;
  }
  auto add_parts = [&]() -> int {
    if (sum.count == 0) return 0;
    bwd_sum_kernel<T, D><<<dim3((unsigned)blocks), dim3(256), 0, st>>>(sum);
    return check_launch("qfa_attn_bwd (sum)");
  };
  if (plan.sum_between) {   // dQ's parts take the place of these
    if (int e = launch_bwd_pair<T, D>(k, plan.blocks_dkv, plan.splits_dkv, a, plan.blocks_dq, 0, BH, x.causal, st)) return e;
    if (int e = add_parts()) return e;
    part = parts;
    sum.count = 0;
    blocks = 0;
  }
  BwdArgs q = a;
  q.per_split = plan.keys_per_split;
  q.last_part = (plan.splits_dq - 1) * plan.keys_per_split;
  q.split_stride = 0;
  if (plan.splits_dq > 1) {
    split(q.dq, q.sdqb, q.sdqh, q.sdqn, x.Nq, plan.splits_dq);
    q.split_stride = x.Nq * D;
    q.grad_f32 = 1;
  }
  if (int e = launch_bwd_pair<T, D>(k, plan.blocks_dkv, plan.sum_between ? 0 : plan.splits_dkv, q, plan.blocks_dq, plan.splits_dq, BH, x.causal, st)) return e;
  return add_parts();
}

int launch_bwd(const AttnArgs &x, hipStream_t st) {
  if (x.io_dtype == QFA_BF16) {
    if (x.D == 256) return launch_bwd_td<__bf16, 256>(x, st);
    if (x.D == 128) return launch_bwd_td<__bf16, 128>(x, st);
    if (x.D == 64) return launch_bwd_td<__bf16, 64>(x, st);
  } else if (x.io_dtype == QFA_F16) {
    if (x.D == 256) return launch_bwd_td<_Float16, 256>(x, st);
    if (x.D == 128) return launch_bwd_td<_Float16, 128>(x, st);
    if (x.D == 64) return launch_bwd_td<_Float16, 64>(x, st);
  } else {
    return set_error(QFA_EINVAL, "attn_bwd: io_dtype must be QFA_BF16 or QFA_F16");
  }
  return set_error(QFA_EUNSUPPORTED, "attn_bwd: head_dim must be 64, 128 or 256");
}

}  // namespace qfa
