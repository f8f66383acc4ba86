// Per-token asymmetric INT8 quantizer and its inverse for gfx950.
//
// Arithmetic contract (asymmetric_quant.py:66-106 of the reference): per token row,
//   scale = (max - min) / 255 (1 if 0);  zp = clamp(roundf(-128 - min/scale));
//   code  = clamp(roundf(x/scale + zp)),  every step one IEEE binary32 operation.
// This file is compiled with -ffp-contract=off and without fast-math so that `/` is the
// correctly rounded division and nothing is fused or re-associated: codes and zero points
// are bit-identical to a CPU evaluation of the same expressions.
//
// Mapping: a token of D elements is held by D/16 adjacent lanes, each with two pieces of 8 elements D/2 apart, so that a
// load instruction covers half rows in 16-byte accesses next to each other (two for fp32).  Head dimensions up to 32 and
// those that are not a power of two take D/8 lanes of one piece, rounded up to a power of two; the idle lanes hold a second
// copy of the token's first eight elements, which changes no minimum or maximum, and neither add to the row sum nor store
// (the reference masks its tail lanes the same way, asymmetric_quant.py:72-75,97-99).  The row is read once, kept in
// registers, reduced with DPP lane permutes inside the lane group, and the codes leave as 8-byte stores.  HBM-bound in
// principle (D*sizeof(in) + D + 9 bytes per token, +2 with the 16-bit scale copy); the exact arithmetic is about as long, so
// the instruction count is kept low (see the division and packing notes in qfa_quant_row.h): what a row costs once, every
// lane of its group computes, hence 16 elements per lane (256 heads of 4096 x 128 binary16: 76 us with 8, 71 us with 16,
// 405 MB at 5.7 TB/s).
#include "qfa_host.h"
#include "qfa_quant_row.h"

namespace qfa {

struct QuantArgs {
  const void *x;
  int8_t *codes;
  float *scale;
  void *scale_lp;
  int8_t *zp;
  int32_t *rowsum;
  int64_t N;
  int64_t H;
  int64_t sxb, sxh, sxn, scb, sch, scn;
  int chunks_per_bh;  // ceil(N / tokens per block)
  int scale_lp_dtype;
  int D;              // head dimension (a multiple of 8, at most the kernel's DP)
};

// A lane's elements: two pieces of eight where every lane of the group is full
template <int DP, bool PARTIAL> constexpr int quant_e() { return DP >= 64 && !PARTIAL ? 16 : 8; }
template <int E> constexpr int quant_u() { return 32 / E; }   // rows a lane holds at once

// One block = 256 threads = U passes over 256/LPT tokens of one (b,h) slice.  DP = the head dimension
// rounded up to a power of two; PARTIAL: the head dimension is smaller than DP.
template <typename T, int DP, bool PARTIAL>
__device__ __forceinline__ void quant_block(const QuantArgs &a, unsigned block) {
  constexpr int E = quant_e<DP, PARTIAL>(), U = quant_u<E>();
  constexpr int LPT = DP / E;         // lanes per token
  constexpr int TPP = 256 / LPT;      // tokens per pass
  const int tid = threadIdx.x;
  const int sub = tid % LPT;
  const bool lane_used = !PARTIAL || sub * 8 < a.D;
  const int sub_ld = lane_used ? sub : 0;   // idle lanes duplicate the token's first eight elements
  const int64_t bh = block / a.chunks_per_bh;
  const int64_t chunk = block % a.chunks_per_bh;
  const int64_t b = bh / a.H, h = bh % a.H;
  const int64_t n0 = chunk * (int64_t)(TPP * U) + tid / LPT;
  const T *xb = reinterpret_cast<const T *>(a.x) + b * a.sxb + h * a.sxh;
  int8_t *cb = a.codes + b * a.scb + h * a.sch;

  float v[U][E];
  bool live[U];
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const int64_t n = n0 + (int64_t)u * TPP;
    live[u] = n < a.N;
    const int64_t nn = live[u] ? n : a.N - 1;   // tail lanes re-read the last token, never store
#pragma unroll
    for (int p = 0; p < E / 8; ++p) {
      float piece[8];
      Load8<T>::run(xb + nn * a.sxn + p * (DP / 2) + sub_ld * 8, piece);
#pragma unroll
      for (int e = 0; e < 8; ++e) v[u][8 * p + e] = piece[e];
    }
  }
  // the per-token results leave through LDS, one token per lane: stored by the lanes that hold them, every store
  // instruction would carry four tokens (128 columns; 256 heads of 4096 x 128 binary16: 81 -> 76 us)
  __shared__ float s_scale[TPP * U];
  __shared__ int s_sum[TPP * U];
  __shared__ int8_t s_zp[TPP * U];
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const int64_t n = n0 + (int64_t)u * TPP;
    const QuantRow<E> r = quant_row<LPT, sizeof(T) == 2, E>(v[u], !PARTIAL || lane_used);
    if (live[u] && lane_used) {
#pragma unroll
      for (int p = 0; p < E / 8; ++p)
        *reinterpret_cast<u32x2 *>(cb + n * a.scn + p * (DP / 2) + sub * 8) = u32x2{r.codes[2 * p], r.codes[2 * p + 1]};
    }
    if (sub == 0) {
      s_scale[u * TPP + tid / LPT] = r.scale;
      s_sum[u * TPP + tid / LPT] = r.sum;
      s_zp[u * TPP + tid / LPT] = (int8_t)(int)r.zp;
    }
  }
  __syncthreads();
  static_assert(TPP * U == 8192 / DP && TPP * U <= 256, "one token per thread, the launcher's count of them");
  const int64_t n = chunk * (int64_t)(TPP * U) + tid;
  if (tid < TPP * U && n < a.N) {
    const int64_t t = bh * a.N + n;
    const float scale = s_scale[tid];
    if (a.scale) a.scale[t] = scale;
    a.zp[t] = s_zp[tid];
    if (a.rowsum) a.rowsum[t] = s_sum[tid];
    if (a.scale_lp) {
      if (a.scale_lp_dtype == QFA_F16) reinterpret_cast<_Float16 *>(a.scale_lp)[t] = (_Float16)scale;
      else reinterpret_cast<__bf16 *>(a.scale_lp)[t] = (__bf16)scale;
    }
  }
}

template <typename T, int DP, bool PARTIAL> __global__ __launch_bounds__(256) void quant_kernel(QuantArgs a) {
  quant_block<T, DP, PARTIAL>(a, blockIdx.x);
}
// Two tensors of one element type and head dimension in one launch (the queries and the keys of an attention call):
// the first blocks0 workgroups take tensor 0, the others tensor 1.  One launch ramp and one tail instead of two.
struct QuantPairArgs {
  QuantArgs t[2];
  unsigned blocks0;
};
template <typename T, int DP, bool PARTIAL> __global__ __launch_bounds__(256) void quant_pair_kernel(QuantPairArgs p) {
  if (blockIdx.x < p.blocks0) quant_block<T, DP, PARTIAL>(p.t[0], blockIdx.x);
  else quant_block<T, DP, PARTIAL>(p.t[1], blockIdx.x - p.blocks0);
}

// The same for fp32 queries and keys with the conversion of the values to bf16 behind them: what an fp32 attention call needs,
// in one launch.  A block takes as many tokens of the values as of the others.
struct QuantQkvArgs {
  QuantPairArgs p;
  unsigned blocks1;     // of the pair
  const float *v;
  __bf16 *v16;          // dense
  int64_t svb, svh, svn;
};
template <int D> __global__ __launch_bounds__(256) void quant_qkv_kernel(QuantQkvArgs a) {
  if (blockIdx.x < a.p.blocks0) {
    quant_block<float, D, false>(a.p.t[0], blockIdx.x);
  } else if (blockIdx.x < a.blocks1) {
    quant_block<float, D, false>(a.p.t[1], blockIdx.x - a.p.blocks0);
  } else {
    constexpr int TOK = 8192 / D;
    const QuantArgs &k = a.p.t[1];   // (the values have the keys' sizes)
    const unsigned block = blockIdx.x - a.blocks1;
    const int64_t bh = block / k.chunks_per_bh, n0 = (int64_t)(block % k.chunks_per_bh) * TOK;
    const float *v = a.v + bh / k.H * a.svb + bh % k.H * a.svh;
    __bf16 *out = a.v16 + bh * k.N * D;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int at = (threadIdx.x + 256 * i) * 8;
      const int64_t n = n0 + at / D;
      if (n < k.N) {
        const f32x4 *src = reinterpret_cast<const f32x4 *>(v + n * a.svn + at % D);
        const f32x4 x = src[0], y = src[1];
        *reinterpret_cast<u32x4 *>(out + n * D + at % D) =
            u32x4{pack2<__bf16>(x[0], x[1]), pack2<__bf16>(x[2], x[3]), pack2<__bf16>(y[0], y[1]), pack2<__bf16>(y[2], y[3])};
      }
    }
  }
}

template <typename T, int DP> static int launch_quant_d(const QuantArgs &a0, int64_t BH, hipStream_t st) {
  constexpr int TOK = 8192 / DP;   // tokens per workgroup, however they are held
  QuantArgs a = a0;
  const int64_t chunks = (a.N + TOK - 1) / TOK;
  if (chunks * BH > 0x7fffffffLL) return set_error(QFA_EUNSUPPORTED, "quant: too many tokens for one launch");
  a.chunks_per_bh = (int)chunks;
  const dim3 grid((unsigned)(chunks * BH)), block(256);
  if (a.D == DP) quant_kernel<T, DP, false><<<grid, block, 0, st>>>(a);
  else quant_kernel<T, DP, true><<<grid, block, 0, st>>>(a);
  return check_launch("qfa_quant_per_token");
}
// head dimension rounded up to a power of two (the lane groups the reductions run over), 32 at least
static int padded_head_dim(int D) { return D <= 32 ? 32 : D <= 64 ? 64 : D <= 128 ? 128 : 256; }
template <typename T> static int launch_quant_t(const QuantArgs &a, int64_t BH, hipStream_t st) {
  switch (padded_head_dim(a.D)) {
    case 32: return launch_quant_d<T, 32>(a, BH, st);
    case 64: return launch_quant_d<T, 64>(a, BH, st);
    case 128: return launch_quant_d<T, 128>(a, BH, st);
  }
  return launch_quant_d<T, 256>(a, BH, st);
}

int launch_quant(const void *x, int x_dtype, int8_t *codes, float *scale, void *scale_lp, int scale_lp_dtype,
                 int8_t *zp, int32_t *rowsum, int64_t B, int64_t H, int64_t N, int D, int64_t sxb, int64_t sxh,
                 int64_t sxn, int64_t scb, int64_t sch, int64_t scn, hipStream_t st) {
  QuantArgs a;
  a.x = x; a.codes = codes; a.scale = scale; a.scale_lp = scale_lp; a.zp = zp; a.rowsum = rowsum;
  a.N = N; a.H = H; a.sxb = sxb; a.sxh = sxh; a.sxn = sxn; a.scb = scb; a.sch = sch; a.scn = scn;
  a.chunks_per_bh = 0; a.scale_lp_dtype = scale_lp_dtype; a.D = D;
  if (D < 8 || D > 256 || D % 8 != 0) return set_error(QFA_EUNSUPPORTED, "quant: head_dim must be a multiple of 8, at most 256");
  switch (x_dtype) {
    case QFA_F32: return launch_quant_t<float>(a, B * H, st);
    case QFA_F16: return launch_quant_t<_Float16>(a, B * H, st);
    case QFA_BF16: return launch_quant_t<__bf16>(a, B * H, st);
  }
  return set_error(QFA_EINVAL, "quant: bad x_dtype");
}

template <typename T, int DP> static int launch_quant_pair_d(QuantPairArgs p, int64_t BH, hipStream_t st) {
  constexpr int TOK = 8192 / DP;   // tokens per workgroup, however they are held
  int64_t blocks[2];
  for (int i = 0; i < 2; ++i) {
    const int64_t chunks = (p.t[i].N + TOK - 1) / TOK;
    p.t[i].chunks_per_bh = (int)chunks;
    blocks[i] = chunks * BH;
  }
  if (blocks[0] + blocks[1] > 0x7fffffffLL) return set_error(QFA_EUNSUPPORTED, "quant_pair: too many tokens for one launch");
  p.blocks0 = (unsigned)blocks[0];
  const dim3 grid((unsigned)(blocks[0] + blocks[1])), block(256);
  if (p.t[0].D == DP) quant_pair_kernel<T, DP, false><<<grid, block, 0, st>>>(p);
  else quant_pair_kernel<T, DP, true><<<grid, block, 0, st>>>(p);
  return check_launch("qfa_quant_per_token_pair");
}
template <typename T> static int launch_quant_pair_t(const QuantPairArgs &p, int64_t BH, hipStream_t st) {
  switch (padded_head_dim(p.t[0].D)) {
    case 32: return launch_quant_pair_d<T, 32>(p, BH, st);
    case 64: return launch_quant_pair_d<T, 64>(p, BH, st);
    case 128: return launch_quant_pair_d<T, 128>(p, BH, st);
  }
  return launch_quant_pair_d<T, 256>(p, BH, st);
}

int launch_quant_pair(const void *const x[2], int x_dtype, int8_t *const codes[2], float *const scale[2],
                      int8_t *const zp[2], int32_t *const rowsum[2], int64_t B, int64_t H, const int64_t N[2], int D,
                      const int64_t sx[2][3], const int64_t sc[2][3], hipStream_t st) {
  QuantPairArgs p;
  for (int i = 0; i < 2; ++i) {
    QuantArgs &a = p.t[i];
    a.x = x[i]; a.codes = codes[i]; a.scale = scale[i]; a.scale_lp = nullptr; a.zp = zp[i]; a.rowsum = rowsum[i];
    a.N = N[i]; a.H = H; a.sxb = sx[i][0]; a.sxh = sx[i][1]; a.sxn = sx[i][2];
    a.scb = sc[i][0]; a.sch = sc[i][1]; a.scn = sc[i][2];
    a.chunks_per_bh = 0; a.scale_lp_dtype = 0; a.D = D;
  }
  p.blocks0 = 0;
  switch (x_dtype) {
    case QFA_F32: return launch_quant_pair_t<float>(p, B * H, st);
    case QFA_F16: return launch_quant_pair_t<_Float16>(p, B * H, st);
    case QFA_BF16: return launch_quant_pair_t<__bf16>(p, B * H, st);
  }
  return set_error(QFA_EINVAL, "quant_pair: bad x_dtype");
}

template <int D> static int launch_quant_qkv_d(QuantQkvArgs a, int64_t BH, hipStream_t st) {
  constexpr int TOK = 8192 / D;
  int64_t blocks[2];
  for (int i = 0; i < 2; ++i) {
    const int64_t chunks = (a.p.t[i].N + TOK - 1) / TOK;
    a.p.t[i].chunks_per_bh = (int)chunks;
    blocks[i] = chunks * BH;
  }
  const int64_t total = blocks[0] + 2 * blocks[1];
  if (total > 0x7fffffffLL) return set_error(QFA_EUNSUPPORTED, "quant_qkv: too many tokens for one launch");
  a.p.blocks0 = (unsigned)blocks[0];
  a.blocks1 = (unsigned)(blocks[0] + blocks[1]);
  quant_qkv_kernel<D><<<dim3((unsigned)total), dim3(256), 0, st>>>(a);
  return check_launch("qfa_quant_qkv_f32");
}
int launch_quant_qkv(const float *const x[2], int8_t *const codes[2], float *const scale[2], int8_t *const zp[2],
                     int32_t *const rowsum[2], const float *v, void *v16, int64_t B, int64_t H, const int64_t N[2], int D,
                     const int64_t sx[2][3], const int64_t sc[2][3], const int64_t sv[3], hipStream_t st) {
  QuantQkvArgs q;
  for (int i = 0; i < 2; ++i) {
    QuantArgs &a = q.p.t[i];
    a.x = x[i]; a.codes = codes[i]; a.scale = scale[i]; a.scale_lp = nullptr; a.zp = zp[i]; a.rowsum = rowsum[i];
    a.N = N[i]; a.H = H; a.sxb = sx[i][0]; a.sxh = sx[i][1]; a.sxn = sx[i][2];
    a.scb = sc[i][0]; a.sch = sc[i][1]; a.scn = sc[i][2];
    a.chunks_per_bh = 0; a.scale_lp_dtype = 0; a.D = D;
  }
  q.p.blocks0 = q.blocks1 = 0;
  q.v = v; q.v16 = static_cast<__bf16 *>(v16);
  q.svb = sv[0]; q.svh = sv[1]; q.svn = sv[2];
  if (D == 256) return launch_quant_qkv_d<256>(q, B * H, st);
  if (D == 128) return launch_quant_qkv_d<128>(q, B * H, st);
  return launch_quant_qkv_d<64>(q, B * H, st);
}

// ---------------------------------------------------------------------------------------------
// Dequantize: out = (code - zp) * scale  (asymmetric_quant.py:160), 8 elements per lane.
struct DequantArgs {
  const int8_t *codes;
  const void *scale;
  const int8_t *zp;
  void *out;
  int64_t N, H;
  int64_t scb, sch, scn, sob, soh, son;
  int chunks_per_bh;
  int scale_dtype;
  int D;   // head dimension (a multiple of 8, at most the kernel's DP)
};

template <typename TO, int DP> __global__ __launch_bounds__(256) void dequant_kernel(DequantArgs a) {
  constexpr int LPT = DP / 8;
  constexpr int TPP = 256 / LPT;
  const int tid = threadIdx.x;
  const int sub = tid % LPT;
  const int64_t bh = blockIdx.x / a.chunks_per_bh;
  const int64_t chunk = blockIdx.x % a.chunks_per_bh;
  const int64_t b = bh / a.H, h = bh % a.H;
  const int64_t n = chunk * (int64_t)TPP + tid / LPT;
  if (n >= a.N || sub * 8 >= a.D) return;
  const int64_t t = bh * a.N + n;
  float scale;
  if (a.scale_dtype == QFA_F32) scale = reinterpret_cast<const float *>(a.scale)[t];
  else if (a.scale_dtype == QFA_F16) scale = (float)reinterpret_cast<const _Float16 *>(a.scale)[t];
  else scale = (float)reinterpret_cast<const __bf16 *>(a.scale)[t];
  const float zp = (float)a.zp[t];
  const u32x2 w = *reinterpret_cast<const u32x2 *>(a.codes + b * a.scb + h * a.sch + n * a.scn + sub * 8);
  float f[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const int c = (int)(int8_t)((w[e / 4] >> (8 * (e % 4))) & 0xff);
    f[e] = ((float)c - zp) * scale;
  }
  TO *o = reinterpret_cast<TO *>(a.out) + b * a.sob + h * a.soh + n * a.son + sub * 8;
  if constexpr (sizeof(TO) == 4) {
    f32x4 lo = {f[0], f[1], f[2], f[3]}, hi = {f[4], f[5], f[6], f[7]};
    reinterpret_cast<f32x4 *>(o)[0] = lo;
    reinterpret_cast<f32x4 *>(o)[1] = hi;
  } else {
    u32x4 p;
#pragma unroll
    for (int e = 0; e < 4; ++e) p[e] = pack2<TO>(f[2 * e], f[2 * e + 1]);
    *reinterpret_cast<u32x4 *>(o) = p;
  }
}

template <typename TO> static int launch_dequant_t(DequantArgs a, int D, int64_t BH, hipStream_t st) {
  if (D < 8 || D > 256 || D % 8 != 0) return set_error(QFA_EUNSUPPORTED, "dequant: head_dim must be a multiple of 8, at most 256");
  a.D = D;
  D = padded_head_dim(D);
  const int tpp = 256 / (D / 8);
  const int64_t chunks = (a.N + tpp - 1) / tpp;
  if (chunks * BH > 0x7fffffffLL) return set_error(QFA_EUNSUPPORTED, "dequant: too many tokens for one launch");
  a.chunks_per_bh = (int)chunks;
  const dim3 grid((unsigned)(chunks * BH)), block(256);
  switch (D) {
    case 32: dequant_kernel<TO, 32><<<grid, block, 0, st>>>(a); break;
    case 64: dequant_kernel<TO, 64><<<grid, block, 0, st>>>(a); break;
    case 128: dequant_kernel<TO, 128><<<grid, block, 0, st>>>(a); break;
    case 256: dequant_kernel<TO, 256><<<grid, block, 0, st>>>(a); break;
    default: return set_error(QFA_EUNSUPPORTED, "dequant: head_dim must be a multiple of 8, at most 256");
  }
  return check_launch("qfa_dequant_per_token");
}

int launch_dequant(const int8_t *codes, const void *scale, int scale_dtype, const int8_t *zp, void *out,
                   int out_dtype, int64_t B, int64_t H, int64_t N, int D, int64_t scb, int64_t sch, int64_t scn,
                   int64_t sob, int64_t soh, int64_t son, hipStream_t st) {
  DequantArgs a;
  a.codes = codes; a.scale = scale; a.zp = zp; a.out = out; a.N = N; a.H = H;
  a.scb = scb; a.sch = sch; a.scn = scn; a.sob = sob; a.soh = soh; a.son = son;
  a.chunks_per_bh = 0; a.scale_dtype = scale_dtype; a.D = D;
  switch (out_dtype) {
    case QFA_F32: return launch_dequant_t<float>(a, D, B * H, st);
    case QFA_F16: return launch_dequant_t<_Float16>(a, D, B * H, st);
    case QFA_BF16: return launch_dequant_t<__bf16>(a, D, B * H, st);
  }
  return set_error(QFA_EINVAL, "dequant: bad out_dtype");
}

// ---------------------------------------------------------------------------------------------
// Row sums of given codes: rowsum[t] = sum_d codes[t][d], the side output the quantizer emits, for codes that
// arrive already quantized (the zero-point term of the INT8 score product needs them).
struct RowsumArgs {
  const int8_t *codes;
  int32_t *rowsum;
  int64_t N, H;
  int64_t scb, sch, scn;
  int chunks_per_bh;
  int D;
};

// Four tokens per lane group, all loads before any sum: with one 8-byte load per lane the kernel waited for memory
// (64 heads of 7001 x 128: 19.6 us).
constexpr int ROWSUM_U = 4;
template <int DP> __global__ __launch_bounds__(256) void rowsum_kernel(RowsumArgs a) {
  constexpr int LPT = DP / 8;
  constexpr int TPP = 256 / LPT;
  const int tid = threadIdx.x;
  const int sub = tid % LPT;
  const int64_t bh = blockIdx.x / a.chunks_per_bh;
  const int64_t chunk = blockIdx.x % a.chunks_per_bh;
  const int64_t b = bh / a.H, h = bh % a.H;
  const int64_t n0 = chunk * (int64_t)(TPP * ROWSUM_U) + tid / LPT;
  const bool used = sub * 8 < a.D;
  u32x2 w[ROWSUM_U];
#pragma unroll
  for (int u = 0; u < ROWSUM_U; ++u) {
    const int64_t n = n0 + u * TPP, nn = n < a.N ? n : a.N - 1;   // every lane takes part in the reduction
    w[u] = *reinterpret_cast<const u32x2 *>(a.codes + b * a.scb + h * a.sch + nn * a.scn + (used ? sub * 8 : 0));
  }
#pragma unroll
  for (int u = 0; u < ROWSUM_U; ++u) {
    const int64_t n = n0 + u * TPP;
    int sum = (int)__builtin_amdgcn_sad_u8(w[u][0] ^ 0x80808080u, 0u, 0u);   // biased bytes: code + 128
    sum = (int)__builtin_amdgcn_sad_u8(w[u][1] ^ 0x80808080u, 0u, (unsigned)sum) - 8 * 128;
    sum = group_sum<LPT>(used ? sum : 0);
    if (n < a.N && sub == 0) a.rowsum[bh * a.N + n] = sum;
  }
}

int launch_rowsum(const int8_t *codes, int32_t *rowsum, int64_t B, int64_t H, int64_t N, int D, int64_t scb,
                  int64_t sch, int64_t scn, hipStream_t st) {
  if (D < 8 || D > 256 || D % 8 != 0) return set_error(QFA_EUNSUPPORTED, "code_rowsum: head_dim must be a multiple of 8, at most 256");
  RowsumArgs a;
  a.codes = codes; a.rowsum = rowsum; a.N = N; a.H = H; a.scb = scb; a.sch = sch; a.scn = scn; a.D = D;
  const int DP = padded_head_dim(D);
  const int tpb = 256 / (DP / 8) * ROWSUM_U;   // tokens per block
  const int64_t chunks = (N + tpb - 1) / tpb;
  if (chunks * B * H > 0x7fffffffLL) return set_error(QFA_EUNSUPPORTED, "code_rowsum: too many tokens for one launch");
  a.chunks_per_bh = (int)chunks;
  const dim3 grid((unsigned)(chunks * B * H)), block(256);
  switch (DP) {
    case 32: rowsum_kernel<32><<<grid, block, 0, st>>>(a); break;
    case 64: rowsum_kernel<64><<<grid, block, 0, st>>>(a); break;
    case 128: rowsum_kernel<128><<<grid, block, 0, st>>>(a); break;
    default: rowsum_kernel<256><<<grid, block, 0, st>>>(a); break;
  }
  return check_launch("qfa_code_rowsum");
}

// ---------------------------------------------------------------------------------------------
// What the INT8-score forward needs of an INT8 K / V cache, in one launch: the row sums of K and its scales in fp32, V
// dequantized, and (where the caller has them) the queries quantized.  Bound by memory (5 bytes per element of K and V; 64 heads of
// 7001 x 128: 229 MB in 40 us).  Four tokens per lane group, all loads before any result, as in rowsum_kernel.  The queries' workgroups
// come first and go under in the rest: as a launch of their own 333 of these heads' queries were 5 us (the whole call 147 -> 142 us).
struct CacheStageArgs {
  QuantArgs q;
  int blocks_q;        // workgroups of the queries (none: 0)
  const int8_t *kc, *vc;
  const void *ks, *vs;
  const int8_t *vz;
  float *ks32;         // nullable
  int32_t *rowsum;
  void *v;             // dense
  int64_t N, H;
  int64_t skb, skh, skn, svb, svh, svn;
  int chunks_per_bh, blocks_k, ks_dtype, vs_dtype;
};
// T: type of the queries
template <typename T, typename TO, int D> __global__ __launch_bounds__(256) void cache_stage_kernel(CacheStageArgs a) {
  if ((int)blockIdx.x < a.blocks_q) {
    quant_block<T, D, false>(a.q, blockIdx.x);
    return;
  }
  constexpr int LPT = D / 8, TPP = 256 / LPT, U = 4;
  const int tid = threadIdx.x, sub = tid % LPT;
  const unsigned block = blockIdx.x - a.blocks_q;
  const bool is_k = (int)block < a.blocks_k;
  const unsigned blk = is_k ? block : block - a.blocks_k;
  const unsigned bh = blk / (unsigned)a.chunks_per_bh, chunk = blk - bh * a.chunks_per_bh;
  const int64_t b = index_div(bh, a.H), h = bh - b * a.H;
  const int64_t n0 = (int64_t)chunk * (TPP * U) + tid / LPT, t0 = (int64_t)bh * a.N;
  const int8_t *c = (is_k ? a.kc + b * a.skb + h * a.skh : a.vc + b * a.svb + h * a.svh) + sub * 8;
  const int64_t sn = is_k ? a.skn : a.svn;
  u32x2 w[U];
  int64_t n[U];
#pragma unroll
  for (int u = 0; u < U; ++u) {
    n[u] = n0 + u * TPP < a.N ? n0 + u * TPP : a.N - 1;   // every lane takes part in the reduction
    w[u] = *reinterpret_cast<const u32x2 *>(c + n[u] * sn);
  }
  if (is_k) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      int sum = (int)__builtin_amdgcn_sad_u8(w[u][0] ^ 0x80808080u, 0u, 0u);   // biased bytes: code + 128
      sum = (int)__builtin_amdgcn_sad_u8(w[u][1] ^ 0x80808080u, 0u, (unsigned)sum) - 8 * 128;
      sum = group_sum<LPT>(sum);
      if (n0 + u * TPP >= a.N || sub != 0) continue;
      a.rowsum[t0 + n[u]] = sum;
      if (a.ks32)
        a.ks32[t0 + n[u]] = a.ks_dtype == QFA_F16 ? (float)static_cast<const _Float16 *>(a.ks)[t0 + n[u]]
                                                  : (float)static_cast<const __bf16 *>(a.ks)[t0 + n[u]];
    }
    return;
  }
  float scale[U], zp[U];
  if (a.vs_dtype == QFA_F32) {
#pragma unroll
    for (int u = 0; u < U; ++u) scale[u] = static_cast<const float *>(a.vs)[t0 + n[u]];
  } else if (a.vs_dtype == QFA_F16) {
#pragma unroll
    for (int u = 0; u < U; ++u) scale[u] = (float)static_cast<const _Float16 *>(a.vs)[t0 + n[u]];
  } else {
#pragma unroll
    for (int u = 0; u < U; ++u) scale[u] = (float)static_cast<const __bf16 *>(a.vs)[t0 + n[u]];
  }
#pragma unroll
  for (int u = 0; u < U; ++u) zp[u] = (float)a.vz[t0 + n[u]];
#pragma unroll
  for (int u = 0; u < U; ++u) {
    if (n0 + u * TPP >= a.N) break;
    u32x4 p;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const unsigned x = w[u][e / 2] >> (16 * (e % 2));
      p[e] = pack2<TO>(((float)(int)(int8_t)(x & 0xff) - zp[u]) * scale[u], ((float)(int)(int8_t)(x >> 8 & 0xff) - zp[u]) * scale[u]);
    }
    *reinterpret_cast<u32x4 *>(static_cast<TO *>(a.v) + (t0 + n[u]) * D + sub * 8) = p;
  }
}
template <typename T, typename TO, int D> static int launch_cache_stage_td(CacheStageArgs a, int64_t BH, hipStream_t st) {
  constexpr int TOK = 8192 / D;   // tokens per workgroup
  const int64_t chunks = (a.N + TOK - 1) / TOK, chunks_q = (a.q.N + TOK - 1) / TOK, total = (2 * chunks + chunks_q) * BH;
  if (total > 0x7fffffffLL) return set_error(QFA_EUNSUPPORTED, "cache_stage: too many tokens for one launch");
  a.chunks_per_bh = (int)chunks;
  a.blocks_k = (int)(chunks * BH);
  a.q.chunks_per_bh = (int)chunks_q;
  a.blocks_q = (int)(chunks_q * BH);
  cache_stage_kernel<T, TO, D><<<dim3((unsigned)total), dim3(256), 0, st>>>(a);
  return check_launch("qfa_cache_stage");
}
template <typename T, typename TO> static int launch_cache_stage_t(const CacheStageArgs &a, int D, int64_t BH, hipStream_t st) {
  if (D == 64) return launch_cache_stage_td<T, TO, 64>(a, BH, st);
  if (D == 128) return launch_cache_stage_td<T, TO, 128>(a, BH, st);
  return launch_cache_stage_td<T, TO, 256>(a, BH, st);
}
int launch_cache_stage(const QuantizeQ *q, const int8_t *kc, const void *ks, int ks_dtype, float *ks32, int32_t *rowsum, const int8_t *vc,
                       const void *vs, int vs_dtype, const int8_t *vz, void *v, int v_dtype, int64_t B, int64_t H, int64_t N, int D,
                       const int64_t sk[3], const int64_t sv[3], hipStream_t st) {
  QuantArgs x = {};   // no queries
  if (q) {
    x.x = q->x; x.codes = q->codes; x.scale = q->scale; x.zp = q->zp; x.rowsum = q->rowsum; x.N = q->N; x.H = H; x.D = D;
    x.sxb = q->sx[0]; x.sxh = q->sx[1]; x.sxn = q->sx[2]; x.scb = q->sc[0]; x.sch = q->sc[1]; x.scn = q->sc[2];
  }
  const CacheStageArgs a = {x, 0, kc, vc, ks, vs, vz, ks32, rowsum, v, N, H, sk[0], sk[1], sk[2], sv[0], sv[1], sv[2], 0, 0, ks_dtype, vs_dtype};
  if (q && q->dtype == QFA_F32) return launch_cache_stage_t<float, __bf16>(a, D, B * H, st);
  if (v_dtype == QFA_BF16) return launch_cache_stage_t<__bf16, __bf16>(a, D, B * H, st);
  return launch_cache_stage_t<_Float16, _Float16>(a, D, B * H, st);
}

}  // namespace qfa
