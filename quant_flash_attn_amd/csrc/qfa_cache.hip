// Attention of a short block of queries on an INT8 cache of keys and values (decoding: one query per (batch, head), or a
// few).  K and V are two quantized tensors; the scores are those of qfa_attn_fwd -- the queries are quantized per token
// here, by the quantizer's own arithmetic, and Q K^T runs on INT8 MFMA with the exact zero-point term -- and V enters as
// its exact codes:
//     O = softmax(sm_scale * Q^ K^^T) V^,   X^ = scale * (codes - zero_point) per token.
// Bound by reading the cache once (2 D + 6 bytes per key).  Through the kernels for long query blocks the same call
// dequantizes V to 16 bits first (2 D more bytes written and read), sums K's codes in a pass of its own and then walks
// each (batch, head) with one workgroup of 128 query rows, nearly all of them padding: B8 H32 Nq1 Nk8192 D128 took 459 us
// that way (dequantize 175, row sums 100, attention 200 with the casts); this kernel and its merge take 83 us (6.6 TB/s of
// cache; 96 before its loads were non-temporal; 35 -> 17.5 for B1).
//
// Work split.  A workgroup = 4 waves = 16 queries of one (batch, head) and a share of its keys (split_plan, qfa_merge.h);
// its 32-key tiles are dealt to the waves, each with its own online softmax.  The tile lives in registers, double-buffered:
// nothing of it is used twice inside a workgroup, so LDS would only add a trip.
//   K    is the A operand of v_mfma_i32_16x16x64_i8 as it lies in memory (lane = key row, 16 bytes of it per k-group); a
//        second product with a column of ones gives the row sums the zero-point term needs.
//   V^T  is the A operand of the P.V product (rows = d, contracted over keys).  A lane loads the D/16 bytes at
//        d = (D/16) * (lane%16) of the eight keys that the score accumulator leaves in its k-group (keys 16rb + 4G + v),
//        and one byte permute plus one XOR turn a pair of keys at one d into two binary16 numbers 1152 + code exactly
//        (qfa_skv_common.h); MFMA i of the D/16 takes byte i, so its row r is d = (D/16) * r + i.
//   The offset 1152 + zero point is removed through sum_j (1152 + zp_j) p'_j, accumulated over the rounded p' = p * scale_j.
//   p' enters the product as binary16, and the scales carry V's magnitude: the reference that p is taken against follows the
//   largest p', not the largest p, so that the largest one seen lies between 2^7 and 2^10, whatever V's size.  (p <= 1 put p'
//   among binary16's subnormals for small V: relative error of O 1.8e-2 at size 1e-3, 1.7e-1 at 1e-4, where dequantizing V
//   first leaves 3e-3 in bf16; and scales above 4e3 overflowed.)
// Per-token scales and zero points pass through 512 bytes of LDS per wave, which turns one load per token into the
// broadcast the accumulator layout wants.
#include <type_traits>

#include "qfa_host.h"
#include "qfa_merge.h"
#include "qfa_quant_row.h"
#include "qfa_skv_common.h"

namespace qfa {

struct CacheArgs {
  const void *q; const int8_t *kc; const void *ks; const int8_t *kz; const int8_t *vc; const void *vs; const int8_t *vz;
  void *o;
  float *lse;          // nullable
  float *po, *pml;     // splits > 1: unnormalised partial results [B*H*Nq][splits][D], and (m in log2 units, l)
  int64_t H;
  int64_t sqb, sqh, sqn, skb, skh, skn, svb, svh, svn, sob, soh, son;
  float sm_scale_log2;
  int Nq, Nk, BH, qblocks, splits, tiles_per_split, causal, q_dtype;
};

// Workgroups per CU that a launch counts on: two tiles in registers (80 of them at head_dim 128, 148 at 256) beside the
// accumulators.  With one tile per wave in flight that keeps 64 KB (48 at head_dim 64) per CU under way.
constexpr int cache_wgs_per_cu(int D) { return D == 256 ? 1 : D == 128 ? 2 : 3; }

// log2 of the largest p' at a new reference, and the p' past which the reference moves.  The key at the reference has an exact
// p' (see `move`), so moving it sooner is more exact: against a reference that moves where p passes 2^4, as in the other
// kernels, the error of fp32 results is 0.85 to 1.0 times as large over head_dim 64, 128 and 256 and all value
// distributions (1.0e-4 to 2.1e-4); moved at 2^15 it is up to 1.38 times as large, moved at 2^9 0.73 to 1.0, for 1 to 3 %
// more time at head_dim 64.
constexpr float CACHE_P_REF = 7.0f, CACHE_P_MAX = 0x1p10f;

__device__ __forceinline__ i32x4 mfma_i8_16(i32x4 a, i32x4 b, i32x4 c) {
  return __builtin_amdgcn_mfma_i32_16x16x64_i8(a, b, c, 0, 0, 0);
}

template <typename S, int D, bool STREAM> __global__ __launch_bounds__(256, D == 64 ? 4 : cache_wgs_per_cu(D)) void cache_fwd_kernel(CacheArgs a) {
  constexpr int HINT = STREAM ? LOAD_ONCE : 0;
  constexpr int KM = D / 64;    // 64-wide k-steps of the score product
  constexpr int DB = D / 16;    // 16-row blocks of O^T
  constexpr int VB = D / 16;    // bytes of a V row per lane
  constexpr int VD = VB / 4;    // ... in dwords
  constexpr int LPT = D / 8, TPP = 256 / LPT;   // quantizer: lanes per token, tokens per pass
  // LDS: query codes and constants, per-wave token constants; the merge of the four waves overlays them
  constexpr int OFF_ST = 16 * D, OFF_TC = OFF_ST + 3 * 16 * 4, MERGE = 4 * 16 * (D + 2) * 4;
  constexpr int TC = 512 + 128;   // per wave: [64] x (scale, zero point operand), exponents of the 32 values' scales
  constexpr int TOTAL = MERGE > OFF_TC + 4 * TC ? MERGE : OFF_TC + 4 * TC;
  __shared__ __attribute__((aligned(16))) unsigned char smem[TOTAL];

  const int per_bh = a.qblocks * a.splits;
  const XcdBlock id(a.BH, per_bh);
  if (!id.live) return;
  const int bh = id.bh, qb = id.sub % a.qblocks, split = id.sub / a.qblocks;
  const int64_t b = bh / a.H, h = bh % a.H;
  const int tid = threadIdx.x, lane = tid % 64, q16 = lane % 16, G = lane / 16;
  const int wave = __builtin_amdgcn_readfirstlane(tid / 64);
  const int nqv = min(16, a.Nq - 16 * qb);
  const int64_t tk0 = (int64_t)bh * a.Nk;

  // keys this block can see, and this wave's tiles: t0 + wave, t0 + wave + 4, ...
  const int first_lim = a.causal ? a.Nk - a.Nq + 16 * qb : a.Nk - 1;   // last key of the block's first query
  const int kv_end = a.causal ? first_lim + nqv : a.Nk;
  const int t0 = split * a.tiles_per_split;
  const int ntiles = min(a.tiles_per_split, (kv_end + SKV_TILE - 1) / SKV_TILE - t0);
  const int my_tiles = ntiles > wave ? (ntiles - wave + 3) / 4 : 0;

  struct Tile {
    i32x4 k[2][KM];
    unsigned v[8][VD];
    unsigned sc, zp;   // scale (its bits) and zero point: lanes 0-31 of key lane, lanes 32-63 of value lane - 32
  };
  const unsigned char *k_bh = reinterpret_cast<const unsigned char *>(a.kc + b * a.skb + h * a.skh);
  const unsigned char *v_bh = reinterpret_cast<const unsigned char *>(a.vc + b * a.svb + h * a.svh);
  const S *sc_l = reinterpret_cast<const S *>(lane < 32 ? a.ks : a.vs) + tk0;
  const int8_t *zp_l = (lane < 32 ? a.kz : a.vz) + tk0;
  const int k_off = q16 * (int)a.skn + 16 * G, v_off = 4 * G * (int)a.svn + VB * q16;
  // (every load is issued whether the tile exists or not -- a missing one has an empty descriptor and fetches nothing --
  // so that the compiler's counted waits see one path)
  auto load = [&](Tile &t, int i) {
    const int tile = t0 + wave + 4 * i;
    const int rows = i < my_tiles ? min(SKV_TILE, a.Nk - tile * SKV_TILE) : 0;
    const rsrc_t rk = make_rsrc(k_bh + (int64_t)tile * SKV_TILE * a.skn, rows > 0 ? (unsigned)((rows - 1) * (int)a.skn + D) : 0u);
    const rsrc_t rv = make_rsrc(v_bh + (int64_t)tile * SKV_TILE * a.svn, rows > 0 ? (unsigned)((rows - 1) * (int)a.svn + D) : 0u);
#pragma unroll
    for (int rb = 0; rb < 2; ++rb)
#pragma unroll
      for (int m = 0; m < KM; ++m)
        t.k[rb][m] = __builtin_bit_cast(
            i32x4, __builtin_amdgcn_raw_buffer_load_b128(rk, k_off + 64 * m, 16 * rb * (int)a.skn, HINT));
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const int soff = (16 * (e / 4) + e % 4) * (int)a.svn;
      if constexpr (VD == 4) {
        const u32x4 w = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rv, v_off, soff, HINT));
#pragma unroll
        for (int x = 0; x < 4; ++x) t.v[e][x] = w[x];
      } else if constexpr (VD == 2) {
        const u32x2 w = __builtin_bit_cast(u32x2, __builtin_amdgcn_raw_buffer_load_b64(rv, v_off, soff, HINT));
        t.v[e][0] = w[0];
        t.v[e][1] = w[1];
      } else {
        t.v[e][0] = (unsigned)__builtin_amdgcn_raw_buffer_load_b32(rv, v_off, soff, HINT);
      }
    }
    const int key = min(tile * SKV_TILE + lane % 32, a.Nk - 1);
    if constexpr (sizeof(S) == 4) t.sc = __builtin_bit_cast(unsigned, sc_l[key]);
    else t.sc = __builtin_bit_cast(unsigned short, sc_l[key]);
    t.zp = (unsigned)(unsigned char)zp_l[key];
  };

  Tile ta, tb;
  load(ta, 0);

  // ---- the block's queries, quantized: codes to LDS, a = scale * sm_scale * log2(e), zero point and c = sum - D * zp
  float *st_a = reinterpret_cast<float *>(smem + OFF_ST);
  int *st_z = reinterpret_cast<int *>(smem + OFF_ST + 64), *st_c = reinterpret_cast<int *>(smem + OFF_ST + 128);
#pragma unroll
  for (int p = 0; p < (16 + TPP - 1) / TPP; ++p) {
    const int tok = p * TPP + tid / LPT, sub = tid % LPT;
    const int64_t off = b * a.sqb + h * a.sqh + (int64_t)min(16 * qb + tok, a.Nq - 1) * a.sqn + sub * 8;
    float v[8];
    if (a.q_dtype == QFA_F32) Load8<float>::run(static_cast<const float *>(a.q) + off, v);
    else if (a.q_dtype == QFA_BF16) Load8<__bf16>::run(static_cast<const __bf16 *>(a.q) + off, v);
    else Load8<_Float16>::run(static_cast<const _Float16 *>(a.q) + off, v);
    const QuantRow<8> r = quant_row<LPT, false, 8>(v, true);
    if (tok < 16) {
      *reinterpret_cast<u32x2 *>(smem + tok * D + sub * 8) = u32x2{r.codes[0], r.codes[1]};
      if (sub == 0) {
        st_a[tok] = r.scale * a.sm_scale_log2;
        st_z[tok] = (int)r.zp;
        st_c[tok] = r.sum - D * (int)r.zp;
      }
    }
  }
  __syncthreads();
  i32x4 qf[KM];
#pragma unroll
  for (int m = 0; m < KM; ++m) qf[m] = *reinterpret_cast<const i32x4 *>(smem + q16 * D + 64 * m + 16 * G);
  const float a_i = st_a[q16];
  const int zq = st_z[q16], c_i = st_c[q16];
  const int qi = 16 * qb + q16;
  const int lim = a.causal ? min(a.Nk - a.Nq + qi, a.Nk - 1) : a.Nk - 1;   // last key of this lane's query

  f32x4 oacc[DB];
#pragma unroll
  for (int i = 0; i < DB; ++i) oacc[i] = f32x4{0.f, 0.f, 0.f, 0.f};
  // p = 2^(a_i * u - ref); a query that sees no key of the wave's first tile sees none later either
  float ref = NO_KEY, l_run = 0.f, w_run = 0.f;
  unsigned *tc = reinterpret_cast<unsigned *>(smem + OFF_TC + wave * TC);
  const i32x4 ones = {0x01010101, 0x01010101, 0x01010101, 0x01010101};

  auto tile = [&](const Tile &t, int i, auto masked_tag) __attribute__((always_inline)) {
    constexpr bool MASKED = decltype(masked_tag)::value;
    // token constants: K (scale, zp as an integer), V (scale, the binary16 number 1152 + zp)
    {
      u32x2 w;
      w[0] = __builtin_bit_cast(unsigned, scale_to_f32<S>(t.sc));
      w[1] = lane < 32 ? (unsigned)(int)(signed char)t.zp : (0x6400u | (t.zp ^ 0x80u));
      *reinterpret_cast<u32x2 *>(tc + 2 * lane) = w;
    }
    // ---- scores of keys 16rb + 4G + v
    f32x4 f[2];
#pragma unroll
    for (int rb = 0; rb < 2; ++rb) {
      i32x4 s = {0, 0, 0, 0}, rk = {0, 0, 0, 0};
#pragma unroll
      for (int m = 0; m < KM; ++m) {
        s = mfma_i8_16(t.k[rb][m], qf[m], s);
        rk = mfma_i8_16(t.k[rb][m], ones, rk);
      }
      const u32x4 c0 = *reinterpret_cast<const u32x4 *>(tc + 2 * (16 * rb + 4 * G)),
                  c1 = *reinterpret_cast<const u32x4 *>(tc + 2 * (16 * rb + 4 * G) + 4);
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const unsigned scw = v < 2 ? c0[2 * v] : c1[2 * v - 4], zw = v < 2 ? c0[2 * v + 1] : c1[2 * v - 3];
        const int x = s[v] - __mul24(zq, rk[v]) - __mul24((int)zw, c_i);
        float u = (float)x * __builtin_bit_cast(float, scw);
        if (MASKED && (t0 + wave + 4 * i) * SKV_TILE + 16 * rb + 4 * G + v > lim) u = -INFINITY;
        f[rb][v] = u;
      }
    }
    // ---- p and its row sum, p' = p * scale_j and the largest of them
    float ps[8], mx = 0.f, l_new = 0.f;
    unsigned zz[4];   // the binary16 numbers 1152 + zero point
    u32x4 cv[4];      // keys 16(x/2) + 4G + 2(x%2) + {0, 1}: scale, 1152 + zero point, and again
    auto load_cv = [&]() __attribute__((always_inline)) {
#pragma unroll
      for (int x = 0; x < 4; ++x) cv[x] = *reinterpret_cast<const u32x4 *>(tc + 2 * (32 + 16 * (x / 2) + 4 * G + 2 * (x % 2)));
    };
    if constexpr (D > 64) load_cv();   // (at 64 the registers of a fourth workgroup per CU are worth more)
    auto probs = [&]() __attribute__((always_inline)) {
      mx = 0.f;
      l_new = l_run;
      if constexpr (D == 64) load_cv();
#pragma unroll
      for (int x = 0; x < 4; ++x) {
        const unsigned s0 = cv[x][0], z0 = cv[x][1], s1 = cv[x][2], z1 = cv[x][3];   // (a bit cast of a vector's element takes element 0)
        zz[x] = z0 | (z1 << 16);
        const float p0 = __builtin_amdgcn_exp2f(__builtin_fmaf(a_i, f[x / 2][2 * (x % 2)], -ref));
        const float p1 = __builtin_amdgcn_exp2f(__builtin_fmaf(a_i, f[x / 2][2 * (x % 2) + 1], -ref));
        l_new += p0 + p1;
        ps[2 * x] = p0 * __builtin_bit_cast(float, s0);
        ps[2 * x + 1] = p1 * __builtin_bit_cast(float, s1);
        mx = fmaxf(mx, fmaxf(fabsf(ps[2 * x]), fabsf(ps[2 * x + 1])));
      }
    };
    // a new reference, common to the four lanes of a query: log2 of the tile's largest p' (and p itself within fp32), but for the
    // scale's mantissa: that key's p is a power of two, and its p' the scale itself, which a binary16 scale is exactly
    auto move = [&]() __attribute__((always_inline)) -> float {
      float *tl = reinterpret_cast<float *>(tc + 128);
      if (lane >= 32) tl[lane - 32] = __builtin_floorf(__builtin_amdgcn_logf(fabsf((*reinterpret_cast<const f32x2 *>(tc + 2 * lane))[0])));
      float t = -INFINITY, u = -INFINITY;
#pragma unroll
      for (int rb = 0; rb < 2; ++rb) {
        const f32x4 ls = *reinterpret_cast<const f32x4 *>(tl + 16 * rb + 4 * G);
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          t = fmaxf(t, __builtin_fmaf(a_i, f[rb][v], ls[v]));
          u = fmaxf(u, f[rb][v]);
        }
      }
      t = fmaxf(t - CACHE_P_REF, __builtin_fmaf(a_i, u, -100.0f));
      t = fmaxf(t, __shfl_xor(t, 16, 64));
      t = fmaxf(t, __shfl_xor(t, 32, 64));
      t = fmaxf(t, ref);
      const float alpha = __builtin_amdgcn_exp2f(ref - t);
      ref = t;
      return alpha;
    };
    if (i == 0) move();   // (nothing summed yet)
    probs();
    if (i != 0 && __builtin_amdgcn_ballot_w64(mx > CACHE_P_MAX || !(l_new <= 0x1p100f)) != 0) {
      const float alpha = move();
      l_run *= alpha;
      w_run *= alpha;
#pragma unroll
      for (int j = 0; j < DB; ++j)
#pragma unroll
        for (int v = 0; v < 4; ++v) oacc[j][v] *= alpha;
      probs();
    }
    l_run = l_new;
    // ---- p' as binary16, offset term
    u32x4 pf;
#pragma unroll
    for (int x = 0; x < 4; ++x) {
      const unsigned pp = pack_h2(ps[2 * x], ps[2 * x + 1]);
      pf[x] = pp;
      w_run = __builtin_amdgcn_fdot2(__builtin_bit_cast(f16x2, pp), __builtin_bit_cast(f16x2, zz[x]), w_run, false);
    }
    // ---- O^T += (1152 + codes)^T . P'^T
#pragma unroll
    for (int j = 0; j < DB; ++j) {
      u32x4 vf;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        constexpr unsigned pick = 0x0c040c00u;
        vf[e] = __builtin_amdgcn_perm(t.v[2 * e + 1][j / 4], t.v[2 * e][j / 4], pick + (unsigned)(j % 4) * 0x00010001u) ^
                0x64806480u;
      }
      oacc[j] = mfma_h16(vf, pf, oacc[j]);
    }
  };
  auto run = [&](const Tile &t, int i) __attribute__((always_inline)) {
    if ((t0 + wave + 4 * i + 1) * SKV_TILE - 1 > first_lim) tile(t, i, std::true_type{});
    else tile(t, i, std::false_type{});
  };
  for (int i = 0; i < my_tiles; i += 2) {
    load(tb, i + 1);
    run(ta, i);
    load(ta, i + 2);
    if (i + 1 < my_tiles) run(tb, i + 1);
  }

  // ---- merge of the four waves, through LDS: [wave][query][D] and (m, l) behind
  float l_tot = l_run + __shfl_xor(l_run, 16, 64), w_tot = w_run + __shfl_xor(w_run, 16, 64);
  l_tot += __shfl_xor(l_tot, 32, 64);
  w_tot += __shfl_xor(w_tot, 32, 64);
  __syncthreads();   // query codes and token constants are done with
  float *mg = reinterpret_cast<float *>(smem), *ml = mg + 4 * 16 * D;
  if (q16 < nqv) {
    float *dst = mg + (wave * 16 + q16) * D;
#pragma unroll
    for (int v = 0; v < 4; ++v)
#pragma unroll
      for (int j = 0; j < DB; j += 4) {
        f32x4 x;
#pragma unroll
        for (int y = 0; y < 4; ++y) x[y] = oacc[j + y][v] - w_tot;
        *reinterpret_cast<f32x4 *>(dst + VB * (4 * G + v) + j) = x;
      }
    if (G == 0) {
      ml[2 * (wave * 16 + q16)] = ref;
      ml[2 * (wave * 16 + q16) + 1] = l_tot;
    }
  }
  __syncthreads();
  for (int x = tid; x < nqv * (D / 4); x += 256) {
    const int q = x / (D / 4), d = 4 * (x % (D / 4));
    float m = NO_KEY, l = 0.f;
#pragma unroll
    for (int w = 0; w < 4; ++w) m = fmaxf(m, ml[2 * (16 * w + q)]);
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      const float s = __builtin_amdgcn_exp2f(ml[2 * (16 * w + q)] - m);
      l += ml[2 * (16 * w + q) + 1] * s;
      const f32x4 y = *reinterpret_cast<const f32x4 *>(mg + (16 * w + q) * D + d);
#pragma unroll
      for (int e = 0; e < 4; ++e) acc[e] += y[e] * s;
    }
    const int qg = 16 * qb + q;
    if (a.splits > 1) {
      const int64_t slot = ((int64_t)bh * a.Nq + qg) * a.splits + split;
      *reinterpret_cast<f32x4 *>(a.po + slot * D + d) = acc;
      if (d == 0) *reinterpret_cast<f32x2 *>(a.pml + 2 * slot) = f32x2{m, l};
    } else {
      const float inv = 1.0f / l;
      if (a.lse && d == 0) a.lse[(int64_t)bh * a.Nq + qg] = (m + __log2f(l)) * kLn2;
      const int64_t off = b * a.sob + h * a.soh + (int64_t)qg * a.son;
      store4(static_cast<char *>(a.o) + off * (a.q_dtype == QFA_F32 ? 4 : 2), a.q_dtype, d,
             f32x4{acc[0] * inv, acc[1] * inv, acc[2] * inv, acc[3] * inv});
    }
  }
}

// How the keys of a query block are split: as many workgroups as are resident at once (cache_wgs_per_cu; a second, partly
// filled round would cost a whole one), or what split_plan finds better
static void cache_split_plan(int64_t BH, int64_t Nq, int64_t Nk, int D, int *splits, int *tiles_per_split) {
  const int64_t wgs = BH * ((Nq + 15) / 16);
  split_plan(wgs, BH * Nq, (Nk + SKV_TILE - 1) / SKV_TILE, D, 256 * cache_wgs_per_cu(D) / wgs, splits, tiles_per_split);
}

int64_t cache_workspace_bytes(int64_t B, int64_t H, int64_t Nq, int64_t Nk, int D) {
  int splits, tps;
  cache_split_plan(B * H, Nq, Nk, D, &splits, &tps);
  return splits > 1 ? split_partial_bytes(B * H * Nq, splits, D) : 0;
}

template <typename S, int D> static int launch_cache_sd(const CacheAttnArgs &x, hipStream_t st) {
  CacheArgs a;
  a.q = x.q; a.kc = x.kc; a.ks = x.ks; a.kz = x.kz; a.vc = x.vc; a.vs = x.vs; a.vz = x.vz; a.o = x.o; a.lse = x.lse;
  a.H = x.H; a.Nq = (int)x.Nq; a.Nk = (int)x.Nk; a.BH = (int)(x.B * x.H);
  a.sqb = x.sqb; a.sqh = x.sqh; a.sqn = x.sqn; a.skb = x.skb; a.skh = x.skh; a.skn = x.skn;
  a.svb = x.svb; a.svh = x.svh; a.svn = x.svn; a.sob = x.sob; a.soh = x.soh; a.son = x.son;
  a.sm_scale_log2 = x.sm_scale * kLog2e;
  a.causal = x.causal; a.q_dtype = x.q_dtype;
  a.qblocks = (int)((x.Nq + 15) / 16);
  a.splits = 1;
  a.tiles_per_split = (int)((x.Nk + SKV_TILE - 1) / SKV_TILE);
  a.po = a.pml = nullptr;
  if (x.workspace) {   // validated: large enough for the plan below
    cache_split_plan(x.B * x.H, x.Nq, x.Nk, D, &a.splits, &a.tiles_per_split);
    a.po = static_cast<float *>(x.workspace);
    a.pml = a.po + x.B * x.H * x.Nq * a.splits * (int64_t)D;
  }
  const int64_t total = xcd_grid(a.BH, (int64_t)a.qblocks * a.splits);
  if (x.B * x.H > 0x7fffffffLL || total > 0x7fffffffLL || x.B * x.H * x.Nq > 0x7fffffffLL)
    return set_error(QFA_EUNSUPPORTED, "attn_fwd_cache: too many query blocks for one launch");
  // Non-temporal loads (LOAD_ONCE), measured over 1400 random calls: from 320 MiB and 1024 keys on, 0.96 of the time at head_dim 64 and 128 on
  // three caches in turn, 0.97 on one and the same; shorter sequences of many heads 1.03 to 1.09, 100 to 256 MiB 0.97 on three caches but
  // 1.06 to 1.1 on one.  Not at 256: 46 calls 0.915 to 1.113, 1.011 in the mean (1.03 with 16 queries: 2083 heads on 1434 keys 321 -> 345 us).
  // 8 x 32 heads, one query on 8192 keys of 128: 95.5 -> 83 us (5.8 -> 6.6 TB/s)
  const bool once = a.qblocks == 1 && x.Nk >= 1024 && 2 * x.B * x.H * x.Nk * D > LAST_LEVEL_BYTES / 4 * 5 &&
                    rows_own_lines(x.kc, x.skb, x.skh, x.skn, D) && rows_own_lines(x.vc, x.svb, x.svh, x.svn, D);
  if (D < 256 && once) cache_fwd_kernel<S, D, (D < 256)><<<dim3((unsigned)total), dim3(256), 0, st>>>(a);
  else cache_fwd_kernel<S, D, false><<<dim3((unsigned)total), dim3(256), 0, st>>>(a);
  if (int e = check_launch("qfa_attn_fwd_cache")) return e;
  if (a.splits > 1) {
    const SplitMergeArgs m = {a.po, a.pml, a.o, a.lse, a.H, a.sob, a.soh, a.son, a.Nq, a.splits, a.q_dtype, nullptr};
    return launch_split_merge<D>(m, x.B * x.H * x.Nq, "qfa_attn_fwd_cache (merge)", st);
  }
  return 0;
}

template <int D> static int launch_cache_d(const CacheAttnArgs &x, hipStream_t st) {
  if (x.scale_dtype == QFA_F32) return launch_cache_sd<float, D>(x, st);
  if (x.scale_dtype == QFA_F16) return launch_cache_sd<_Float16, D>(x, st);
  return launch_cache_sd<__bf16, D>(x, st);
}

int launch_cache_fwd(const CacheAttnArgs &x, hipStream_t st) {
  if (x.D == 256) return launch_cache_d<256>(x, st);
  if (x.D == 128) return launch_cache_d<128>(x, st);
  if (x.D == 64) return launch_cache_d<64>(x, st);
  return set_error(QFA_EUNSUPPORTED, "attn_fwd_cache: head_dim must be 64, 128 or 256");
}

}  // namespace qfa
