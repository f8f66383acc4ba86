// The quantizer's arithmetic on one token row, shared by the stand-alone quantizer and the kernels that quantize their
// queries themselves.  Every step is one IEEE binary32 operation (see qfa_quant.hip): the file that includes this is
// compiled with -ffp-contract=off.
#pragma once
#include "qfa_device.h"

namespace qfa {

// Minimum and maximum over the LPT lanes of a token.  One reduction step = one instruction: the lane permute is the DPP
// modifier of the min / max itself.  (Written as asm: through the builtin the permuted value comes back as an integer, and
// the compiler then spends a v_mov_b32_dpp and a canonicalising v_max on every step.  A DPP read needs two wait states after
// a vector write of the same register, which the compiler does not insert for instructions it cannot see: the two chains
// are each other's first one, an s_nop the second; all steps are one statement, so that nothing comes between.)
template <int LPT> __device__ __forceinline__ void group_min_max(float &mn, float &mx) {
#define QFA_STEP(CTRL) \
  "v_min_f32_dpp %0, %0, %0 " CTRL " row_mask:0xf bank_mask:0xf\n\tv_max_f32_dpp %1, %1, %1 " CTRL " row_mask:0xf bank_mask:0xf\n\t"
#define QFA_QUADS "s_nop 1\n\t" QFA_STEP("quad_perm:[1,0,3,2]") "s_nop 0\n\t" QFA_STEP("quad_perm:[2,3,0,1]")
  static_assert(LPT >= 4, "a token takes four lanes at least");
  if constexpr (LPT == 4) asm(QFA_QUADS : "+v"(mn), "+v"(mx));
  else if constexpr (LPT == 8) asm(QFA_QUADS "s_nop 0\n\t" QFA_STEP("row_half_mirror") : "+v"(mn), "+v"(mx));
  else asm(QFA_QUADS "s_nop 0\n\t" QFA_STEP("row_half_mirror") "s_nop 0\n\t" QFA_STEP("row_mirror") : "+v"(mn), "+v"(mx));
  if constexpr (LPT >= 32) {
    mn = fminf(mn, __shfl_xor(mn, 16, 64));
    mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
  }
#undef QFA_QUADS
#undef QFA_STEP
}
// integer sum: `old` = 0, the identity of the addition (never used: every lane reads a valid lane),
// lets the compiler fold the permute into v_add_u32_dpp
template <int CTRL> __device__ __forceinline__ int dpp_zero(int x) { return __builtin_amdgcn_update_dpp(0, x, CTRL, 0xf, 0xf, false); }
template <int LPT> __device__ __forceinline__ int group_sum(int v) {
  v += dpp_zero<0xB1>(v);
  if (LPT >= 4) v += dpp_zero<0x4E>(v);
  if (LPT >= 8) v += dpp_zero<0x141>(v);
  if (LPT >= 16) v += dpp_zero<0x140>(v);
  if (LPT >= 32) v += __shfl_xor(v, 16, 64);
  return v;
}

template <typename T> struct Load8;
template <> struct Load8<float> {
  static __device__ __forceinline__ void run(const void *p, float (&v)[8]) {
    const f32x4 *q = reinterpret_cast<const f32x4 *>(p);
    f32x4 a = __builtin_nontemporal_load(q), b = __builtin_nontemporal_load(q + 1);
#pragma unroll
    for (int e = 0; e < 4; ++e) { v[e] = a[e]; v[4 + e] = b[e]; }
  }
};
template <> struct Load8<__bf16> {
  static __device__ __forceinline__ void run(const void *p, float (&v)[8]) {
    u32x4 w = __builtin_nontemporal_load(reinterpret_cast<const u32x4 *>(p));
#pragma unroll
    for (int e = 0; e < 4; ++e) {   // bf16 -> fp32 is a 16-bit shift
      v[2 * e] = __builtin_bit_cast(float, w[e] << 16);
      v[2 * e + 1] = __builtin_bit_cast(float, w[e] & 0xffff0000u);
    }
  }
};
template <> struct Load8<_Float16> {
  static __device__ __forceinline__ void run(const void *p, float (&v)[8]) {
    f16x8 w = __builtin_bit_cast(f16x8, __builtin_nontemporal_load(reinterpret_cast<const u32x4 *>(p)));
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = (float)w[e];
  }
};

// The row arithmetic: E (8 or 16) elements per lane, a token in LPT adjacent lanes.  Returns the lane's codes and, in
// every lane of the token, its scale, zero point (an integer in [-128, 127]) and code sum.  `used`: false in the lanes
// past the row's end (they hold a copy of elements of the row and add nothing to the sum).
template <int E> struct QuantRow {
  unsigned codes[E / 4];
  float scale, zp;
  int sum;
};
// Division by the per-token scale.  In the common exponent range the quotient is formed with the same FMA refinement the
// hardware division sequence uses (reciprocal refined once, two residual corrections of the quotient), which gives the
// correctly rounded x/scale without the per-element operand scaling.  Quotients below 2^-30 in magnitude may differ in their
// last bits, which cannot matter: they vanish in the addition of the zero point or round to zero.  SHORT: elements of at most
// 11 significant bits (16-bit tensors) need one correction only: no pair of such a significand with a scale's 24-bit one
// gives another quotient than `/` (tests/test_quant_division_gpu.py compares all 2^33; the steps do not depend on the
// exponents).
__device__ __forceinline__ float quant_reciprocal(float scale) {
#pragma clang fp contract(off)
  const float r = __builtin_amdgcn_rcpf(scale);
  return __builtin_fmaf(__builtin_fmaf(-scale, r, 1.0f), r, r);
}
template <bool SHORT> __device__ __forceinline__ float quant_quotient(float x, float scale, float r) {
#pragma clang fp contract(off)
  float q = x * r;
  q = __builtin_fmaf(__builtin_fmaf(-scale, q, x), r, q);
  if (!SHORT) q = __builtin_fmaf(__builtin_fmaf(-scale, q, x), r, q);
  return q;
}

// SHORT: as above.
template <int LPT, bool SHORT, int E> __device__ __forceinline__ QuantRow<E> quant_row(const float (&v)[E], bool used) {
#pragma clang fp contract(off)
  float mn = v[0], mx = v[0];
#pragma unroll
  for (int e = 1; e < E; ++e) { mn = fminf(mn, v[e]); mx = fmaxf(mx, v[e]); }
  group_min_max<LPT>(mn, mx);
  float scale = (mx - mn) / 255.0f;
  scale = (scale == 0.0f) ? 1.0f : scale;
  // the shared reciprocal's range: a tiny scale, huge values and NaN take the IEEE `/`
  const bool fast = (scale >= 0x1p-60f) && (fmaxf(fabsf(mn), fabsf(mx)) <= 0x1p60f);
  const float r = quant_reciprocal(scale);
  auto fdiv = [&](float x) -> float { return quant_quotient<SHORT>(x, scale, r); };
  // roundf (ties away from zero) in three instructions: add the largest float below one half with the
  // sign of y, truncate.  Equal to roundf for every binary32 value (checked exhaustively on the CPU; the
  // classic y + 0.5 fails at 0.49999997).
  auto round_away = [](float y) -> float {
    return __builtin_truncf(y + __builtin_copysignf(0x1.fffffep-2f, y));
  };
  float q[E], qmn;
  if (fast) {
    qmn = fdiv(mn);
#pragma unroll
    for (int e = 0; e < E; ++e) q[e] = fdiv(v[e]);
  } else {
    qmn = mn / scale;
#pragma unroll
    for (int e = 0; e < E; ++e) q[e] = v[e] / scale;
  }
  const float zpf = -128.0f - qmn;
  const float zp = fmaxf(-128.0f, fminf(127.0f, round_away(zpf)));
  // codes leave as biased bytes: roundf(.) + 128 converted with unsigned saturation (= the clamp to
  // [-128, 127]), flipped back to two's complement with one XOR per dword
  QuantRow<E> row;
#pragma unroll
  for (int e = 0; e < E; ++e) {
    const float y = q[e] + zp;
    const float c = round_away(y) + 128.0f;
    row.codes[e / 4] = __builtin_amdgcn_cvt_pk_u8_f32(c, e % 4, e % 4 == 0 ? 0u : row.codes[e / 4]);
  }
  unsigned sum = 0;
#pragma unroll
  for (int i = 0; i < E / 4; ++i) {
    sum = __builtin_amdgcn_sad_u8(row.codes[i], 0u, sum);
    row.codes[i] ^= 0x80808080u;
  }
  row.sum = group_sum<LPT>(used ? (int)sum - E * 128 : 0);
  row.scale = scale;
  row.zp = zp;
  return row;
}

}  // namespace qfa
