// Merge of the partial results of an attention whose keys are split over workgroups (shared-KV and INT8-score forward, cache decode).
#pragma once
#include <cfloat>

#include "qfa_device.h"
#include "qfa_host.h"

namespace qfa {

// row maximum of a wave or split that saw no key: finite, so that differences of two of them are zero and not NaN (a
// split may also leave -inf: the merges start from the lowest finite value)
constexpr float NO_KEY = -1e30f;

// four consecutive outputs of a row, rounded to the queries' type
__device__ __forceinline__ void store4(void *row, int q_dtype, int d, f32x4 x) {
  if (q_dtype == QFA_F32) {
    *reinterpret_cast<f32x4 *>(static_cast<float *>(row) + d) = x;
  } else {
    u32x2 w;
    if (q_dtype == QFA_BF16) w = u32x2{pack2<__bf16>(x[0], x[1]), pack2<__bf16>(x[2], x[3])};
    else w = u32x2{pack2<_Float16>(x[0], x[1]), pack2<_Float16>(x[2], x[3])};
    *reinterpret_cast<u32x2 *>(static_cast<unsigned short *>(row) + d) = w;
  }
}

struct SplitMergeArgs {
  const float *po, *pml;   // [B*H*Nq][splits][D] unnormalised O, and (m in log2 units, l)
  void *o;
  float *lse;              // nullable, [B*H*Nq]
  int64_t H, sob, soh, son;
  int Nq, splits, o_dtype;
  float *o32;   // nullable: O in fp32, dense; then o is nullable too
};

// one row's columns d .. d + 3, normalised, to where they go
__device__ __forceinline__ void merge_store(const SplitMergeArgs &a, int64_t row, int D, int d, const f32x4 &acc, float m, float l) {
  const float inv = 1.0f / l;
  const f32x4 x = {acc[0] * inv, acc[1] * inv, acc[2] * inv, acc[3] * inv};
  if (a.lse && d == 0) a.lse[row] = (m + __log2f(l)) * kLn2;
  if (a.o32) *reinterpret_cast<f32x4 *>(a.o32 + row * D + d) = x;
  if (!a.o) return;
  const int64_t bh = index_div(row, a.Nq), b = index_div(bh, a.H), h = bh - b * a.H, off = b * a.sob + h * a.soh + (row - bh * a.Nq) * a.son;
  store4(static_cast<char *>(a.o) + off * (a.o_dtype == QFA_F32 ? 4 : 2), a.o_dtype, d, x);
}

// O of one query from the partial results of its splits: one workgroup per query, D/4 lanes of four columns times
// 1024/D groups of splits.  All loads of a thread are independent, so the kernel is one memory latency long.
template <int D> __global__ __launch_bounds__(256) void split_merge_kernel(SplitMergeArgs a) {
  constexpr int CL = D / 4, SG = 256 / CL;
  __shared__ float red[SG][D + 4];
  const int tid = threadIdx.x, d = 4 * (tid % CL), sg = tid / CL;
  const int64_t row = blockIdx.x, slot = row * a.splits;
  float m = -FLT_MAX, l = 0.f;
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
  for (int s = sg; s < a.splits; s += SG) {
    const f32x2 ml = *reinterpret_cast<const f32x2 *>(a.pml + 2 * (slot + s));
    const f32x4 y = *reinterpret_cast<const f32x4 *>(a.po + (slot + s) * D + d);
    const float m_new = fmaxf(m, ml[0]), s0 = __builtin_amdgcn_exp2f(m - m_new), s1 = __builtin_amdgcn_exp2f(ml[0] - m_new);
    m = m_new;
    l = l * s0 + ml[1] * s1;
#pragma unroll
    for (int e = 0; e < 4; ++e) acc[e] = acc[e] * s0 + y[e] * s1;
  }
  *reinterpret_cast<f32x4 *>(&red[sg][d]) = acc;
  if (tid % CL == 0) {
    red[sg][D] = m;
    red[sg][D + 1] = l;
  }
  __syncthreads();
  if (sg > 0) return;
  float ma = -FLT_MAX, la = 0.f;
#pragma unroll
  for (int s = 0; s < SG; ++s) ma = fmaxf(ma, red[s][D]);
  acc = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int s = 0; s < SG; ++s) {
    const float w = __builtin_amdgcn_exp2f(red[s][D] - ma);
    la += red[s][D + 1] * w;
    const f32x4 y = *reinterpret_cast<const f32x4 *>(&red[s][d]);
#pragma unroll
    for (int e = 0; e < 4; ++e) acc[e] += y[e] * w;
  }
  merge_store(a, row, D, d, acc, ma, la);
}

// The same for few splits: D/4 lanes per query, 1024/D queries per workgroup.  A workgroup per query is as many workgroups
// as rows, most of whose lanes have nothing to do where there are fewer splits than groups (64 heads, 200 queries, two
// splits: the whole forward 32 -> 24 us).
template <int D> __global__ __launch_bounds__(256) void split_merge_few_kernel(SplitMergeArgs a, int64_t rows) {
  constexpr int CL = D / 4, RPW = 256 / CL;
  const int d = 4 * (threadIdx.x % CL);
  const int64_t row = (int64_t)blockIdx.x * RPW + threadIdx.x / CL, slot = row * a.splits;
  if (row >= rows) return;
  float m = -FLT_MAX, l = 0.f;
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
  for (int s = 0; s < a.splits; ++s) {
    const f32x2 ml = *reinterpret_cast<const f32x2 *>(a.pml + 2 * (slot + s));
    const f32x4 y = *reinterpret_cast<const f32x4 *>(a.po + (slot + s) * D + d);
    const float m_new = fmaxf(m, ml[0]), s0 = __builtin_amdgcn_exp2f(m - m_new), s1 = __builtin_amdgcn_exp2f(ml[0] - m_new);
    m = m_new;
    l = l * s0 + ml[1] * s1;
#pragma unroll
    for (int e = 0; e < 4; ++e) acc[e] = acc[e] * s0 + y[e] * s1;
  }
  merge_store(a, row, D, d, acc, m, l);
}

inline int64_t split_partial_bytes(int64_t rows, int64_t splits, int D) { return rows * splits * (int64_t)(D + 2) * 4; }

// How `ntiles` tiles of keys are dealt: `wgs` workgroups of up to 16 of `rows` queries per split, at least 8 tiles each.
// `fill` is the number of splits that fills the resident slots once, as far as whole splits go.  Two kinds of shapes lose by
// it: where the remainder is large (300 workgroups on 512 slots: no split, and 44 CUs work twice as long as the others), and
// where the keys are so few that the merge costs more than the split brings (256 workgroups of 700 keys).  Another number is
// taken when the estimate below -- the tiles of the busiest of 256 CUs, four per workgroup for its start and end, and the
// merge, which is about as long as 16 tiles of 128 -- says 30 % better, which is where measuring agrees with it.
// Measured over 1398 shapes (head_dim 64, 128, 256; 1 to 1300 workgroups; 513 to 32768 keys; both callers) against `fill`
// alone: 0 to 4 % faster on average; the most 300 workgroups, 8192 keys of 128 (145 -> 112 us) and 256 workgroups of 16
// queries, 700 keys of 64 (14.6 -> 8.8 us); none slower by more than 7 %, nearly all within 3 %.
// Partial results stay within 16 MB, unless those of `fill` do not (callers may bring a fixed scratch of that size).
inline void split_plan(int64_t wgs, int64_t rows, int64_t ntiles, int D, int64_t fill, int *splits, int *tiles_per_split) {
  const auto even = [&](int64_t s) { return (ntiles + s - 1) / s; };   // tiles per split
  const auto cost = [&](int64_t s) {
    const int64_t tps = even(s), n = wgs * ((ntiles + tps - 1) / tps);
    return (float)((n + 255) / 256 * (tps + 4)) + (s > 1 ? 2048.0f / (float)D + 0.001f * (float)(rows * s) : 0.0f);
  };
  const int64_t most = ntiles / 8;
  int64_t best = fill > most ? most : fill;
  if (best < 1) best = 1;
  const int64_t room = split_partial_bytes(rows, best, D) > (16 << 20) ? split_partial_bytes(rows, best, D) : 16 << 20;
  float least = cost(best) / 1.3f;
  for (int64_t s = 1; s <= 32 && s <= most && s * wgs <= 2600; ++s)
    if (split_partial_bytes(rows, s, D) <= room && cost(s) < least) {
      least = cost(s);
      best = s;
    }
  const int64_t tps = even(best);
  *tiles_per_split = (int)tps;
  *splits = (int)((ntiles + tps - 1) / tps);
}
template <int D> int launch_split_merge(const SplitMergeArgs &a, int64_t rows, const char *who, hipStream_t st) {
  constexpr int RPW = 1024 / D;
  if (a.splits <= 16 && rows >= 1024) split_merge_few_kernel<D><<<dim3((unsigned)((rows + RPW - 1) / RPW)), dim3(256), 0, st>>>(a, rows);
  else split_merge_kernel<D><<<dim3((unsigned)rows), dim3(256), 0, st>>>(a);
  return check_launch(who);
}

}  // namespace qfa
