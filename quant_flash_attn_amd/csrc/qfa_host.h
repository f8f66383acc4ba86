// Host-side declarations shared by the translation units of libqfa.so: the error
// channel behind qfa_last_error() and the launchers the C entry points dispatch to.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../../include/qfa.h"

namespace qfa {

// Records a thread-local message and returns `code` (so `return set_error(...)` reads naturally).
int set_error(int code, const char *fmt, ...) __attribute__((format(printf, 2, 3)));
// hipGetLastError() after a launch; 0 or the positive hipError_t, with the message recorded.
int check_launch(const char *what);

int launch_quant(const void *x, int x_dtype, int8_t *codes, float *scale, void *scale_lp, int scale_lp_dtype,
                 int8_t *zp, int32_t *rowsum, int64_t B, int64_t H, int64_t N, int D, int64_t sxb, int64_t sxh,
                 int64_t sxn, int64_t scb, int64_t sch, int64_t scn, hipStream_t st);
// the same for two tensors of one element type and head dimension in one launch (no 16-bit scale copy)
int launch_quant_pair(const void *const x[2], int x_dtype, int8_t *const codes[2], float *const scale[2],
                      int8_t *const zp[2], int32_t *const rowsum[2], int64_t B, int64_t H, const int64_t N[2], int D,
                      const int64_t sx[2][3], const int64_t sc[2][3], hipStream_t st);
// fp32 queries and keys quantized, fp32 values converted to bf16 (dense), in one launch; head_dim 64, 128 or 256
int launch_quant_qkv(const float *const x[2], int8_t *const codes[2], float *const scale[2], int8_t *const zp[2],
                     int32_t *const rowsum[2], const float *v, void *v16, int64_t B, int64_t H, const int64_t N[2], int D,
                     const int64_t sx[2][3], const int64_t sc[2][3], const int64_t sv[3], hipStream_t st);
// queries that are quantized on the way (their strides and their codes': batch, head, token)
struct QuantizeQ {
  const void *x;
  int dtype;
  int8_t *codes;
  float *scale;
  int8_t *zp;
  int32_t *rowsum;
  int64_t N, sx[3], sc[3];
};
int launch_cache_stage(const QuantizeQ *q, const int8_t *kc, const void *ks, int ks_dtype, float *ks32, int32_t *rowsum, const int8_t *vc,
                       const void *vs, int vs_dtype, const int8_t *vz, void *v, int v_dtype, int64_t B, int64_t H, int64_t N, int D,
                       const int64_t sk[3], const int64_t sv[3], hipStream_t st);   // q: nullable
int launch_rowsum(const int8_t *codes, int32_t *rowsum, int64_t B, int64_t H, int64_t N, int D, int64_t scb,
                  int64_t sch, int64_t scn, hipStream_t st);
int launch_dequant(const int8_t *codes, const void *scale, int scale_dtype, const int8_t *zp, void *out,
                   int out_dtype, int64_t B, int64_t H, int64_t N, int D, int64_t scb, int64_t sch, int64_t scn,
                   int64_t sob, int64_t soh, int64_t son, hipStream_t st);

// How the backward's two kinds of workgroups are launched: 32-row blocks per wave, and the parts of the streamed rows; the memory of the
// parts, and whether dQ is a launch of its own (its parts then take the place of the others)
struct BwdPlan { int blocks_dkv, splits_dkv, queries_per_split, blocks_dq, splits_dq, keys_per_split, sum_between; int64_t part_bytes; };

// Tensors of one attention call, after validation.  Strides in elements.
struct AttnArgs {
  const int8_t *qc; const float *sq; const int8_t *zq; const int32_t *rq;
  const int8_t *kc; const float *sk; const int8_t *zk; const int32_t *rk;
  const void *v; void *o; float *lse;
  const void *dout; void *workspace; void *dq; void *dk; void *dv;   // backward only (the workspace: also forward, see launch_fwd)
  int64_t B, H, Nq, Nk;
  int64_t sqb, sqh, sqn, skb, skh, skn, svb, svh, svn, sob, soh, son;
  int64_t sdob, sdoh, sdon, sdqb, sdqh, sdqn, sdkb, sdkh, sdkn, sdvb, sdvh, sdvn;
  float sm_scale;
  int causal;
  int D;
  int io_dtype;
  float *o32;   // forward: nullable, O in fp32 (dense); o is nullable then
  int f32;      // backward: dO and the gradients are fp32, the workspace holds bwd_f32_workspace_bytes
  BwdPlan bwd;  // backward: and bwd.part_bytes behind them
};

int launch_fwd(const AttnArgs &a, hipStream_t st, bool qk_only = false);   // workspace: nullable, the keys are split with one
// workgroups that share the keys of 128 queries, given a workspace, and the keys of each (a multiple of 64)
void fwd_plan(int64_t BH, int64_t Nq, int64_t Nk, int D, int causal, int *splits, int *keys_per_split);
int64_t fwd_workspace_bytes(int64_t B, int64_t H, int64_t Nq, int64_t Nk, int D, int causal);
int launch_delta(const void *o, const void *dout, float *delta, int io_dtype, int64_t B, int64_t H, int64_t N, int D,
                 int64_t sob, int64_t soh, int64_t son, int64_t sdb, int64_t sdh, int64_t sdn, hipStream_t st);
int launch_bwd(const AttnArgs &a, hipStream_t st);
int launch_sum16(const void *a, const void *b, void *out, int dtype, int64_t n, hipStream_t st);   // out = a + b, n % 8 == 0
int64_t bwd_workspace_bytes(int64_t B, int64_t H, int64_t Nq, int64_t Nk, int D);
inline int64_t bwd_f32_workspace_bytes(int64_t B, int64_t H, int64_t Nq, int64_t Nk, int D) {
  return bwd_workspace_bytes(B, H, Nq, Nk, D) + B * H * Nq * D * 2;
}

// causal: log2 of the heads whose blocks are dispatched together, `streamed` rows of 5 bytes per element each.  Pairs (N=4096,
// D=128: 5.2 MB against the XCD's 4 MB L2) are 1 % better than single heads, four heads are not: within about 6 MB
inline int bwd_group_log2(int64_t streamed, int D, bool dq) {
  const int64_t head_bytes = streamed * D * 5;
  int g = dq ? 1 : 0;
  while (g < (dq ? 3 : 2) && (head_bytes << (g + 1)) <= (6 << 20)) ++g;
  return g;
}
BwdPlan bwd_plan(int64_t BH, int64_t Nq, int64_t Nk, int D, int causal, int may_split);
// what a call with `room` bytes for parts launches (an entry makes it once: up to 7 us, which small calls notice)
BwdPlan bwd_plan_within(int64_t BH, int64_t Nq, int64_t Nk, int D, int causal, int64_t room);
int64_t bwd_split_bytes(int64_t B, int64_t H, int64_t Nq, int64_t Nk, int D, int causal);

// grid of a kernel that maps ids with XcdBlock (qfa_skv_common.h): per_bh workgroups for each of BH heads
__host__ __device__ inline bool xcd_whole_heads(int64_t BH) { return BH >= 64 || BH % 8 == 0; }
inline int64_t xcd_grid(int64_t BH, int64_t per_bh) {
  return xcd_whole_heads(BH) ? (BH + 7) / 8 * 8 * per_bh : (BH * per_bh + 7) / 8 * 8;
}

// What a launch reads and writes beyond this, nobody finds in the last-level cache afterwards: what is touched once is better kept out of
// the caches then, which others still need
constexpr int64_t LAST_LEVEL_BYTES = 256 << 20;
// Whether no line of 128 bytes holds rows of two heads, which two workgroups would read (rows of row_bytes, strides in elements of `es`
// bytes): a head's rows in one piece, or each row whole lines.  Rows of 64 bytes with those of other heads between them, read with
// non-temporal loads, took 1.06 to 1.35 times as long as without (16 x 32 heads, one query on 8192 keys of 64, [B, N, H, D]: 171 -> 199 us)
inline bool rows_own_lines(const void *p, int64_t sb, int64_t sh, int64_t sn, int row_bytes, int es = 1) {
  return sn * es == row_bytes || (((int64_t)reinterpret_cast<uintptr_t>(p) | sb * es | sh * es | sn * es | row_bytes) & 127) == 0;
}

// Whether the forward's O, 16 bit, is written past the caches (qfa_split_plan.cpp)
bool fwd_o_once(int64_t BH, int64_t Nq, int64_t Nk, int D, const void *o, int64_t sob, int64_t soh, int64_t son);

// Shared-KV attention (K = V = one quantized tensor, Q in 16-bit float), after validation.
struct SkvAttnArgs {
  const void *q; const int8_t *codes; const void *scale; const int8_t *zp;
  void *o; float *lse;
  const void *dout; void *dq; void *dkv;   // backward only
  void *workspace;                         // nullable: partial results when the keys are split
  int64_t B, H, Nq, Nk;
  int64_t sqb, sqh, sqn, scb, sch, scn, sob, soh, son;
  int64_t sdob, sdoh, sdon, sdqb, sdqh, sdqn, sdkb, sdkh, sdkn;
  float sm_scale;
  int D, io_dtype, scale_dtype;
  int grad_dtype; const float *grad_scale;   // backward only: type of dq / dkv, optional device scalar multiplying them
  int direct, dout_dtype;   // backward: q and o of io_dtype, dO of dout_dtype, cast and scaled inside (where skv_bwd_direct)
};
int launch_skv_bwd(const SkvAttnArgs &a, hipStream_t st);        // io_dtype QFA_F16, Nq <= 32: one fused pass
// dO * 2^k as binary16 plus 2^-k for the binary16 backward kernels (k from max|dO| and the largest key scale);
// partials: dout_normalise_workspace_bytes() of scratch
int64_t dout_normalise_workspace_bytes();
int launch_dout_normalise(const void *dout, int dout_dtype, int64_t n, const void *scale, int scale_dtype, int64_t ns,
                          float *partials, void *out, float *back, const void *x0, void *y0, const void *x1,
                          void *y1, hipStream_t st);
// Query blocks of more than 16: forward and dQ on tiles of 64 keys that a workgroup expands once.  qw: waves side by side on
// the queries (0: not this kernel), splits: workgroups that share the keys, tiles of 64 keys each
struct SkvTilePlan { int qw, splits, tiles; };
// The forward: on tiles where tile.qw is not 0, otherwise 16 queries per workgroup and that many splits of 32-key tiles; the bytes
// of the partial results.  An entry makes it once (up to 0.4 us, which calls of two small launches, 10 us in all, notice)
struct SkvFwdPlan { SkvTilePlan tile; int splits, tiles_per_split; int64_t part_bytes; };
SkvFwdPlan skv_fwd_plan(int64_t BH, int64_t Nq, int64_t Nk, int D);
int launch_skv_fwd(const SkvAttnArgs &a, const SkvFwdPlan &p, hipStream_t st);
// the same with the partial results of a split in the library's own static device array (a.workspace is ignored)
int launch_skv_fwd_static(const SkvAttnArgs &a, hipStream_t st);
SkvTilePlan skv_tile_dq_plan(int64_t BH, int64_t Nq, int64_t Nk, int D);
int launch_skv_tile_fwd(const SkvAttnArgs &a, const SkvTilePlan &p, hipStream_t st);
int launch_skv_tile_dq(const SkvAttnArgs &a, const SkvTilePlan &p, hipStream_t st);
int launch_skv_dkv(const SkvAttnArgs &a, hipStream_t st);
// dQ and dKV of 33 to 128 queries in one pass (head_dim 64 and 128): a workgroup per head, where there are enough of them
bool skv_pass_takes(int64_t BH, int64_t Nq, int64_t Nk, int D);
bool skv_pass_takes_unsplit(int64_t BH, int64_t Nq, int64_t Nk, int D);   // ... of a call without scratch
// ... if the offsets of a head's rows, those of a few tiles past its end included, fit 31 bits
inline bool skv_pass_fits(int64_t Nk, int64_t scn, int64_t sdqn, int64_t sdkn) {
  const int64_t rows = Nk + 512, most = 1 << 23;
  return rows * scn < (1LL << 31) && rows * sdkn < (1LL << 30) && sdqn < most && sdkn < most;
}
int launch_skv_pass(const SkvAttnArgs &a, hipStream_t st);
// dQ = the sum of its partial results [B*H*Nq][splits][D] in a.workspace, times *grad_scale, rounded
int launch_split_sum(const SkvAttnArgs &a, int splits, hipStream_t st);
// one fused backward pass while the per-wave accumulators of dQ fit: 32 queries up to head_dim 128, 16 at 256
inline bool skv_bwd_one_pass(int64_t Nq, int D) { return D == 256 ? Nq <= 16 : Nq <= 32; }
// whether the backward's kernels cast and scale their rows themselves: that pass, and the two kernels while dKV's rows stay in LDS
inline bool skv_bwd_direct(int64_t Nq, int D) { return skv_bwd_one_pass(Nq, D) || (D <= 128 && Nq <= 128); }
// workgroups that share the keys of a (batch, head) in that pass, given a workspace
int skv_bwd_splits(int64_t BH, int64_t Nq, int64_t Nk, int D);
int64_t skv_bwd_workspace_bytes(int64_t B, int64_t H, int64_t Nq, int64_t Nk, int D);
int launch_skv_bwd_long(const SkvAttnArgs &a, hipStream_t st);   // io_dtype QFA_F16, any Nq: dQ kernel + dKV kernel

// Attention of a short query block on an INT8 cache (K and V quantized separately, Q quantized inside), after validation.
struct CacheAttnArgs {
  const void *q; const int8_t *kc; const void *ks; const int8_t *kz; const int8_t *vc; const void *vs; const int8_t *vz;
  void *o;
  float *lse;        // nullable
  void *workspace;   // nullable: partial results when the keys are split
  int64_t B, H, Nq, Nk;
  int64_t sqb, sqh, sqn, skb, skh, skn, svb, svh, svn, sob, soh, son;
  float sm_scale;
  int causal, D, q_dtype, scale_dtype;
};
int launch_cache_fwd(const CacheAttnArgs &a, hipStream_t st);
int64_t cache_workspace_bytes(int64_t B, int64_t H, int64_t Nq, int64_t Nk, int D);

}  // namespace qfa
