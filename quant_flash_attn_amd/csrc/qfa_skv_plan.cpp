// Which shared-KV kernel takes a call and how its keys are split over workgroups: pure functions of the sizes.
//
// A launch of n workgroups is estimated as rounds of the workgroups that are resident at once; a round costs its tiles per
// workgroup (and `extra` of them for start and end) times what a tile takes on the busiest CU: `alone` with one workgroup on
// it, `each` times their number with more.  A split adds the launch that merges (`merge` and `per_mb` for every 10^6 floats
// of partial results).  Constants in microseconds, fitted to measured launches of 1 to 1500 heads, 1 to 512 queries and 300
// to 24000 keys: forward 2439 / 862 (head_dim 64: 2 / 4 waves side by side), 2140 / 715 (128), 1775 / 575 (256) of them with
// 3 to 7 % rms, one-pass backward 650 / 650, 646 / 641 and 636 with 5 to 8 %, dQ 2 to 4 %.  What the estimates choose is
// within 0.3 to 2 % of the best measured choice on average.
#include "qfa_host.h"
#include "qfa_merge.h"

namespace qfa {
namespace {

struct Cost {
  float base, alone, each, extra, merge, per_mb;
  int resident;   // workgroups per CU
  float of(int64_t n, float tiles, int64_t splits, int64_t partials) const {
    const int64_t slots = 256 * resident, full = n / slots, rem = n % slots;
    const auto step = [&](int64_t c) { const float t = (float)c * each; return t > alone ? t : alone; };
    float rounds = (float)full * step(resident);
    if (rem) rounds += step((rem + 255) / 256);
    return base + rounds * (tiles + extra) + (splits > 1 ? merge + per_mb * 1e-6f * (float)partials : 0.0f);
  }
};
int by_dim(int D) { return D == 256 ? 2 : D == 128 ? 1 : 0; }

//                               head_dim 64                              128                                      256
// 16 queries per workgroup, tiles of 32 keys dealt to four waves
const Cost kFwd16[3] = {{4.3f, .542f, .385f, 1.16f, 3.2f, 2.0f, 3}, {5.4f, .451f, .597f, 1.40f, 3.1f, 1.2f, 3}, {4.4f, 1.324f, 1.059f, 2.18f, 3.4f, 1.0f, 2}};
// 32 queries per wave, tiles of 64 keys; two and four waves side by side
const Cost kFwdTile[2][3] = {
    {{5.6f, .662f, .390f, 0.f, 2.5f, 2.9f, 3}, {7.0f, .877f, .579f, 0.f, 1.9f, 3.0f, 2}, {7.3f, 1.543f, 1.252f, 1.94f, 0.9f, 3.0f, 1}},
    {{5.4f, .957f, .661f, 0.f, 2.9f, 2.6f, 3}, {4.5f, 1.182f, .881f, 1.72f, 2.8f, 2.5f, 2}, {4.6f, 2.437f, 0.f, 1.56f, 2.9f, 2.7f, 1}}};
// one-pass backward: up to 16 queries, up to 32
const Cost kPass[2][3] = {
    {{6.1f, 1.638f, 1.159f, 0.45f, 2.7f, 2.4f, 2}, {6.0f, 2.717f, 2.163f, 1.17f, 1.8f, 1.5f, 2}, {2.2f, 5.371f, 4.535f, 2.47f, 0.6f, 1.7f, 1}},
    {{4.6f, 1.898f, 1.309f, 1.34f, 2.6f, 1.9f, 2}, {6.6f, 3.010f, 2.324f, 1.02f, 1.7f, 1.6f, 2}, {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 1}}};
// dQ: 16 queries per workgroup; tiles with two and four waves side by side (only their differences matter: no base)
const Cost kDq16[3] = {{0.f, .602f, .356f, 0.97f, 0.f, 0.f, 3}, {0.f, .810f, .664f, 0.39f, 0.f, 0.f, 3}, {0.f, 1.151f, .912f, 3.13f, 0.f, 0.f, 2}};
const Cost kDqTile[2][3] = {
    {{0.f, .998f, .548f, 0.f, 2.7f, 1.8f, 3}, {0.f, 1.336f, .932f, 0.21f, 2.4f, 2.0f, 2}, {0.f, 2.672f, 2.535f, 1.81f, 2.6f, 1.7f, 1}},
    {{0.f, 1.284f, .482f, 0.f, 4.0f, 1.9f, 3}, {0.f, 2.015f, 1.326f, 0.f, 3.8f, 1.7f, 2}, {0.f, 3.697f, 2.142f, 0.70f, 6.6f, 1.6f, 1}}};

const int kSplits[] = {1, 2, 3, 4, 6, 8, 12, 16, 24, 32, 48, 64};

// the best split of `tiles` tiles for `wgs` workgroups; at least two tiles each, partial results of at most `room` floats
void best_split(const Cost &c, int64_t wgs, int64_t rows, int64_t tiles, float per, int64_t row_floats, int64_t room, int *splits,
                int64_t *tiles_each, float *cost) {
  *splits = 1;
  *cost = 3e38f;
  for (const int s : kSplits) {
    if (s > 1 && (2 * s > tiles || wgs * s > 1600 || rows * s * row_floats > room)) break;
    const int64_t each = (tiles + s - 1) / s, used = (tiles + each - 1) / each;
    const float t = c.of(wgs * used, per * (float)each, used, rows * used * row_floats);
    if (t < (s > 1 && *splits == 1 ? 0.9f : 1.0f) * *cost) {   // (a split has to promise a tenth)
      *cost = t;
      *splits = (int)used;
      *tiles_each = each;
    }
  }
}
// two or four waves side by side on the queries, the keys split
SkvTilePlan best_tile(const Cost (*c)[3], int64_t BH, int64_t Nq, int64_t Nk, int D, int64_t row_floats, int64_t room, float *cost) {
  const int64_t blocks = (Nq + 31) / 32, tiles = (Nk + 63) / 64;
  SkvTilePlan p = {2, 1, (int)tiles};
  *cost = 3e38f;
  for (int i = 0; i < (blocks > 2 ? 2 : 1); ++i) {
    const int qw = i ? 4 : 2;
    int splits = 1;
    int64_t each = tiles;
    float t;
    best_split(c[i][by_dim(D)], BH * ((blocks + qw - 1) / qw), BH * Nq, tiles, 1.0f, row_floats, room, &splits, &each, &t);
    if (t < *cost) {
      *cost = t;
      p = {qw, splits, (int)each};
    }
  }
  return p;
}

}  // namespace

void skv_fwd16_plan(int64_t BH, int64_t Nq, int64_t Nk, int D, int *splits, int *tiles_per_split) {
  // as many workgroups as are resident at once (three per CU; a second, partly filled round costs a whole one), at head_dim
  // 256 about four per CU (two are resident), or what split_plan finds better
  const int64_t wgs = BH * ((Nq + 15) / 16);
  const int64_t fill = D == 256 ? (wgs >= 512 ? 1 : (1024 + wgs - 1) / wgs) : 768 / wgs;
  split_plan(wgs, BH * Nq, (Nk + 31) / 32, D, fill, splits, tiles_per_split);
}

SkvTilePlan skv_tile_fwd_plan(int64_t BH, int64_t Nq, int64_t Nk, int D) {
  const SkvTilePlan none = {0, 1, 0};
  if (Nq <= 16) return none;
  // (partial results within the built-in scratch at every head_dim)
  float t;
  const SkvTilePlan p = best_tile(kFwdTile, BH, Nq, Nk, D, D + 2, QFA_STATIC_SCRATCH_BYTES / 4, &t);
  int splits, each;
  skv_fwd16_plan(BH, Nq, Nk, D, &splits, &each);
  const float t16 = kFwd16[by_dim(D)].of(BH * ((Nq + 15) / 16) * splits, 0.25f * (float)each, splits, BH * Nq * splits * (D + 2));
  // (with 32 queries or fewer half of the waves have none)
  return t < (Nq <= 32 ? 0.85f : 0.97f) * t16 ? p : none;
}

SkvTilePlan skv_tile_dq_plan(int64_t BH, int64_t Nq, int64_t Nk, int D) {
  float t;
  const SkvTilePlan p = best_tile(kDqTile, BH, Nq, Nk, D, D, 16 << 20, &t);
  const float t16 = kDq16[by_dim(D)].of(BH * ((Nq + 15) / 16), 0.25f * (float)((Nk + 31) / 32), 1, 0);
  // (33 to 48 queries leave a quarter of two waves' work to padding: 1024 heads, 48 queries, 3000 keys of 128 take 178 us with
  // the one kernel and 208 with the other)
  return t < (Nq <= 48 ? 0.75f : 0.93f) * t16 ? p : SkvTilePlan{0, 1, 0};
}

int skv_bwd_splits(int64_t BH, int64_t Nq, int64_t Nk, int D) {
  int splits = 1;
  int64_t each;
  float t;
  best_split(kPass[Nq <= 16 ? 0 : 1][by_dim(D)], BH, BH * Nq, (Nk + 31) / 32, 0.25f, D, 16 << 20, &splits, &each, &t);
  return splits;
}

int64_t skv_bwd_workspace_bytes(int64_t B, int64_t H, int64_t Nq, int64_t Nk, int D) {
  const int s = skv_bwd_one_pass(Nq, D) ? skv_bwd_splits(B * H, Nq, Nk, D) : skv_tile_dq_plan(B * H, Nq, Nk, D).splits;
  return s > 1 ? B * H * Nq * s * (int64_t)D * 4 : 0;
}

}  // namespace qfa
