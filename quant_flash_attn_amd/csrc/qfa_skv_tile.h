// Tiles of keys that a workgroup expands once, as binary16 integers code - zero_point in LDS: their layout, the way of a tile from
// memory into it and the two kinds of reads (forward and dQ: qfa_skv_tile.hip; the whole backward: qfa_skv_pass.hip).
#pragma once
#include "qfa_skv_common.h"

namespace qfa {

// Offset of 8 columns (half h of slab c) of row r inside a tile.  The halves are swapped for rows 8-15 and 24-31 (16 lanes
// that read 16 rows of a slab, and 32 lanes of a transposing read, hit all banks once) and for slabs 2, 3, 6, 7, ... (so do
// 16 lanes that write 4 rows of 4 slabs).
template <int SLAB> __device__ __forceinline__ int skv_tile_off(int r, int c, int h) {
  return c * SLAB + r * 32 + ((h ^ (r >> 3 & 1) ^ (c >> 1 & 1)) << 4);
}

// A thread's share of a tile on its way from memory to LDS: N chunks of 16 codes with their rows' zero points, one key scale
template <int D, int TK, int SLAB> struct SkvTileStage {
  static constexpr int CPR = D / 16, RPW = 64 / CPR, N = TK * CPR / 256, STEP = 4 * RPW;   // STEP: rows between a thread's chunks
  unsigned off, row_step;   // of chunk 0; bytes between a thread's chunks
  int row, lds;
  int tid;
  u32x4 w[N];
  unsigned z[N];
  unsigned s;
  int live;   // keys of the tile that exist
  __device__ __forceinline__ void init(unsigned stride, int tid_) {
    tid = tid_;
    const int lane = tid % 64, wave = tid / 64, hi = lane / 16;
    constexpr int CH = CPR / 4;   // chunk groups of 4 side by side in a wave
    const int c = lane % 4 + 4 * (hi % CH);
    row = wave * RPW + (lane / 4) % 4 + 4 * (hi / CH);
    off = (unsigned)row * stride + (unsigned)c * 16u;
    row_step = (unsigned)STEP * stride;
    lds = skv_tile_off<SLAB>(row, c, 0);
  }
  // tile of `rows` keys that exist (at least one); what lies past them arrives as zeros
  __device__ __forceinline__ void issue(const unsigned char *codes, const void *scale, int s32, const int8_t *zp, int64_t key0,
                                        int64_t stride, int rows) {
    rows = live = min(rows, TK);
    const rsrc_t rk = make_rsrc(codes, (unsigned)((rows - 1) * (int)stride + D)), rz = make_rsrc(zp + key0, (unsigned)rows);
#pragma unroll
    for (int i = 0; i < N; ++i) {
      w[i] = __builtin_amdgcn_raw_buffer_load_b128(rk, (int)(off + row_step * (unsigned)i), 0, 0);
      z[i] = (unsigned char)__builtin_amdgcn_raw_buffer_load_b8(rz, row + STEP * i, 0, 0);
    }
    if (s32) {
      const rsrc_t rs = make_rsrc(static_cast<const float *>(scale) + key0, (unsigned)rows * 4u);
      s = __builtin_amdgcn_raw_buffer_load_b32(rs, (tid % TK) * 4, 0, 0);
    } else {
      const rsrc_t rs = make_rsrc(static_cast<const unsigned short *>(scale) + key0, (unsigned)rows * 2u);
      s = (unsigned short)__builtin_amdgcn_raw_buffer_load_b16(rs, (tid % TK) * 2, 0, 0);
    }
  }
  // chunk i of the tile into buf
  __device__ __forceinline__ void commit_chunk(unsigned char *buf, int i) {
    const unsigned nz = 0xe400u | (z[i] ^ 0x80u), nz2 = nz | nz << 16;   // -(1152 + zero_point), twice
    const f16x2 neg = __builtin_bit_cast(f16x2, nz2);
    u32x4 e[2];
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      const u32x4 m = expand_codes(w[i][2 * k], w[i][2 * k + 1]);
#pragma unroll
      for (int x = 0; x < 4; ++x) {
        const unsigned mx = m[x];
        e[k][x] = __builtin_bit_cast(unsigned, __builtin_bit_cast(f16x2, mx) + neg);
      }
    }
    static_assert(STEP % 16 == 0, "the swap of halves repeats: they stay where they are");
    *reinterpret_cast<u32x4 *>(buf + lds + i * (STEP * 32)) = e[0];
    *reinterpret_cast<u32x4 *>(buf + (lds ^ 16) + i * (STEP * 32)) = e[1];
  }
  // the key scales are multiplied by `mul`; keys past the end get a scale of one (their scores become -inf)
  __device__ __forceinline__ void commit_scale(unsigned char *buf, int scale_dtype, float mul) {
    if (tid < TK) {
      const unsigned sw = s;
      const float f = scale_dtype == QFA_F32 ? __builtin_bit_cast(float, sw)
                      : scale_dtype == QFA_F16 ? lo_to_f32<_Float16>(sw) : lo_to_f32<__bf16>(sw);
      *reinterpret_cast<float *>(buf + CPR * SLAB + tid * 4) = tid < live ? f * mul : 1.0f;
    }
  }
  __device__ __forceinline__ void commit(unsigned char *buf, int scale_dtype, float mul) {
#pragma unroll
    for (int i = 0; i < N; ++i) commit_chunk(buf, i);
    commit_scale(buf, scale_dtype, mul);
  }
};

typedef __fp16 tr16_t __attribute__((vector_size(8)));
typedef __attribute__((address_space(3))) tr16_t *lds_h4;
// transposing read of 4 rows x 16 columns per 16 lanes (ds_read_b64_tr_b16, see qfa_device.h); no direct copies are in
// flight in these kernels, so the compiler's own waits cost nothing
__device__ __forceinline__ u32x2 lds_read_tr16(const unsigned char *p) {
  return __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4f16((lds_h4)(lptr_t)p));
}

// per-lane offsets of the two kinds of reads, [slab pair odd]: rows (row lr, half g) and transposing (rows 4g + {0..3} of
// slabs u; rows 8 further have their halves swapped)
template <int SLAB> struct SkvTileReads {
  int row[2], tr[2];
  __device__ __forceinline__ SkvTileReads(int lane) {
    const int lr = lane % 32, g = lane / 32, s16 = lane % 16, u = lane / 16 % 2;
#pragma unroll
    for (int x = 0; x < 2; ++x) {
      row[x] = skv_tile_off<SLAB>(lr, 2 * x, g) - 2 * x * SLAB;
      tr[x] = skv_tile_off<SLAB>(4 * g + s16 / 4, u + 2 * x, s16 % 4 / 2) - 2 * x * SLAB + s16 % 2 * 8;
    }
  }
  __device__ __forceinline__ u32x4 rows(const unsigned char *p, int m) const {   // columns 16m + 8g + {0..7} of rows lr
    return *reinterpret_cast<const u32x4 *>(p + m * SLAB + row[m >> 1 & 1]);
  }
  // columns 32db + lr of rows 16hh + 4g + {0..3} and those + 8
  __device__ __forceinline__ u32x4 cols(const unsigned char *p, int db, int hh) const {
    const unsigned char *c = p + 2 * db * SLAB + hh * 512;
    const u32x2 a = lds_read_tr16(c + tr[db & 1]), b = lds_read_tr16(c + 256 + (tr[db & 1] ^ 16));
    return u32x4{a[0], a[1], b[0], b[1]};
  }
};

// a row of D 16-bit elements as B operands: k-step m, k-group g holds columns 16m + 8g + {0..7}; bf16 becomes binary16
template <int D> __device__ __forceinline__ void skv_load_row(const void *p, int64_t at, int bf16, int g, u32x4 (&f)[D / 16]) {
  const unsigned short *row = static_cast<const unsigned short *>(p) + at + 8 * g;
#pragma unroll
  for (int m = 0; m < D / 16; ++m) f[m] = *reinterpret_cast<const u32x4 *>(row + 16 * m);
  if (bf16) {
#pragma unroll
    for (int m = 0; m < D / 16; ++m)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const unsigned w = f[m][e];
        f[m][e] = pack_h2(lo_to_f32<__bf16>(w), hi_to_f32<__bf16>(w));
      }
  }
}

// ---- the backward in one pass (qfa_skv_pass.hip: head_dim 128, qfa_skv_pass64.hip: 64)
struct SkvPassArgs {
  const void *q; const int8_t *codes; const void *scale; const int8_t *zp;
  const void *o; const float *lse; const void *dout;
  void *dq, *dkv;
  const float *grad_scale;     // nullable device scalar: dQ and dKV are multiplied by it before rounding (where not direct)
  int64_t H;
  int Nq, Nk, BH, io_bf16, scale_dtype;
  int direct, do_bf16;   // q, o (io_bf16) and dO as the caller has them, dO scaled here (grad_scale is not used)
  int64_t sqb, sqh, sqn, scb, sch, scn, sob, soh, son, sdob, sdoh, sdon, sdqb, sdqh, sdqn, sdkb, sdkh, sdkn;
  float sm_scale, sm_scale_log2;
};
int launch_skv_pass128(const SkvPassArgs &a, unsigned grid, bool grad_bf16, hipStream_t st);

}  // namespace qfa
