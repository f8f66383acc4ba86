// Workspace layout, arguments and small helpers shared by the backward kernels (qfa_bwd.hip: staging passes;
// qfa_bwd_pair.h: dK, dV and dQ).
#pragma once
#include "qfa_device.h"
#include "qfa_host.h"

namespace qfa {

// Rows streamed per step: 64, or 32 at head_dim 256, where a 64-row step of codes, 16-bit rows and transposed tile
// (80 KB) could not be double-buffered in a CU's 160 KB.
// Workspace layout: per (batch*head, query tile) a Q-side blob, then per (batch*head, key tile)
// a K-side blob.  Transposed tiles are [D][TILE] 16-bit values (128- or 64-byte rows), positions permuted.
template <int D> struct BwdWs {
  static constexpr int TILE = D > 128 ? 32 : 64;
  static constexpr int CSH = D > 128 ? 8 : 7;             // bits per digit of rq - D*zq (|.| <= 65280 at head_dim 256)
  static constexpr int T_BYTES = D * TILE * 2;            // one transposed tile
  static constexpr int CQ_BYTES = 5 * TILE * 4;           // digits (2 dwords/query), a, -lse*log2e, -delta
  static constexpr int CK_BYTES = 3 * TILE * 4;           // digits (2 dwords/key), key scale
  static constexpr int Q_BLOB = T_BYTES + CQ_BYTES;           // Qz^T, constants
  static constexpr int K_BLOB = T_BYTES + CK_BYTES;           // Kz^T, constants
};

struct BwdArgs {
  const int8_t *qc; const float *sq; const int8_t *zq; const int32_t *rq;
  const int8_t *kc; const float *sk; const int8_t *zk; const int32_t *rk;
  const void *v; const void *o; const void *dout; const float *lse;
  unsigned char *ws_q; unsigned char *ws_k;
  void *dq; void *dk; void *dv;
  int64_t H;
  int Nq, Nk;
  int tiles_q, tiles_k;
  int64_t sqb, sqh, sqn, skb, skh, skn, svb, svh, svn, sob, soh, son;
  int64_t sdob, sdoh, sdon, sdqb, sdqh, sdqn, sdkb, sdkh, sdkn, sdvb, sdvh, sdvn;
  float sm_scale, sm_scale_log2;
  int nblocks;          // query blocks (dq) or key blocks (dkdv) per (b,h)
  int total_blocks, blocks_per_xcd;
  const float *dout32;  // nullable: dO in fp32; the staging pass then writes the 16-bit one to do16, which is `dout`
  void *do16;
  int64_t sd32b, sd32h, sd32n;
  int grad_f32;         // dQ, dK, dV are fp32
  int per_split;        // streamed rows per part (a multiple of 64); all of them in one where not split
  int last_part;        // first row of the last part
  int64_t split_stride; // fp32 elements from one part's gradients to the next's
  int group_log2;       // causal: log2 of the number of heads whose blocks are dispatched together (set per launch)
};

// position of streamed row r (0..63, or 0..31 in a 32-row tile) inside a transposed tile: the order in which the 32x32
// accumulator layout hands out rows to a lane (two runs of 4 per 16-row MFMA k-slice)
__device__ __forceinline__ int perm_pos4(int r4) {   // r4 = r / 4
  return 32 * (r4 / 8) + 16 * ((r4 / 4) % 2) + 8 * (r4 % 2) + 4 * ((r4 / 2) % 2);
}
// byte offset of (column d, position pos) in a staged transposed tile: in the order in which the MFMA kernels read it, one
// 1 KB block per (16-row slice, 32 columns) with 32 bytes per column, the two 16-byte halves (k-groups) of columns 8-15
// and 24-31 swapped so that 16 consecutive columns read at one k-group hit 16 different slots of the 256-byte bank line.
template <int D> __device__ __forceinline__ int qt_offset(int d, int pos) {
  return (pos / 16 * (D / 32) + d / 32) * 1024 + d % 32 * 32 + (((pos / 8) % 2 ^ (d / 8) % 2) << 4) + pos % 8 * 2;
}

// ---- slab layout of row tiles in LDS (see the head of qfa_bwd_dkv.inc)
template <int D> struct BwdSlab {
  static constexpr int SLAB = BwdWs<D>::TILE * 32 + 128;   // bytes between slabs
};
// offset of row r, k-group g (16 bytes) inside a slab
__device__ __forceinline__ int slab_row(int r, int g) { return r * 32 + ((g ^ ((r >> 3) & 1)) << 4); }
// Copies of a tile go out one instruction (1 KB per wave) at a time: the four waves of a workgroup together keep the
// address unit busy for 16 cycles per instruction, and all of a tile's 44 in one burst would stall every wave for 700
// cycles at the turn of the tile (measured: 13 % of the dK / dV kernel).
//
// TILE rows of SLABS * 32 bytes -> slabs: 32 rows of a slab per piece, dealt to four waves
template <int TILE, int SLABS> struct SlabCopy {
  static constexpr int HALVES = TILE / 32, N = SLABS * HALVES / 4;   // pieces per wave
  static_assert(SLABS * HALVES % 4 == 0, "every wave copies the same number of pieces");
  unsigned off, stride;
  __device__ __forceinline__ SlabCopy(int lane, unsigned row_stride) : stride(row_stride) {
    const int row = lane / 2;
    off = (unsigned)row * row_stride + (unsigned)(((lane % 2) ^ ((row >> 3) & 1)) * 16);
  }
  // rows: valid rows (<= 0: none, nothing is fetched); rows past the end arrive as zeros
  __device__ __forceinline__ rsrc_t desc(const unsigned char *base, int rows) const {
    return make_rsrc(base, rows > 0 ? (unsigned)(rows - 1) * stride + SLABS * 32 : 0u);
  }
  __device__ __forceinline__ void piece(int i, rsrc_t rs, unsigned char *dst, int wave) const {
    const int p = wave * N + i, slab = p / HALVES, half = p % HALVES;
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (lptr_t)(dst + slab * (TILE * 32 + 128) + half * 1024), 16, (int)off,
                                             (int)((unsigned)(half * 32) * stride) + slab * 32, 0, 0);
  }
};
// A staged blob: T_BYTES of transposed tile dealt to four waves, and C_COPY bytes of constants behind it (with fewer pieces
// than waves several waves copy the same bytes)
template <int T_BYTES, int C_COPY> struct BlobCopy {
  static constexpr int N = T_BYTES / 4096 + 1;
  __device__ __forceinline__ static void piece(int i, rsrc_t rs, unsigned char *dst_t, unsigned char *dst_c, int wave, int lane) {
    if (i < N - 1) {
      const int p = wave * (N - 1) + i;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (lptr_t)(dst_t + p * 1024), 16, lane * 16, p * 1024, 0, 0);
    } else {
      const int p = wave % (C_COPY / 1024);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (lptr_t)(dst_c + p * 1024), 16, lane * 16, T_BYTES + p * 1024, 0, 0);
    }
  }
};

// dK and dV by `dkv`, dQ by `dq`, either of them or both in one launch (qfa_bwd_pair.h).  blocks: 32-row blocks per wave (2 only at
// head_dim 128), splits: parts of the streamed rows; 0: that part is not wanted
template <typename T, int D>
int launch_bwd_pair(const BwdArgs &dkv, int blocks_dkv, int splits_dkv, const BwdArgs &dq, int blocks_dq, int splits_dq, int64_t BH, bool causal, hipStream_t st);

}  // namespace qfa
