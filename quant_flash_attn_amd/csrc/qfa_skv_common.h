// Shared pieces of the shared-KV kernels (forward and backward): tile geometry and the helpers that
// turn INT8 codes into exact binary16 MFMA operands.
//
// A code byte c (two's complement) with its top bit flipped is the unsigned byte c + 128; placed
// under the constant high byte 0x64 it is the binary16 number 1152 + c exactly.  One XOR per dword
// and one byte permute per pair of elements therefore make a 16-bit MFMA operand out of codes, and
// the offset 1152 + zero_point is taken out again exactly by the kernels (a rank-1 MFMA update where
// the codes are contracted over d, a v_dot2 accumulation where they are contracted over tokens).
#pragma once
#include "qfa_device.h"
#include "qfa_host.h"

namespace qfa {

constexpr int SKV_TILE = 32;     // keys per tile
constexpr float SKV_RESCALE_THRESHOLD = 4.0f;   // p <= 2^4: p * scale stays inside binary16 for any fp16 K

__device__ __forceinline__ f32x16 mfma_h(u32x4 a, u32x4 b, f32x16 c) { return mfma_16b<_Float16>(a, b, c); }
// two unsigned bytes (positions A and A+1 of w) -> packed binary16 pair (1024 + byte)
template <int A> __device__ __forceinline__ unsigned magic_pair(unsigned w) {
  constexpr unsigned sel = 0x04000400u | (unsigned)A | ((unsigned)(A + 1) << 16);
  return __builtin_amdgcn_perm(0x64646464u, w, sel);
}
// 8 code bytes (two dwords) -> 8 binary16 values 1152 + code
__device__ __forceinline__ u32x4 expand_codes(unsigned w0, unsigned w1) {
  w0 ^= 0x80808080u;
  w1 ^= 0x80808080u;
  return u32x4{magic_pair<0>(w0), magic_pair<2>(w0), magic_pair<0>(w1), magic_pair<2>(w1)};
}
__device__ __forceinline__ unsigned pack_h2(float a, float b) { return pack2<_Float16>(a, b); }
// binary16 pair (1152 + za, 1152 + zb) from two zero points held in the low bytes of za and zb
__device__ __forceinline__ unsigned magic_zp_pair(unsigned za, unsigned zb) {
  return __builtin_amdgcn_perm(za, zb, 0x0c000c04u) ^ 0x64806480u;
}
// Operands of the rank-1 MFMA that removes the offset where codes are contracted over d:
//     sum_d (1152 + c_jd) x_d  -  (1152 + zp_j) * rs,      rs = sum_d x_d.
// The key side carries 1152 + zp_j in three k-slots, the query side -rs as three binary16 terms (33
// significant bits, every product exact in fp32).  When some |rs| of the block reaches 2^15 (`big`, decided
// for all queries of the MFMA together) the key side carries 32 * (1152 + zp_j) instead -- bits
// 0x7800 | (zp_j + 128), still exact -- and the query side -rs / 32, which extends the range to 2^21.
__device__ __forceinline__ bool offset_needs_x32(float rs) {
  return __builtin_amdgcn_ballot_w64(!(fabsf(rs) < 32768.0f)) != 0;
}
// dwords 0 and 1 of the key-side operand (the caller zeroes them outside k-group 0; dwords 2, 3 are zero)
__device__ __forceinline__ u32x2 offset_key_operand(unsigned z, bool big) {
  const unsigned cz = __builtin_amdgcn_perm(z, z, 0x0c000c04u) ^ (big ? 0x78807880u : 0x64806480u);
  return u32x2{cz, cz & 0xffffu};
}
// dwords 0 and 1 of the query-side operand
__device__ __forceinline__ u32x2 offset_query_operand(float rs, bool big) {
  const float x = big ? rs * 0.03125f : rs;
  const _Float16 h0 = (_Float16)x;
  const float r1 = x - (float)h0;
  const _Float16 h1 = (_Float16)r1;
  const _Float16 h2 = (_Float16)(r1 - (float)h1);
  return u32x2{pack_h2(-(float)h0, -(float)h1), pack_h2(-(float)h2, 0.f)};
}

// a token's scale out of the dword its tile copy left (a 16-bit scale in the low half)
template <typename S> __device__ __forceinline__ float scale_to_f32(unsigned w) {
  if constexpr (sizeof(S) == 4) return __builtin_bit_cast(float, w);
  else return lo_to_f32<S>(w);
}

// ds_read_b64_tr_b8, issued like lds_read_tr16_async: invisible to the compiler's wait bookkeeping
// (which would make it wait for every direct-to-LDS load in flight); use the result only after
// lds_wait_all() and through tie().
__device__ __forceinline__ u32x2 lds_read_tr8_async(unsigned addr) {
  u32x2 r;
  asm volatile("ds_read_b64_tr_b8 %0, %1" : "=v"(r) : "v"(addr) : "memory");
  return r;
}

// 16x16x32 MFMA, used on blocks of 16 queries: a 32-key tile is two 16-key row blocks of S^T and one
// k-step of the products contracted over keys.  A lane owns query lane%16 and the keys
// 16rb + 4(lane/16) + {0..3} of each tile.
__device__ __forceinline__ f32x4 mfma_h16(u32x4 a, u32x4 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
}
// Chunk swizzle of a code tile for the 16-query kernels: as Swz<D>, plus a term in row/16 so that the eight
// keys one transposing read touches (4G + {0..3} and 16 + 4G + {0..3}) fall into different bank groups.
template <int D> struct SwzSkv {
  static constexpr int CPR = D / 16;
  static __device__ __forceinline__ int swz(int row) {
    return D == 256 ? (row ^ ((row / 16) * 4)) % 16
           : D == 128 ? ((row / 2) ^ ((row / 16) * 4)) % 8 : ((row / 4) ^ ((row / 16) * 2)) % 4;
  }
};

// Copy of 32-key tile t of one (batch, head) into an LDS slot by direct global->LDS loads: the codes
// through `cp` (rows dense, chunks swizzled), then one dword per key for the scale and one for the zero
// point (sub-dword direct loads write lane l's zero-extended value to the dword at 4*l).  Rows past the
// end of the sequence read as zeros.  Copy::N + 2 vector-memory instructions per wave.
template <typename S, int D, typename Copy>
__device__ __forceinline__ void skv_issue_tile(const Copy &cp, unsigned char *slot, const unsigned char *codes_bh,
                                               const void *scale, const int8_t *zp, int64_t tk0, int t, int Nk,
                                               int64_t scn, int lane) {
  const int rows = min(SKV_TILE, Nk - t * SKV_TILE);
  const rsrc_t rs_k = make_rsrc(codes_bh + (int64_t)t * SKV_TILE * scn, (unsigned)((rows - 1) * (int)scn + D));
#pragma unroll
  for (int c = 0; c < Copy::N; ++c) cp.issue_one(rs_k, slot, 0, lane, c);
  const rsrc_t rs_s = make_rsrc(reinterpret_cast<const S *>(scale) + tk0 + (int64_t)t * SKV_TILE,
                                (unsigned)rows * (unsigned)sizeof(S));
  const rsrc_t rs_z = make_rsrc(zp + tk0 + (int64_t)t * SKV_TILE, (unsigned)rows);
  if (lane < SKV_TILE) {
    if constexpr (sizeof(S) == 4)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rs_s, (lptr_t)(slot + SKV_TILE * D), 4, lane * 4, 0, 0, 0);
    else
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rs_s, (lptr_t)(slot + SKV_TILE * D), 2, lane * 2, 0, 0, 0);
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rs_z, (lptr_t)(slot + SKV_TILE * D + SKV_TILE * 4), 1, lane, 0, 0, 0);
  }
}

// Workgroup -> (batch*head, workgroup of it).  Consecutive ids go round the 8 XCDs.  The workgroups of a (batch, head) run on
// one XCD close in time and share its L2 copy of the codes: whole heads are dealt to the XCDs in turn, which keeps all of
// them in the same region of memory (a cache of 256 heads, 8192 keys: 97 us, 100 with a contiguous eighth of the heads each).
// Few heads that 8 does not divide would leave XCDs idle (two heads ran on two of them): there every XCD takes a contiguous
// eighth of all pairs.  Ids past the last pair are not live.
struct XcdBlock {
  int bh, sub;
  bool live;
  __device__ __forceinline__ XcdBlock(int BH, int per_bh) {
    const unsigned xcd = blockIdx.x % 8, at = blockIdx.x / 8;
    const bool whole = xcd_whole_heads(BH);
    const unsigned id = whole ? at : xcd * (gridDim.x / 8) + at, head = id / (unsigned)per_bh;
    bh = (int)(whole ? head * 8 + xcd : head);
    sub = (int)(id - head * (unsigned)per_bh);
    live = bh < BH;
  }
};

// Codes that one workgroup reads, and nobody again before as much as the last-level cache holds has passed: their loads are
// non-temporal then (the cache hint of a buffer load) and leave the caches to others.  Whoever shares codes between workgroups
// (several blocks of queries, or lines that hold rows of two heads: rows_own_lines), or finds them in that cache when it is called
// again, loses by it: up to 30 % for a decoding loop over one cache of 200 MB.
constexpr int LOAD_ONCE = 2;

// wait for every LDS operation of this wave; `tie` keeps the users of an asynchronously loaded
// register pair behind the wait that precedes it in program order
__device__ __forceinline__ void lds_wait_all() { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); }
__device__ __forceinline__ u32x2 tie(u32x2 w) {
  asm volatile("" : "+v"(w));
  return w;
}

// ---- the power of two by which dO is scaled (see dout_max_kernel, qfa_skv_bwd.hip)
template <typename T> __device__ __forceinline__ float max_abs8(const u32x4 w, float m) {
#pragma unroll
  for (int e = 0; e < 4; ++e) m = fmaxf(m, fmaxf(fabsf(lo_to_f32<T>(w[e])), fabsf(hi_to_f32<T>(w[e]))));
  return m;
}
// largest magnitude of the 16 bytes of scales a thread loads at a time
template <typename S> __device__ __forceinline__ float max_abs_chunk(const u32x4 w, float m) {
  if constexpr (sizeof(S) == 2) {
    return max_abs8<S>(w, m);
  } else {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const unsigned x = w[e];   // (this compiler's bit cast of a vector's element takes element 0)
      m = fmaxf(m, fabsf(__builtin_bit_cast(float, x)));
    }
    return m;
  }
}
__device__ __forceinline__ float block_max_256(float m, float *red) {
  for (int off = 32; off > 0; off >>= 1) m = fmaxf(m, __shfl_xor(m, off, 64));
  __syncthreads();
  if (threadIdx.x % 64 == 0) red[threadIdx.x / 64] = m;
  __syncthreads();
  return fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
}
// floor(log2(c / y)) for c = 2^ce and a positive normal y, exactly (no logarithm): y = m * 2^e with m in [1, 2)
__device__ __forceinline__ int floor_log2_quot(int ce, float y) {
  const unsigned b = __builtin_bit_cast(unsigned, y);
  const int e = (int)((b >> 23) & 0xff) - 127;
  return ce - e - ((b & 0x7fffffu) != 0 ? 1 : 0);
}

// k of the largest magnitudes of dO (m), of the key scales (ms) and of sm_scale * delta (md).  What the kernels round to binary16
// is dS = p * (sm_scale * dP - sm_scale * delta) and that times its key's scale.  m * 2^k * ms <= 8 bounds the first term by
// 8 * 255 * head_dim * sm_scale (32640 at most for 1 / sqrt(head_dim)).  It bounds the second term too where ms is the largest scale
// of all keys that O is made of; a workgroup that looks at the scales of a part of them passes md, which is kept below 2^15.
__device__ __forceinline__ int dout_exponent(float m, float ms, float md = 0.f) {
  m = fmaxf(m, 1e-30f);     // inf stays inf: k = -100 below
  ms = fmaxf(ms, 1e-30f);
  md = fmaxf(md * fmaxf(ms, 1.0f), 1e-30f);
  return max(-100, min(100, min(min(floor_log2_quot(3, m * ms), floor_log2_quot(14, m)), floor_log2_quot(15, md))));
}
// sum of O * dO over N x 8 values, O in binary16
template <int N> __device__ __forceinline__ float dot_dout(const u32x4 (&o)[N], const u32x4 (&w)[N], int bf16) {
  float sum = 0.f;
  auto add = [&](auto type) __attribute__((always_inline)) {
    typedef decltype(type) T;
#pragma unroll
    for (int i = 0; i < N; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const unsigned ow = o[i][e], dw = w[i][e];
        sum += lo_to_f32<_Float16>(ow) * lo_to_f32<T>(dw) + hi_to_f32<_Float16>(ow) * hi_to_f32<T>(dw);
      }
  };
  if (bf16) add(__bf16{});
  else add(_Float16{});
  return sum;
}
// |sm_scale * delta| for dout_exponent: a row that is not finite has no say in how the others are scaled
__device__ __forceinline__ float finite_abs(float x) { return fabsf(x) <= 3.4e38f ? fabsf(x) : 0.f; }
// eight bf16 values as binary16
__device__ __forceinline__ u32x4 half_of_bf16(u32x4 w) {
  u32x4 r;
#pragma unroll
  for (int e = 0; e < 4; ++e) r[e] = pack2<_Float16>(lo_to_f32<__bf16>(w[e]), hi_to_f32<__bf16>(w[e]));
  return r;
}
// largest magnitude of N x 8 values of dO; the same times 2^k, as binary16.  (One branch on the type around all of them: selected
// value by value, dQ of 99 x 53 heads, 97 x 689 takes 5 us of 490 more.)
template <int N> __device__ __forceinline__ float max_abs_dout(const u32x4 (&w)[N], int bf16) {
  float m = 0.f;
  if (bf16) {
#pragma unroll
    for (int i = 0; i < N; ++i) m = max_abs8<__bf16>(w[i], m);
  } else {
#pragma unroll
    for (int i = 0; i < N; ++i) m = max_abs8<_Float16>(w[i], m);
  }
  return m;
}
template <int N> __device__ __forceinline__ void scale_dout(u32x4 (&w)[N], int bf16, int k) {
  const float f = __builtin_ldexpf(1.0f, k);
  if (bf16) {
#pragma unroll
    for (int i = 0; i < N; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const unsigned x = w[i][e];
        w[i][e] = pack2<_Float16>(lo_to_f32<__bf16>(x) * f, hi_to_f32<__bf16>(x) * f);
      }
  } else if (k >= -14 && k <= 15) {   // 2^k is a normal binary16 number: one rounding too
    const f16x2 f2 = {(_Float16)f, (_Float16)f};
#pragma unroll
    for (int i = 0; i < N; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const unsigned x = w[i][e];
        w[i][e] = __builtin_bit_cast(unsigned, __builtin_bit_cast(f16x2, x) * f2);
      }
  } else {
#pragma unroll
    for (int i = 0; i < N; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const unsigned x = w[i][e];
        w[i][e] = pack2<_Float16>(lo_to_f32<_Float16>(x) * f, hi_to_f32<_Float16>(x) * f);
      }
  }
}
// The largest of n key scales (fp32 or fp16) from k0 on, as one of 256 threads finds it: the first thousand are requested here
// and looked at with the others later, so that the rows that the caller loads in between hide them.
struct KeyScaleMax {
  const void *p;
  int n, tid;
  bool f32;
  float first[4];
  __device__ __forceinline__ float at(int j) const {
    return f32 ? static_cast<const float *>(p)[j] : (float)static_cast<const _Float16 *>(p)[j];
  }
  __device__ __forceinline__ KeyScaleMax(const void *scale, int dtype, int64_t k0, int n_, int tid_) : n(n_), tid(tid_), f32(dtype == QFA_F32) {
    p = f32 ? static_cast<const void *>(static_cast<const float *>(scale) + k0)
            : static_cast<const void *>(static_cast<const _Float16 *>(scale) + k0);
    if (f32) {
#pragma unroll
      for (int i = 0; i < 4; ++i) first[i] = static_cast<const float *>(p)[min(tid + 256 * i, n - 1)];
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i) first[i] = (float)static_cast<const _Float16 *>(p)[min(tid + 256 * i, n - 1)];
    }
  }
  __device__ __forceinline__ float get() const {
    float ms = fmaxf(fmaxf(fabsf(first[0]), fabsf(first[1])), fmaxf(fabsf(first[2]), fabsf(first[3])));
#pragma unroll 8
    for (int j = tid + 1024; j < n; j += 256) ms = fmaxf(ms, fabsf(at(j)));
    return ms;
  }
};
// Every load so far has arrived.  For the end of a prologue whose branches leave loads that one side never reads (KeyScaleMax): the
// compiler then guards their registers wherever the main loop first writes them, and that wait is for the next tile's loads as well
// (dQ of 99 x 53 heads, 97 x 689: 485 us with such waits in the loop, 452 with this one in front of it).
__device__ __forceinline__ void wait_loads() { __builtin_amdgcn_s_waitcnt(0x0f70); }   // vmcnt(0), the other counters at their maximum
// 2^-k, in a scalar register
__device__ __forceinline__ float exp2_neg(int k) {
  const int bits = (127 - k) << 23;   // |k| <= 100
  return __builtin_bit_cast(float, __builtin_amdgcn_readfirstlane(bits));
}
// dout_exponent of 256 threads' m, ms and md; red: 12 floats of LDS that nobody uses
__device__ __forceinline__ int block_dout_exponent(float m, float ms, float md, float *red) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    m = fmaxf(m, __shfl_xor(m, off, 64));
    ms = fmaxf(ms, __shfl_xor(ms, off, 64));
    md = fmaxf(md, __shfl_xor(md, off, 64));
  }
  if (threadIdx.x % 64 == 0) {
    red[threadIdx.x / 64] = m;
    red[4 + threadIdx.x / 64] = ms;
    red[8 + threadIdx.x / 64] = md;
  }
  __syncthreads();
  m = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
  ms = fmaxf(fmaxf(red[4], red[5]), fmaxf(red[6], red[7]));
  md = fmaxf(fmaxf(red[8], red[9]), fmaxf(red[10], red[11]));
  return __builtin_amdgcn_readfirstlane(dout_exponent(m, ms, md));
}

}  // namespace qfa
