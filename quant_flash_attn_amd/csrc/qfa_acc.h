// Accumulators kept in AccVGPRs by hand.  With more than 256 registers per wave the compiler puts either all MFMA results
// into AccVGPRs (and copies every score out again) or none, and as C++ values accumulators are copied around wherever
// control flow joins, without the wait states that a copy behind an MFMA needs when the MFMA is inline assembly.  Here tile
// i of a wave's accumulators (32x32, 16 registers) IS a[16i : 16i+15]: the statements below name the registers, and every
// one of them clobbers all that the kernel has tiles in.  That keeps the compiler's values out of them ACROSS a statement; it
// does not keep it from using one of them between two statements, and there are stretches of a hundred instructions without
// one.  What does is the build: it reads the assembly of these files and fails if an instruction of the compiler's names a
// register that a statement uses, anywhere in the kernel, if one of the two rules below is broken, or if anything was
// spilled (acc_check.py).  The scores and the other MFMA results that vector instructions read use the builtins (files that
// include this are compiled with -amdgpu-mfma-vgpr-form: results in vector registers, wait states by the compiler).
//
// The caller keeps two rules: A and B of acc_mfma were written at least two instructions earlier, and acc_settle() stands
// between the last acc_mfma and the first acc_read.
#pragma once
#include <utility>

#include "qfa_device.h"

namespace qfa {

#define QFA_ACC_32 \
  "a0", "a1", "a2", "a3", "a4", "a5", "a6", "a7", "a8", "a9", "a10", "a11", "a12", "a13", "a14", "a15", \
  "a16", "a17", "a18", "a19", "a20", "a21", "a22", "a23", "a24", "a25", "a26", "a27", "a28", "a29", "a30", "a31"
#define QFA_ACC_64 QFA_ACC_32, \
  "a32", "a33", "a34", "a35", "a36", "a37", "a38", "a39", "a40", "a41", "a42", "a43", "a44", "a45", "a46", "a47", \
  "a48", "a49", "a50", "a51", "a52", "a53", "a54", "a55", "a56", "a57", "a58", "a59", "a60", "a61", "a62", "a63"
#define QFA_ACC_128 QFA_ACC_64, \
  "a64", "a65", "a66", "a67", "a68", "a69", "a70", "a71", "a72", "a73", "a74", "a75", "a76", "a77", "a78", "a79", \
  "a80", "a81", "a82", "a83", "a84", "a85", "a86", "a87", "a88", "a89", "a90", "a91", "a92", "a93", "a94", "a95", \
  "a96", "a97", "a98", "a99", "a100", "a101", "a102", "a103", "a104", "a105", "a106", "a107", "a108", "a109", "a110", "a111", \
  "a112", "a113", "a114", "a115", "a116", "a117", "a118", "a119", "a120", "a121", "a122", "a123", "a124", "a125", "a126", "a127"
#define QFA_ACC_256 QFA_ACC_128, \
  "a128", "a129", "a130", "a131", "a132", "a133", "a134", "a135", "a136", "a137", "a138", "a139", "a140", "a141", "a142", "a143", \
  "a144", "a145", "a146", "a147", "a148", "a149", "a150", "a151", "a152", "a153", "a154", "a155", "a156", "a157", "a158", "a159", \
  "a160", "a161", "a162", "a163", "a164", "a165", "a166", "a167", "a168", "a169", "a170", "a171", "a172", "a173", "a174", "a175", \
  "a176", "a177", "a178", "a179", "a180", "a181", "a182", "a183", "a184", "a185", "a186", "a187", "a188", "a189", "a190", "a191", \
  "a192", "a193", "a194", "a195", "a196", "a197", "a198", "a199", "a200", "a201", "a202", "a203", "a204", "a205", "a206", "a207", \
  "a208", "a209", "a210", "a211", "a212", "a213", "a214", "a215", "a216", "a217", "a218", "a219", "a220", "a221", "a222", "a223", \
  "a224", "a225", "a226", "a227", "a228", "a229", "a230", "a231", "a232", "a233", "a234", "a235", "a236", "a237", "a238", "a239", \
  "a240", "a241", "a242", "a243", "a244", "a245", "a246", "a247", "a248", "a249", "a250", "a251", "a252", "a253", "a254", "a255"
// eight tiles and up to eight fragments behind them
#define QFA_ACC_160 QFA_ACC_128, \
  "a128", "a129", "a130", "a131", "a132", "a133", "a134", "a135", "a136", "a137", "a138", "a139", "a140", "a141", "a142", "a143", \
  "a144", "a145", "a146", "a147", "a148", "a149", "a150", "a151", "a152", "a153", "a154", "a155", "a156", "a157", "a158", "a159"

// tile I += A.B; TILES: the wave's tiles (2, 4, 8 or 16 of them take the first 32, 64, 128 or 256
// AccVGPRs, the compiler has the others)
template <typename T, int I, int TILES> __device__ __forceinline__ void acc_mfma(u32x4 a, u32x4 b) {
  static_assert(I >= 0 && I < TILES && TILES <= 16, "a wave has 256 AccVGPRs");
#ifdef __HIP_DEVICE_COMPILE__
#define QFA_M(TYPE, REGS) \
  asm volatile("v_mfma_f32_32x32x16_" TYPE " a[%2:%3], %0, %1, a[%2:%3]" ::"v"(a), "v"(b), "n"(16 * I), "n"(16 * I + 15) : REGS)
  if constexpr (TILES <= 2) {
    if constexpr (__is_same(T, __bf16)) QFA_M("bf16", QFA_ACC_32);
    else QFA_M("f16", QFA_ACC_32);
  } else if constexpr (TILES <= 4) {
    if constexpr (__is_same(T, __bf16)) QFA_M("bf16", QFA_ACC_64);
    else QFA_M("f16", QFA_ACC_64);
  } else if constexpr (TILES <= 8) {
    if constexpr (__is_same(T, __bf16)) QFA_M("bf16", QFA_ACC_128);
    else QFA_M("f16", QFA_ACC_128);
  } else {
    if constexpr (__is_same(T, __bf16)) QFA_M("bf16", QFA_ACC_256);
    else QFA_M("f16", QFA_ACC_256);
  }
#undef QFA_M
#endif
}
// A fragments that stay in flight across a branch (an LDS read that the compiler does not know of may not have its register
// copied or spilled before it arrives): fragment F of eight IS a[128 + 4F : 131 + 4F], behind eight tiles.
// acc_request: the transposing read of 8 bytes at a0 + OFF and 8 at a1 + OFF + 256, to be waited for by count;
// acc_mfma_frag: tile I += fragment F . B
template <int F, int OFF> __device__ __forceinline__ void acc_request(unsigned a0, unsigned a1) {
  static_assert(F >= 0 && F < 8, "eight fragments");
#ifdef __HIP_DEVICE_COMPILE__
  asm volatile("ds_read_b64_tr_b16 a[%2:%3], %0 offset:%6\n\tds_read_b64_tr_b16 a[%4:%5], %1 offset:%7"
               ::"v"(a0), "v"(a1), "n"(128 + 4 * F), "n"(129 + 4 * F), "n"(130 + 4 * F), "n"(131 + 4 * F), "n"(OFF), "n"(OFF + 256)
               : QFA_ACC_160, "memory");
#endif
}
template <typename T, int I, int F> __device__ __forceinline__ void acc_mfma_frag(u32x4 b) {
  static_assert(I >= 0 && I < 8 && F >= 0 && F < 8, "eight tiles, eight fragments");
#ifdef __HIP_DEVICE_COMPILE__
#define QFA_M(TYPE) \
  asm volatile("v_mfma_f32_32x32x16_" TYPE " a[%1:%2], a[%3:%4], %0, a[%1:%2]" ::"v"(b), "n"(16 * I), "n"(16 * I + 15), \
               "n"(128 + 4 * F), "n"(131 + 4 * F) : QFA_ACC_160)
  if constexpr (__is_same(T, __bf16)) QFA_M("bf16");
  else QFA_M("f16");
#undef QFA_M
#endif
}
// Any registers: a[C : C+15] = (FIRST ? 0 : itself) + a[A : A+3] . b, A a constant operand that acc_request_const has put there
template <int C, int A, bool FIRST> __device__ __forceinline__ void acc_mfma_const(u32x4 b) {
  static_assert(C % 4 == 0 && A % 4 == 0 && C + 16 <= 256 && A + 4 <= 256 && (A + 4 <= C || A >= C + 16), "a wave has 256 AccVGPRs");
#ifdef __HIP_DEVICE_COMPILE__
  if constexpr (FIRST)
    asm volatile("v_mfma_f32_32x32x16_f16 a[%1:%2], a[%3:%4], %0, 0" ::"v"(b), "n"(C), "n"(C + 15), "n"(A), "n"(A + 3) : QFA_ACC_256);
  else
    asm volatile("v_mfma_f32_32x32x16_f16 a[%1:%2], a[%3:%4], %0, a[%1:%2]" ::"v"(b), "n"(C), "n"(C + 15), "n"(A), "n"(A + 3) : QFA_ACC_256);
#endif
}
// the transposing read of 8 bytes at a0 + OFF and 8 at a1 + OFF + 256 into a[A : A+3], which are there behind lds_wait_for<0>()
template <int A, int OFF> __device__ __forceinline__ void acc_request_const(unsigned a0, unsigned a1) {
#ifdef __HIP_DEVICE_COMPILE__
  asm volatile("ds_read_b64_tr_b16 a[%2:%3], %0 offset:%6\n\tds_read_b64_tr_b16 a[%4:%5], %1 offset:%7"
               ::"v"(a0), "v"(a1), "n"(A), "n"(A + 1), "n"(A + 2), "n"(A + 3), "n"(OFF), "n"(OFF + 256) : QFA_ACC_256, "memory");
#endif
}
// tile I = 0 (one statement for the tile: between statements that clobber the same registers the compiler puts wait states)
template <int I, int TILES> __device__ __forceinline__ void acc_zero_tile() {
#ifdef __HIP_DEVICE_COMPILE__
#define QFA_Z(N) "v_accvgpr_write_b32 a[%" #N "], 0\n\t"
#define QFA_Z16(REGS) \
  asm volatile(QFA_Z(0) QFA_Z(1) QFA_Z(2) QFA_Z(3) QFA_Z(4) QFA_Z(5) QFA_Z(6) QFA_Z(7) QFA_Z(8) QFA_Z(9) QFA_Z(10) QFA_Z(11) \
                   QFA_Z(12) QFA_Z(13) QFA_Z(14) QFA_Z(15)::"n"(16 * I), "n"(16 * I + 1), "n"(16 * I + 2), "n"(16 * I + 3), \
               "n"(16 * I + 4), "n"(16 * I + 5), "n"(16 * I + 6), "n"(16 * I + 7), "n"(16 * I + 8), "n"(16 * I + 9), \
               "n"(16 * I + 10), "n"(16 * I + 11), "n"(16 * I + 12), "n"(16 * I + 13), "n"(16 * I + 14), "n"(16 * I + 15) \
               : REGS)
  if constexpr (TILES <= 2) QFA_Z16(QFA_ACC_32);
  else if constexpr (TILES <= 4) QFA_Z16(QFA_ACC_64);
  else if constexpr (TILES <= 8) QFA_Z16(QFA_ACC_128);
  else QFA_Z16(QFA_ACC_256);
#undef QFA_Z16
#undef QFA_Z
#endif
}
template <int R> __device__ __forceinline__ float acc_read_reg() {
  float x = 0.f;
#ifdef __HIP_DEVICE_COMPILE__
  asm volatile("v_accvgpr_read_b32 %0, a[%1]" : "=v"(x) : "n"(R));
#endif
  return x;
}
template <int... I> __device__ __forceinline__ void acc_zero_tiles(std::integer_sequence<int, I...>) { (acc_zero_tile<I, sizeof...(I)>(), ...); }
// tiles 0 .. TILES-1 = 0
template <int TILES> __device__ __forceinline__ void acc_zero() { acc_zero_tiles(std::make_integer_sequence<int, TILES>{}); }
template <int R0, int... R> __device__ __forceinline__ f32x16 acc_read_regs(std::integer_sequence<int, R...>) {
  return f32x16{acc_read_reg<R0 + R>()...};
}
template <int I> __device__ __forceinline__ f32x16 acc_read() { return acc_read_regs<16 * I>(std::make_integer_sequence<int, 16>{}); }
// tiles T0 .. T0 + N - 1 times x (a factor per column); acc_settle() in front of it and behind it
template <int R> __device__ __forceinline__ void acc_write_reg(float x) {
#ifdef __HIP_DEVICE_COMPILE__
  asm volatile("v_accvgpr_write_b32 a[%1], %0" ::"v"(x), "n"(R) : QFA_ACC_160);
#endif
}
template <int R0, int... R> __device__ __forceinline__ void acc_scale_regs(float x, std::integer_sequence<int, R...>) {
  (acc_write_reg<R0 + R>(acc_read_reg<R0 + R>() * x), ...);
}
template <int T0, int N> __device__ __forceinline__ void acc_scale(float x) {
  acc_scale_regs<16 * T0>(x, std::make_integer_sequence<int, 16 * N>{});
}
__device__ __forceinline__ void acc_settle() { asm volatile("s_nop 15\n\ts_nop 15" ::: "memory"); }

// 32 rows of a row-major tensor from tiles T0 .. T0 + D/32 - 1, scaled and rounded (store_tile_rows)
template <typename T, int D, int T0, int... DB>
__device__ __forceinline__ void acc_store_rows_seq(std::integer_sequence<int, DB...>, float scale, unsigned char *stage, T *rows,
                                                   int64_t stride, int row0, int nrows, int lane, bool once) {
  const f32x16 acc[sizeof...(DB)] = {acc_read<T0 + DB>()...};
  store_tile_rows<T, D>(acc, scale, stage, rows, stride, row0, nrows, lane, once);
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // the stage may be written again
}
template <int D, int T0, int... DB>
__device__ __forceinline__ void acc_store_rows_f32_seq(std::integer_sequence<int, DB...>, float scale, float *rows, int64_t stride,
                                                       int row0, int nrows, int lane) {
  const f32x16 acc[sizeof...(DB)] = {acc_read<T0 + DB>()...};
  store_tile_rows_f32<D>(acc, scale, rows, stride, row0, nrows, lane);
}
template <int D, int T0>
__device__ __forceinline__ void acc_store_rows_f32(float scale, float *rows, int64_t stride, int row0, int nrows, int lane) {
  acc_store_rows_f32_seq<D, T0>(std::make_integer_sequence<int, D / 32>{}, scale, rows, stride, row0, nrows, lane);
}
template <typename T, int D, int T0>
__device__ __forceinline__ void acc_store_rows(float scale, unsigned char *stage, T *rows, int64_t stride, int row0, int nrows,
                                               int lane, bool once = false) {
  acc_store_rows_seq<T, D, T0>(std::make_integer_sequence<int, D / 32>{}, scale, stage, rows, stride, row0, nrows, lane, once);
}

// ---- INT8 scores that need no conversion: with 0x4B400000, the bits of 1.5 * 2^23, as their initial value the int32 results
// n (|n| <= 2^22 up to head_dim 256) are the bits of the float 1.5 * 2^23 + n, and the product that adds the zero-point
// term takes the bias out again in a k-slot of its own: A = -3072 times B = 4096 in an operand's low half.  All are integers
// below 2^24.
#define QFA_BIAS_BITS 0x4B400000
#define QFA_BIAS_A(T) (__is_same(T, __bf16) ? 0xC540u : 0xEA00u)
#define QFA_BIAS_B(T) (__is_same(T, __bf16) ? 0x4580u : 0x6C00u)

// ---- straight-line code written out: compile-time indices, and a fence the scheduler moves nothing across
template <int V> using ic = std::integral_constant<int, V>;
template <typename F, int... I> __device__ __forceinline__ void static_for_seq(F &&f, std::integer_sequence<int, I...>) { (f(ic<I>{}), ...); }
// f(ic<0>), ..., f(ic<N-1>)
template <int N, typename F> __device__ __forceinline__ void static_for(F &&f) { static_for_seq(f, std::make_integer_sequence<int, N>{}); }
#define QFA_FENCE() __builtin_amdgcn_sched_barrier(0)

}  // namespace qfa
