// The kernel of a backward: workgroups of dK and dV (qfa_bwd_dkv.inc), and behind them workgroups of dQ (qfa_bwd_dq.inc), in ONE launch.
//
// Neither reads what the other writes, and both take a SIMD's registers and most of a CU's LDS (one workgroup per CU, two at head_dim
// 64).  As two launches each left CUs idle: all that its blocks do not fill, the last round of a launch, and the time between the two.
// dK and dV come first: their workgroups take longer, so those of dQ fill up what they leave.  Either goes out alone where
// the parts of one take the memory of the other's, or one launch does not hold both (BwdPlan::sum_between).
// Measured, the whole backward with two launches, each divided by itself, and now, us, bf16, one GPU: 8 heads of 1000 x 128 causal 64 -> 43;
// 18 x 805 x 128 62 -> 45; 45 x 1500 x 256 432 -> 360; 3 x 1866 x 64 causal 45 -> 35; 100 x 1000 x 128 causal 181 -> 148; 33 x 4626 x 128
// 1113 -> 1024; 525 x 140 x 64 causal 60 -> 51; 20 x 4000 x 64 364 -> 303; chips that both fill in whole rounds take as long as before
// (128 x 4096 x 128 causal 1636 -> 1631; 256 x 2048 x 64 causal 592 -> 584; 16 x 16384 x 128 5293 -> 5276).
// Counters of the last three and of 64 x 4096 x 256 causal: matrix pipe busy 55, 43, 70 and 51 % of the time at 2.04, 2.08, 1.79 and 1.98 GHz,
// waits 21, 27, 15 and 25 % of the waves' time, issue stalls 24, 28, 24 and 25 %: the long sequence is bound by power, the others are not.
#pragma once
#include <cstddef>

#include <type_traits>

#include "qfa_acc.h"
#include "qfa_bwd_common.h"

namespace qfa {

template <int D> struct DkvSmem : BwdSlab<D> {
  static constexpr int SLAB = BwdSlab<D>::SLAB;
  static constexpr int OFF_Q = 0, OFF_DO = OFF_Q + D / 32 * SLAB, OFF_QT = OFF_DO + D / 16 * SLAB,
                       OFF_C = OFF_QT + BwdWs<D>::T_BYTES, C_COPY = (BwdWs<D>::CQ_BYTES + 1023) / 1024 * 1024,
                       BUF = OFF_C + C_COPY;
  static_assert(3 * BUF <= 160 * 1024, "three tile buffers");
};

template <int D> struct DqSmem : BwdSlab<D> {
  static constexpr int SLAB = BwdSlab<D>::SLAB;
  static constexpr int OFF_K = 0, OFF_V = OFF_K + D / 32 * SLAB, OFF_KT = OFF_V + D / 16 * SLAB,
                       OFF_C = OFF_KT + BwdWs<D>::T_BYTES, C_COPY = (BwdWs<D>::CK_BYTES + 1023) / 1024 * 1024,
                       BUF = OFF_C + C_COPY;
  static_assert(3 * BUF <= 160 * 1024, "three tile buffers");
};

struct BwdPairArgs {
  BwdArgs dkv, dq;
  int dkv_wgs, dkv_part, dq_part;   // workgroups of dK and dV; of one part of either
};

// KB, QB: 32-row blocks per wave
template <typename T, int D, int KB, int QB, bool CAUSAL>
__global__ __launch_bounds__(256, D == 64 ? 2 : 1) void bwd_pair_kernel(BwdPairArgs args) {
#ifdef __HIP_DEVICE_COMPILE__   // (with the body in view the host pass of this compiler emits no launch stub)
  constexpr int BUF = DkvSmem<D>::BUF > DqSmem<D>::BUF ? DkvSmem<D>::BUF : DqSmem<D>::BUF;
  __shared__ __attribute__((aligned(256))) unsigned char smem[3 * BUF];
  if ((int)blockIdx.x < args.dkv_wgs) {
    const BwdArgs &a = args.dkv;
    constexpr int ARGS_AT = offsetof(BwdPairArgs, dkv);
    const int part = __builtin_amdgcn_readfirstlane((int)blockIdx.x / args.dkv_part), L = (int)blockIdx.x - part * args.dkv_part;
#include "qfa_bwd_dkv.inc"
  } else {
    const BwdArgs &a = args.dq;
    constexpr int ARGS_AT = offsetof(BwdPairArgs, dq);
    const int at = (int)blockIdx.x - args.dkv_wgs, part = __builtin_amdgcn_readfirstlane(at / args.dq_part), L = at - part * args.dq_part;
#include "qfa_bwd_dq.inc"
  }
#endif
}

template <typename T, int D, int KB, int QB> static void launch_pair_blocks(const BwdPairArgs &a, unsigned grid, bool causal, hipStream_t st) {
  if (causal) bwd_pair_kernel<T, D, KB, QB, true><<<dim3(grid), dim3(256), 0, st>>>(a);
  else bwd_pair_kernel<T, D, KB, QB, false><<<dim3(grid), dim3(256), 0, st>>>(a);
}

template <typename T, int D>
int launch_bwd_pair(const BwdArgs &dkv, int blocks_dkv, int splits_dkv, const BwdArgs &dq, int blocks_dq, int splits_dq, int64_t BH, bool causal, hipStream_t st) {
  BwdPairArgs a = {dkv, dq, 0, 8, 8};
  int64_t grid = 0;
  auto part = [&](BwdArgs &x, int64_t rows, int64_t streamed, int blocks, int splits, bool is_dq, int *wgs) {
    x.nblocks = (int)((rows + 128 * blocks - 1) / (128 * blocks));
    x.group_log2 = bwd_group_log2(streamed, D, is_dq);   // per head either streams codes and two 16-bit rows: 5 bytes per row and d
    const int64_t total = (int64_t)x.nblocks * BH;
    x.total_blocks = (int)std::min<int64_t>(total, 0x3fffffff);
    x.blocks_per_xcd = (x.total_blocks + 7) / 8;
    *wgs = x.blocks_per_xcd * 8;
    grid += (int64_t)*wgs * splits;
    return total <= 0x3fffffff;
  };
  if (splits_dkv > 0 && !part(a.dkv, dkv.Nk, dkv.Nq, blocks_dkv, splits_dkv, false, &a.dkv_part))
    return set_error(QFA_EUNSUPPORTED, "attn_bwd: too many key blocks for one launch");
  a.dkv_wgs = (int)grid;
  if (splits_dq > 0 && !part(a.dq, dq.Nq, dq.Nk, blocks_dq, splits_dq, true, &a.dq_part))
    return set_error(QFA_EUNSUPPORTED, "attn_bwd: too many query blocks for one launch");
  if constexpr (D == 128) {
    if (blocks_dkv == 2 && blocks_dq == 2) launch_pair_blocks<T, D, 2, 2>(a, (unsigned)grid, causal, st);
    else if (blocks_dkv == 2) launch_pair_blocks<T, D, 2, 1>(a, (unsigned)grid, causal, st);
    else if (blocks_dq == 2) launch_pair_blocks<T, D, 1, 2>(a, (unsigned)grid, causal, st);
    else launch_pair_blocks<T, D, 1, 1>(a, (unsigned)grid, causal, st);
  } else {
    // (head_dim 256: the registers hold the operands and accumulators of 32 keys; head_dim 64: of 32 keys in two waves per
    // SIMD, which share the issue slots better than one wave of 64 keys: 3 - 10 % faster, 20 % when the chip is not full)
    launch_pair_blocks<T, D, 1, 1>(a, (unsigned)grid, causal, st);
  }
  return check_launch("qfa_attn_bwd (dk, dv, dq)");
}

}  // namespace qfa
