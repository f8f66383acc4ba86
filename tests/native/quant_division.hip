// The quantizer's quotient (quant_quotient) against the IEEE division, for every pair of significands: one thread per scale
// significand (2^23), 2^10 significands of an element of 11 bits each (for the long form: of 24 bits, 2^10 of them spread
// over the range by the caller's `offset`).  wrong[0]: pairs that differ.
#include "../../quant_flash_attn_amd/csrc/qfa_quant_row.h"

template <bool SHORT> __global__ __launch_bounds__(256) void compare(unsigned offset, unsigned long long *wrong) {
#pragma clang fp contract(off)
  const float scale = __builtin_bit_cast(float, 0x3f800000u | (blockIdx.x * 256 + threadIdx.x));
  const float r = qfa::quant_reciprocal(scale);
  unsigned n = 0;
  for (unsigned m = 0; m < 1024; ++m) {
    const float x = __builtin_bit_cast(float, 0x3f800000u | (m << 13) | offset);
    n += qfa::quant_quotient<SHORT>(x, scale, r) != x / scale;
  }
  if (n) atomicAdd(wrong, (unsigned long long)n);
}

// offset: 0 in the short form, below 2^13.  wrong: one counter in device memory, set to zero by the caller.
extern "C" int compare_quotients(int short_form, unsigned offset, unsigned long long *wrong, hipStream_t stream) {
  if (offset >= 8192u || (short_form && offset)) return -1;
  if (short_form) compare<true><<<dim3((1 << 23) / 256), dim3(256), 0, stream>>>(0u, wrong);
  else compare<false><<<dim3((1 << 23) / 256), dim3(256), 0, stream>>>(offset, wrong);
  return (int)hipGetLastError();
}
