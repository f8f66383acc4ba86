// Which loads through a buffer descriptor of `records` bytes arrive as zeros: every one whose vector and scalar offset together reach
// past the descriptor's end, also where the scalar offset alone does and where the descriptor is empty.
#include "../../quant_flash_attn_amd/csrc/qfa_device.h"

using namespace qfa;

// One workgroup of 64 lanes: lane l loads at 16 * l + soffset of the words behind `base`, once straight to LDS and once in each of the
// widths that the kernels use.  out: [6][64][4] words, the bytes read (the rest of a narrow load's words is zero).
__global__ __launch_bounds__(64) void load_all(const unsigned *base, unsigned records, unsigned soffset, unsigned *out) {
  __shared__ __attribute__((aligned(256))) unsigned char smem[1024];
  const int lane = threadIdx.x;
  const rsrc_t rs = make_rsrc(base, records);
  reinterpret_cast<u32x4 *>(smem)[lane] = u32x4{~0u, ~0u, ~0u, ~0u};
  __syncthreads();
  __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (lptr_t)smem, 16, lane * 16, (int)soffset, 0, 0);
  dma_wait();
  __syncthreads();
  u32x4 r[6];
  r[0] = reinterpret_cast<const u32x4 *>(smem)[lane];
  r[1] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rs, lane * 16, (int)soffset, 0));
  const u32x2 w = __builtin_bit_cast(u32x2, __builtin_amdgcn_raw_buffer_load_b64(rs, lane * 16, (int)soffset, 0));
  r[2] = u32x4{w[0], w[1], 0u, 0u};
  r[3] = u32x4{(unsigned)__builtin_amdgcn_raw_buffer_load_b32(rs, lane * 16, (int)soffset, 0), 0u, 0u, 0u};
  r[4] = u32x4{(unsigned)(unsigned short)__builtin_amdgcn_raw_buffer_load_b16(rs, lane * 16, (int)soffset, 0), 0u, 0u, 0u};
  r[5] = u32x4{(unsigned)(unsigned char)__builtin_amdgcn_raw_buffer_load_b8(rs, lane * 16, (int)soffset, 0), 0u, 0u, 0u};
#pragma unroll
  for (int i = 0; i < 6; ++i) reinterpret_cast<u32x4 *>(out)[i * 64 + lane] = r[i];
}

// base: `bytes` of device memory that hold every load, whatever the descriptor says
extern "C" int load_through_descriptor(const unsigned *base, unsigned bytes, unsigned records, unsigned soffset, unsigned *out, hipStream_t stream) {
  if (soffset > bytes || bytes - soffset < 64 * 16 || records > bytes) return -1;
  load_all<<<dim3(1), dim3(64), 0, stream>>>(base, records, soffset, out);
  return (int)hipGetLastError();
}
