// Activation layout shared by the batched-prefill kernels (cq_prefill.hip,
// cq_pf_attention.hip).
#pragma once

#include "cq_device.h"

namespace cq {

// Activation layout of the GEMM inputs, chosen by the weights' format so the
// A operand needs no shuffle: int4 stores each 8-group in the order
// [0,4,1,5,2,6,3,7] with the odd elements divided by 16 (the unpack yields the
// odd nibbles as 16 n without a shift); int8 and fp16 keep natural order.
__device__ __forceinline__ int pf_pos(int k, bool int4) {
  if (!int4) return k;
  const int e = k & 7;
  return (k & ~7) | (e < 4 ? 2 * e : 2 * e - 7);
}
// value stored for element k.  The /16 is a power-of-two scale, exact for
// |v| >= 2^-10; below that v/16 falls in fp16's subnormal range and keeps
// fewer bits (at most 2^-21 absolute error on the element: half the 2^-24
// subnormal spacing, times 16).
__device__ __forceinline__ _Float16 pf_val(float v, int k, bool int4) {
  return (_Float16)((int4 && (k & 1)) ? v * 0.0625f : v);
}

// One 8-element group (natural order) in the layout of the weights' format.
__device__ __forceinline__ h8_t pf_group(h8_t v, bool int4) {
  if (!int4) return v;
  h8_t o;
#pragma unroll
  for (int e = 0; e < 8; ++e) o[pf_pos(e, true)] = pf_val((float)v[e], e, true);
  return o;
}

}  // namespace cq
