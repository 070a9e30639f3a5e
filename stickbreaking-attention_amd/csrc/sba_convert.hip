// float32 operands of a caller, rounded to the 16-bit element type the matrix cores take.
//
// Bound by memory: 6 bytes per element.  One launch for q, k and v, because a small call is launches (2 x 8 heads x
// 1500 tokens x 64: 3.5 us for each of three conversions of 6 MB); 8 elements per lane, two 16-byte
// loads and one 16-byte store, four groups of a lane in flight.
#include "sba_kernels.hpp"

namespace sba {

constexpr int ROUND_GROUPS = 4;   // 8-element groups per lane

template <class H>
__global__ void __launch_bounds__(256) round_f32_kernel(const RoundArgs a) {
  typedef __attribute__((ext_vector_type(4))) float f4;
  typedef __attribute__((ext_vector_type(8))) float f8;
  typedef __attribute__((ext_vector_type(8))) H h8;
  const int64_t first = (int64_t)blockIdx.x * (256 * ROUND_GROUPS) + threadIdx.x;
  f4 lo[ROUND_GROUPS], hi[ROUND_GROUPS];
  h8* to[ROUND_GROUPS];
#pragma unroll
  for (int j = 0; j < ROUND_GROUPS; ++j) {
    const int64_t g = first + 256 * j;
    const int i = (g >= a.upto[0]) + (g >= a.upto[1]);
    const int64_t at = g - (i == 0 ? 0 : i == 1 ? a.upto[0] : a.upto[1]);
    to[j] = nullptr;
    if (g < a.upto[2]) {
      const f4* from = reinterpret_cast<const f4*>(i == 0 ? a.src[0] : i == 1 ? a.src[1] : a.src[2]) + 2 * at;
      to[j] = reinterpret_cast<h8*>(i == 0 ? a.dst[0] : i == 1 ? a.dst[1] : a.dst[2]) + at;
      lo[j] = from[0];
      hi[j] = from[1];
    }
  }
#pragma unroll
  for (int j = 0; j < ROUND_GROUPS; ++j)
    if (to[j] != nullptr) *to[j] = __builtin_convertvector(__builtin_shufflevector(lo[j], hi[j], 0, 1, 2, 3, 4, 5, 6, 7), h8);
}

hipError_t launch_round_f32(const RoundArgs& a, bool f16, hipStream_t s) {
  const dim3 grid((unsigned)((a.upto[2] + 256 * ROUND_GROUPS - 1) / (256 * ROUND_GROUPS))), block(256);
  if (f16) hipLaunchKernelGGL(round_f32_kernel<_Float16>, grid, block, 0, s, a);
  else hipLaunchKernelGGL(round_f32_kernel<__bf16>, grid, block, 0, s, a);
  return hipGetLastError();
}

}  // namespace sba
