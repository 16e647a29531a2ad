// What the kernels that pack two-term filter copies share (mie_pack_terms.hip, mie_upconv2x.hip).  `groups` groups of eight weights in two
// terms: the terms (32 bytes a group), the fp32 values (32), MIE_F16X2_END_BYTES, in which the blocks' ranges stand behind the first 48.
#pragma once
#include "mie_conv.h"

constexpr int F2_PARTS = 1024;      // blocks of the first launch, at most
static_assert(MIE_F16X2_END_BYTES == 48 + 2 * 4 * F2_PARTS, "a range per block");

static inline int mie_f2_blocks(long long groups) {
  const long long b = (groups + 255) / 256;
  return (int)(b < F2_PARTS ? b : F2_PARTS);
}
static inline float* mie_f2_values(void* terms, long long groups) { return (float*)terms + 8 * groups; }
static inline unsigned* mie_f2_parts(void* terms, long long groups) { return (unsigned*)terms + 16 * groups + 12; }
// The terms and the scale from the values and `blocks` ranges.
void mie_f2_split(void* terms, long long groups, int blocks, int cout, hipStream_t st);
// A whole [cin][kk][cout] filter: its three bf16 terms (48 bytes a group), then the above.
void mie_pack_f16x2(const float* filter, int cin, int kk, int cout, void* packed, hipStream_t st);

// The eight weights of a group (block of 16 channels x tap `t`, half, column) to their places, and their largest into the range, as bits of magnitudes
// (NaN above the infinities); groups of zeros do not count for the least.
static __device__ __forceinline__ void f2_put_values(float* values, long long t, int half, int co, int cout, const float (&v)[8], unsigned& most,
                                                     unsigned& least) {
  const long long at = (t * 4 + half) * cout + co;
  *reinterpret_cast<float4*>(values + 4 * at) = make_float4(v[0], v[1], v[2], v[3]);
  *reinterpret_cast<float4*>(values + 4 * (at + 2LL * cout)) = make_float4(v[4], v[5], v[6], v[7]);
  unsigned m = 0u;
#pragma unroll
  for (int j = 0; j < 8; ++j) m = max(m, __float_as_uint(v[j]) & 0x7fffffffu);
  most = max(most, m);
  if (m != 0u) least = min(least, m);
}
// The range over the block's threads, to all of them.
static __device__ __forceinline__ void f2_block_range(unsigned (&s_m)[2][4], unsigned& most, unsigned& least) {
#pragma unroll
  for (int d = 32; d > 0; d >>= 1) most = max(most, (unsigned)__shfl_xor((int)most, d)), least = min(least, (unsigned)__shfl_xor((int)least, d));
  if ((threadIdx.x & 63) == 0) s_m[0][threadIdx.x >> 6] = most, s_m[1][threadIdx.x >> 6] = least;
  __syncthreads();
#pragma unroll
  for (int k = 0; k < 4; ++k) most = max(most, s_m[0][k]), least = min(least, s_m[1][k]);
}
static __device__ __forceinline__ void f2_put_parts(unsigned* parts, unsigned most, unsigned least) {
  __shared__ unsigned s_m[2][4];
  f2_block_range(s_m, most, least);
  if (threadIdx.x == 0) parts[blockIdx.x] = most, parts[F2_PARTS + blockIdx.x] = least;
}
