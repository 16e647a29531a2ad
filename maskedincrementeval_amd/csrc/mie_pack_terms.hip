// Filter copies for MIE_DTYPE_F32_F16X2 (the form: mie_conv_mfma_impl.h): the three bf16 terms of the forms that keep them, the two fp16
// terms, the fp32 values in the same order, the scale.  Two launches a filter, once per weight update: the first writes what needs no scale and
// leaves the largest and the smallest group of its blocks, the second takes the scale from these and writes the fp16 terms.  Bound by
// memory (22 bytes a weight).
#include "mie_conv_mfma_impl.h"
#include "mie_pack_terms.h"

namespace {

// A thread: eight input channels of a tap and a column.  (co fastest, then the half of the 16 channels, the tap, the block of 16.)
__global__ __launch_bounds__(256) void k_f2_values(const float* __restrict__ f, float4* __restrict__ three, float* __restrict__ values,
                                                   unsigned* __restrict__ parts, long long groups, int kk, int cout) {
  unsigned most = 0u, least = ~0u;
  for (long long g = (long long)blockIdx.x * 256 + threadIdx.x; g < groups; g += (long long)gridDim.x * 256) {
    const int co = (int)(g % cout), half = (int)((g / cout) & 1);
    const long long t = g / cout / 2;
    const int tap = (int)(t % kk);
    const long long ci = t / kk * 16 + half * 8;
    float v[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] = f[((ci + j) * kk + tap) * cout + co];
    f2_put_values(values, t, half, co, cout, v, most, least);
    float4 pl[3];
    split3(v, pl);
#pragma unroll
    for (int q = 0; q < 3; ++q) three[((t * 3 + q) * 2 + half) * cout + co] = pl[q];
  }
  f2_put_parts(parts, most, least);
}

__global__ __launch_bounds__(256) void k_f2_split(const float* __restrict__ values, float4* __restrict__ terms, const unsigned* __restrict__ parts,
                                                  int blocks, float* __restrict__ end, long long groups, int cout) {
  __shared__ unsigned s_m[2][4];
  unsigned most = 0u, least = ~0u;
  for (int i = threadIdx.x; i < blocks; i += 256) most = max(most, parts[i]), least = min(least, parts[F2_PARTS + i]);
  f2_block_range(s_m, most, least);
  // the largest weight to [2^14, 2^15); marked as not fitting: infinities and NaN, weights too large or small altogether, groups 2^29 below
  int e = (int)(most >> 23) - 127;
  e = most == 0u ? 14 : e < -46 ? -46 : e > 74 ? 74 : e;
  const float scale = __int_as_float((127 + 14 - e) << 23);
  const bool fits = most == 0u || (most < 0x7f800000u && __uint_as_float(most) * scale < 32768.f && __uint_as_float(least) * scale >= 6.1035156e-5f);      // 2^-14
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    end[0] = f2_unscale(scale);
    end[1] = fits ? 1.f : 0.f;
    end[2] = most >= F2_HUGE ? 1.f : 0.f;
#pragma unroll
    for (int i = 3; i < 12; ++i) end[i] = 0.f;
  }
  const long long g = (long long)blockIdx.x * 256 + threadIdx.x;
  if (g >= groups) return;
  const int co = (int)(g % cout), half = (int)((g / cout) & 1);
  const long long t = g / cout / 2, at = (t * 4 + half) * cout + co, step = 2LL * cout;
  const float4 u = *reinterpret_cast<const float4*>(values + 4 * at), v = *reinterpret_cast<const float4*>(values + 4 * (at + step));
  const float w[8] = {u.x, u.y, u.z, u.w, v.x, v.y, v.z, v.w};
  float4 pl[2];
  split2(w, scale, pl);
#pragma unroll
  for (int q = 0; q < 2; ++q) terms[at + q * step] = pl[q];
}

}  // namespace

void mie_f2_split(void* terms, long long groups, int blocks, int cout, hipStream_t st) {
  float* const values = mie_f2_values(terms, groups), *const end = values + 8 * groups;
  hipLaunchKernelGGL(k_f2_split, dim3((unsigned)((groups + 255) / 256)), dim3(256), 0, st, values, (float4*)terms, mie_f2_parts(terms, groups), blocks,
                     end, groups, cout);
}

void mie_pack_f16x2(const float* filter, int cin, int kk, int cout, void* packed, hipStream_t st) {
  const long long groups = (long long)cin / 8 * kk * cout;
  const int blocks = mie_f2_blocks(groups);
  char* const terms = (char*)packed + 48 * groups;      // behind the three bf16 terms
  hipLaunchKernelGGL(k_f2_values, dim3(blocks), dim3(256), 0, st, filter, (float4*)packed, mie_f2_values(terms, groups), mie_f2_parts(terms, groups), groups,
                     kk, cout);
  mie_f2_split(terms, groups, blocks, cout, st);
}
