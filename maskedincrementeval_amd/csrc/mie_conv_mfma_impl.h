// Kernel and launch templates of the matrix-core conv path, included by one translation unit per
// element type (mie_conv_mfma_f32.hip, mie_conv_mfma_bf16.hip) so that they compile in parallel.
//
// Masked conv on the matrix cores, gfx950: fp32 deltas with v_mfma_f32_32x32x2_f32, bf16 deltas
// with v_mfma_f32_32x32x16_bf16 (fp32 accumulation, fp32 reservoirs).  The two element types share
// one kernel: every operand access is a 16-byte access, which holds 4 fp32 or 8 bf16 channels, so
// the bf16 kernel is the fp32 kernel with twice the channels per LDS stage, per unit and per load.
// The text below gives the fp32 numbers.  Two more forms multiply fp32 deltas at fp32 accuracy on the 16-bit instructions: X3 (three
// bf16 terms per value, six term products per multiply; described at the kernel template) and F2 (two fp16 terms, three products; described
// beside split2), which is what fp32 deltas take by default wherever it exists.
//
// Work decomposition.  One 256-thread workgroup (4 waves) computes one active
// 8x8 output tile (M = 64 pixels) x CO_BLK output channels as an implicit GEMM
// over k = (input channel, tap):
//   * A (pixels x k): the input tile plus halo is staged in LDS, CC input
//     channels at a time, by all 256 threads with 16-byte loads of the NHWC
//     rows; pixels whose mask byte is 0 (or that lie outside the image) are
//     zero-filled without touching HBM.  The global loads of chunk c+1 are in
//     flight (in registers) while chunk c is multiplied; fp32 stride-1 tiles
//     also double-buffer the LDS copy, the others store it between two barriers.
//   * B (k x channels): units of the matrix-core filter copy (mie_pack_filter) are
//     read straight from L2 into a register ring, 16 bytes per lane (each value is
//     used by exactly one wave of the workgroup), 3 to 8 units ahead of the MFMAs
//     that consume them.
//   * The 4 waves split the workgroup's work WN ways over output channels and
//     WK = 4/WN ways over k (units = tap x 8-channel sub-chunk, round robin).
//     Layers with few tiles (33x44 bottleneck: 30 tiles) take WN=1, WK=4 so
//     that tiles x Cout/32 workgroups of 4 busy waves fill the chip; wide
//     layers take WN=4.  K-split partial sums meet in LDS and are added in a
//     fixed order (bit-reproducible).
//   * Epilogue: plain delta, or reservoir update + activation increment (values
//     fetched at kernel start in the k-split variants), or -- GATES -- the whole
//     ConvLSTM gate chain on the four gate columns of each hidden channel.
// A lane's operand layout: lanes 0-31 = the 32 pixels of an M block, the lane
// half selects 4 of the 8 channels of a sub-chunk, read as ONE ds_read_b128
// that feeds 4 k-steps (k-step j pairs channel j of the low half with channel
// 4+j of the high half; the B operand is loaded with the same pairing).  The
// LDS layout (pixel stride CC+4 dwords, row pitch 32 mod 64 dwords, half swap
// for stride 2) keeps the 16-byte reads of 16 neighbouring lanes on disjoint banks.
//
// What bounds it (measured on MI355X).  A register-only loop of the same MFMAs sustains 27.2 ns per
// v_mfma_f32_32x32x2_f32 and wave (64 cycles at 2.36 GHz; 152-155 TFLOP/s over the chip, constant or random
// operands alike) -- and 13.8 ns per v_mfma_f32_32x32x16_bf16 with constant operands but 20.6 ns (1.63 PFLOP/s,
// 0.65 of the nominal peak) with random ones: the bf16 rate is power-limited by the data.  In this kernel a
// 3x3 chunk of 72 MFMAs per wave takes 2.92 us = 40.6 ns per MFMA (one workgroup per CU, 3x3 256->256 at
// 33x44), a 5x5 chunk of 200 about 6.2 us = 31 ns.  Builds with parts of the loop compiled out (timing only)
// put the 3x3 kernel at 28.8 us complete, 27.6 without the A reads from LDS, 24.3 without any load, store or
// barrier in the loop; of those 24.3 us, 5.6 are tile pick, first staging round trip and epilogue.  The
// chunk hand-over, the B prefetch depth, the staging depth (64 channels per chunk), 8-wave workgroups, a
// third resident workgroup per CU (registers cut to fit) and splitting the contraction of the decoder convs
// over two or four workgroups were each built and measured: none moved a layer by more than 2 %, the last
// three for the worse.  Launches of a few workgroups per CU stay quantised: ceil(workgroups / 256) rounds.
// The X3 form does the same 3x3 chunk's work in 54 MFMAs of 32 cycles, 0.95 us, and takes 2.4 us for it: with one wave
// per SIMD nothing overlaps that wave's own staging work (88 VALU instructions to split a chunk's values, address
// arithmetic, waits -- the load counter is in order, so a filter prefetch behind the staging loads waits for them).
// A three-chunk software pipeline with two staging register sets changed nothing (19.8 us either way) and was removed;
// so were two extra waves that did all the staging with loads in flight four chunks ahead (chunk 2.2 -> 1.9 us, but a
// longer head: 20.8 -> 20.5 us).  With every filter load and LDS read of the loop made cache-resident on top of that
// (timing only) the chunk still takes 1.5 us: the staging latency is 0.3 us of it, all memory effects 0.7 us.
#pragma once
#include "mie_conv.h"
#include <stdlib.h>
#include <type_traits>

namespace {

typedef float v16f __attribute__((ext_vector_type(16)));
#ifndef MIE_PIPE
#define MIE_PIPE 1
#endif

// Build-time instrumentation (-DMIE_WG_PROFILE, measurement builds only): thread 0 of every workgroup
// records the 100 MHz device clock at the stages of its life into a buffer handed over with
// mie_set_profile_buffer, 16 slots per workgroup (slot 15 = number of stamps).  Compiled out otherwise.
#ifdef MIE_WG_PROFILE
static __device__ long long* mie_prof_buf;       // set by mie_set_profile_buffer (measurement builds only)
#define MIE_STAMP(k)                                                                                   \
  do {                                                                                                 \
    if (mie_prof_buf != nullptr && threadIdx.x == 0 && (k) < 15) {                                     \
      long long* slot_ = mie_prof_buf + (((long long)blockIdx.z * gridDim.y + blockIdx.y) * gridDim.x + blockIdx.x) * 16; \
      slot_[(k)] = (long long)wall_clock64();                                                          \
      if ((k) == 0) slot_[12] = (long long)clock64();                                                  \
      if ((k) == 14) slot_[13] = (long long)clock64();                                                 \
      slot_[15] = (k) + 1;                                                                             \
    }                                                                                                  \
  } while (0)
#else
#define MIE_STAMP(k) do { } while (0)
#endif

// fp32 channels staged in LDS per chunk (bf16: twice as many), by kernel size and stride, bounded
// by 64 KB of LDS.  Stride 1 double-buffers the staged tile of (7+K)^2 pixels.  Stride 2 tiles
// are (14+K)^2 pixels: they are single-buffered (the next chunk waits in registers and is
// stored between two barriers), which affords the same depth as stride 1 -- and with it the
// 4-way k-split that fills the chip on planes of a few dozen tiles; HALF is the shallower
// variant for channel counts that are not a multiple of the full depth.
__host__ __device__ constexpr int stage_channels(int K, int S, bool HALF = false) {
  return ((K <= 5) ? 32 : 16) / (HALF ? 2 : 1);
}
// x extent of a grid in the XCD-aware launch order: the tile capacity rounded up to a multiple of 8, plus 16 (the shares of active
// and of stale work are rounded up separately).  The kernel works its place out of it by the same formula: gridDim.x would be
// one more trip to the launch's packet.
__host__ __device__ constexpr int xcd_grid_x(int cap) { return ((cap + 7) & ~7) + 16; }
// bf16 tiles are single-buffered at stride 1 as well: a bf16 workgroup spends a few microseconds on
// the matrix cores, so what hides its latencies is the number of workgroups resident on the CU (LDS
// per workgroup halves), not the overlap inside one (measured: +10 % on the 8x480x640 decoder conv).
__host__ __device__ constexpr int stage_buffers(int S, int elem_size) { return (S == 1 && elem_size == 4) ? 2 : 1; }

// LDS dwords per row of the staged input tile.  The 16-byte operand reads of 16 neighbouring lanes
// (8 pixels of one tile row and of the next) must fall on 64 distinct banks: the pixel stride
// (CC + 4 dwords) spreads one row over every other group of 4 banks, and a row pitch of
// 32 (mod 64) dwords puts the next row on the groups in between (stride 1).  For stride 2 the
// pixel stride doubles and every row falls on the same bank groups whatever the pitch; there
// the two 16-byte halves of a unit are swapped in every other pair of input rows instead
// (`swz` below), which moves the neighbouring tile row by 4 banks.
__host__ __device__ constexpr int row_pitch_dw(int it, int ls_dw, int s) {
  int rp = it * ls_dw;
  if (s == 1)
    while (rp % 64 != 32) rp += 4;
  return rp;
}

// Ring size of the B-operand prefetch: the smallest divisor of the units per chunk that is
// at least 4, so that ring slot (unit % ring) means the same registers in every chunk.
__host__ __device__ constexpr int ring_size(int upc, int least = 4) {
  for (int r = least; r < upc; ++r)
    if (upc % r == 0) return r;
  return upc;
}

// Unit positions per chunk for the k-split over taps: at least n, padded until the ring size is at most 6
// (the extra positions hold no unit for any wave and compile to nothing).
__host__ __device__ constexpr int pad_units(int n) {
  while (ring_size(n) > 6) ++n;
  return n;
}

typedef float v4f __attribute__((ext_vector_type(4)));

// Waves per SIMD the register allocation must leave room for.  The stride-2 5x5 bf16 kernels stage a 19x19 tile
// (52 KB of LDS: three workgroups fit a CU) and spend two thirds of a workgroup's life outside the MFMA loop
// (tile pick, mask bytes, the one staging round trip, a 128-column epilogue), so a third resident workgroup
// is what fills the matrix cores; their natural allocation (172 registers) stops at two.
#ifndef MIE_S2_WAVES
#define MIE_S2_WAVES 3
#endif
__host__ __device__ constexpr int conv_min_waves(int elem_size, int K, int S, bool HALF, bool GATES, bool UP, bool SPLIT,
                                                 bool X3) {
  if (X3) return 2;      // 64 accumulator registers: the three-term kernels sit at the edge of two waves per SIMD
  return (elem_size == 2 && S == 2 && K == 5 && !HALF && !GATES && !UP && !SPLIT) ? MIE_S2_WAVES : 1;
}

// One unit of the contraction on the matrix core: the 16 bytes of A and of B a lane holds.
__device__ __forceinline__ void mma_unit(v16f& acc, const float4& av, const float4& bv, float) {
  acc = __builtin_amdgcn_mfma_f32_32x32x2f32(av.x, bv.x, acc, 0, 0, 0);
  acc = __builtin_amdgcn_mfma_f32_32x32x2f32(av.y, bv.y, acc, 0, 0, 0);
  acc = __builtin_amdgcn_mfma_f32_32x32x2f32(av.z, bv.z, acc, 0, 0, 0);
  acc = __builtin_amdgcn_mfma_f32_32x32x2f32(av.w, bv.w, acc, 0, 0, 0);
}
__device__ __forceinline__ void mma_unit(v16f& acc, const float4& av, const float4& bv, mie_bf16) {
  const v4f a4 = {av.x, av.y, av.z, av.w}, b4 = {bv.x, bv.y, bv.z, bv.w};
  acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(mie_bf16x8, a4),
                                                __builtin_bit_cast(mie_bf16x8, b4), acc, 0, 0, 0);
}

// The same for the two pixel blocks of a tile against one B operand, the k-steps of the two accumulators
// interleaved: consecutive MFMAs are independent, so none waits for the result of the one before it.
__device__ __forceinline__ void mma_unit2(v16f& acc0, v16f& acc1, const float4& a0, const float4& a1, const float4& bv, float) {
  acc0 = __builtin_amdgcn_mfma_f32_32x32x2f32(a0.x, bv.x, acc0, 0, 0, 0);
  acc1 = __builtin_amdgcn_mfma_f32_32x32x2f32(a1.x, bv.x, acc1, 0, 0, 0);
  acc0 = __builtin_amdgcn_mfma_f32_32x32x2f32(a0.y, bv.y, acc0, 0, 0, 0);
  acc1 = __builtin_amdgcn_mfma_f32_32x32x2f32(a1.y, bv.y, acc1, 0, 0, 0);
  acc0 = __builtin_amdgcn_mfma_f32_32x32x2f32(a0.z, bv.z, acc0, 0, 0, 0);
  acc1 = __builtin_amdgcn_mfma_f32_32x32x2f32(a1.z, bv.z, acc1, 0, 0, 0);
  acc0 = __builtin_amdgcn_mfma_f32_32x32x2f32(a0.w, bv.w, acc0, 0, 0, 0);
  acc1 = __builtin_amdgcn_mfma_f32_32x32x2f32(a1.w, bv.w, acc1, 0, 0, 0);
}
__device__ __forceinline__ void mma_unit2(v16f& acc0, v16f& acc1, const float4& a0, const float4& a1, const float4& bv, mie_bf16) {
  mma_unit(acc0, a0, bv, mie_bf16());
  mma_unit(acc1, a1, bv, mie_bf16());
}

// X3 (fp32 deltas multiplied as three bf16 terms each): v = hi + mid + lo with every term rounded to nearest
// even, so |mid| <= 2^-9 |v|, |lo| <= 2^-18 |v| and the three terms carry all 24 bits of v.  The six products
// hi*hi, hi*mid, mid*hi, hi*lo, mid*mid, lo*hi are exact in the fp32 accumulator's input; what is left out
// (mid*lo, lo*mid, lo*lo) is at most 2^-23 of |a*b| and typically 2^-26 (an fp32 multiply-add rounds at 2^-24); the
// measured error of whole convs against fp64 is 0.6-0.8 of the fp32 instruction's in the same decomposition.  (Non-finite values do
// not survive the split: inf - inf is NaN.)
typedef float v2f __attribute__((ext_vector_type(2)));
typedef __bf16 mie_bf16x2 __attribute__((ext_vector_type(2)));
// two values at a time: one packed conversion per term, the bf16 pair widened again with a shift and a mask
__device__ __forceinline__ void split3_pair(float f0, float f1, float& p0, float& p1, float& p2) {
  const v2f v = {f0, f1};
  const mie_bf16x2 hi = __builtin_convertvector(v, mie_bf16x2);
  const unsigned uh = __builtin_bit_cast(unsigned, hi);
  const v2f r1 = {f0 - __builtin_bit_cast(float, uh << 16), f1 - __builtin_bit_cast(float, uh & 0xffff0000u)};
  const mie_bf16x2 mid = __builtin_convertvector(r1, mie_bf16x2);
  const unsigned um = __builtin_bit_cast(unsigned, mid);
  const v2f r2 = {r1[0] - __builtin_bit_cast(float, um << 16), r1[1] - __builtin_bit_cast(float, um & 0xffff0000u)};
  const mie_bf16x2 lo = __builtin_convertvector(r2, mie_bf16x2);
  p0 = __builtin_bit_cast(float, hi);
  p1 = __builtin_bit_cast(float, mid);
  p2 = __builtin_bit_cast(float, lo);
}
__device__ __forceinline__ void split3(const float (&f)[8], float4 (&pl)[3]) {
  split3_pair(f[0], f[1], pl[0].x, pl[1].x, pl[2].x);
  split3_pair(f[2], f[3], pl[0].y, pl[1].y, pl[2].y);
  split3_pair(f[4], f[5], pl[0].z, pl[1].z, pl[2].z);
  split3_pair(f[6], f[7], pl[0].w, pl[1].w, pl[2].w);
}
// F2 (fp32 deltas multiplied as two fp16 terms each): v * s = hi + lo with s a power of two, hi = v * s rounded to fp16, lo the
// rest of it, kept as lo * 2^11 so that it has the exponents of hi.  The two carry 23 bits of v, sign included, and the three products
// hi*hi, lo*hi, hi*lo (what is left out, lo*lo, is at most 2^-24 of |a*b|) are exact in the fp32 accumulator's input: half the
// matrix instructions of the three bf16 terms, two thirds of their LDS and filter bytes.  Only one rounding a unit at the size of
// the sum instead of three (the cross products are added up among themselves) more than pays for the bit: error of whole contractions
// against fp64, relative 2-norm, of 288 / 1152 / 4608 terms in four chains 1.05 / 1.40 / 2.33e-7, three bf16 terms 1.09 / 1.89 /
// 3.70e-7.
// The price is fp16's range.  A workgroup takes s from the largest value of its first chunk (of both inputs'), which goes to [2^12, 2^13),
// so that a value is held to 2^-23 of itself or 2^-48 of that largest one, whichever is more.  The largest of every eight staged channels of a
// pixel has to lie below 65000 and not below 2^-12, or be zero: outputs that such groups alone make up are then no further from fp64 than three
// terms (norm of the error of 2304 terms, groups at 2^-12 .. -14: 2.4, 2.6, 3.5e-7, three terms 3.7e-7, far above it 2.3e-7).  (So the two terms
// hold 2^-24 of a group's largest at the least, also for its small values.)
// Over the networks' steps the largest value of a window was up to 3.5 times its first chunk's, and such groups lay within 2^24 of it but for a few
// tiles of a recurrent state fed back (within 2^30, 2 tiles of 4767 2^36).  The threads note the chunks that do not fit, and the workgroup leaves
// its loop in front of the first of these and goes on from there in three bf16 terms: X3's planes of the input, and the terms of the filter split
// in registers, from an fp32 copy behind its two.  Where a value is too large for these (F2_HUGE: infinities, NaN) all of it is done over on
// v_mfma_f32_32x32x2_f32.  us where all fit | all but the first chunk's channels 2^8 larger | half the pixels 2^-28 of the others, no chunk fits
// | three terms: 3x3 256->256 at 33x44 13.6 | 17.5 | 20.6 | 16.6, 64->64 at 132x176 14.4 | 18.1 | 20.8 | 16.8, 5x5 stride 2 128->256 at 66x88 17.3 |
// 22.1 | 25.9 | 23.5 (both contractions one after the other, the second on the fp32 instruction: 34, 32 and 45).  The look at every chunk costs
// 0.1-0.2 us a launch; at the end only, it would cost the whole of the two terms' contraction once more.
// The filter's scale takes its largest weight to [2^14, 2^15); a filter one of whose groups of eight input channels lies below 2^-29
// of it is marked, and contracted in three terms from the first chunk on.
typedef _Float16 mie_f16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 mie_f16x8 __attribute__((ext_vector_type(8)));
constexpr float F2_STEP = 2048.f;
// (as multiply-adds whose results are fp16: seven instructions a pair)
__device__ __forceinline__ void split2_pair(float f0, float f1, float s, float s_lo, float& p0, float& p1) {
  const mie_f16x2 hi = {(_Float16)__builtin_fmaf(f0, s, 0.f), (_Float16)__builtin_fmaf(f1, s, 0.f)};
  const mie_f16x2 lo = {(_Float16)__builtin_fmaf((float)hi[0], -F2_STEP, f0 * s_lo), (_Float16)__builtin_fmaf((float)hi[1], -F2_STEP, f1 * s_lo)};
  p0 = __builtin_bit_cast(float, hi);
  p1 = __builtin_bit_cast(float, lo);
}
__device__ __forceinline__ void split2(const float (&f)[8], float s, float4 (&pl)[2]) {
  const float s_lo = s * F2_STEP;
  split2_pair(f[0], f[1], s, s_lo, pl[0].x, pl[1].x);
  split2_pair(f[2], f[3], s, s_lo, pl[0].y, pl[1].y);
  split2_pair(f[4], f[5], s, s_lo, pl[0].z, pl[1].z);
  split2_pair(f[6], f[7], s, s_lo, pl[0].w, pl[1].w);
}
// Three bf16 terms of an operand that is there as fp32, its first four channels in the first half.
__device__ __forceinline__ void split3_raw(const float4 (&raw)[2], float4 (&pl)[3]) {
  const float f[8] = {raw[0].x, raw[0].y, raw[0].z, raw[0].w, raw[1].x, raw[1].y, raw[1].z, raw[1].w};
  split3(f, pl);
}
// (NaN if one of them is)
__device__ __forceinline__ float f2_max3(float a, float b, float c) { return __builtin_elementwise_maximum(__builtin_elementwise_maximum(a, b), c); }
__device__ __forceinline__ float f2_amax8(const float (&f)[8]) {
  const float m = f2_max3(fabsf(f[0]), fabsf(f[1]), fabsf(f[2]));
  return __builtin_elementwise_maximum(f2_max3(f2_max3(m, fabsf(f[3]), fabsf(f[4])), fabsf(f[5]), fabsf(f[6])), fabsf(f[7]));
}
// Largest magnitude of a wave's lanes (m >= 0), the same for all of them.
__device__ __forceinline__ float f2_wave_max(float m) {
  const auto step = [&](auto ctrl) {
    m = __builtin_elementwise_maximum(m, __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(m), decltype(ctrl)::value, 0xf, 0xf, false)));
  };
  step(std::integral_constant<int, 0x111>()); step(std::integral_constant<int, 0x112>());      // row_shr 1, 2, 4, 8
  step(std::integral_constant<int, 0x114>()); step(std::integral_constant<int, 0x118>());
  step(std::integral_constant<int, 0x142>()); step(std::integral_constant<int, 0x143>());      // row_bcast 15, 31
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(m), 63));
}
// The scale for values whose largest is m (anything: what does not fit is found later).  Zeros tell nothing of what follows: 2^73, which
// values above 2^-57 do not fit.
__device__ __forceinline__ float f2_scale(float m) {
  int e = (__float_as_int(m) >> 23) - 127;
  e = m == 0.f ? -61 : e < -60 ? -60 : e > 52 ? 52 : e;
  return __int_as_float((127 + 12 - e) << 23);
}
__device__ __forceinline__ float f2_unscale(float s) { return __int_as_float((254 << 23) - __float_as_int(s)); }      // 1 / s
constexpr unsigned F2_HUGE = (127u + 127u) << 23;      // bits of 2^127: from here on, infinities and NaN among them, values may have no finite bf16 terms
// The groups a thread stages: in terms at their scale, and noted.
struct F2Groups {
  float scale;
  unsigned most, least;                   // bits of the largest, bits less one of the least, zeros left out
  __device__ __forceinline__ void start(float s) { scale = s; most = 0u; least = ~0u; }
  __device__ __forceinline__ void note(const float (&f)[8]) {
    const unsigned u = __float_as_uint(f2_amax8(f));
    most = max(most, u);
    least = min(least, u - 1u);
  }
  __device__ __forceinline__ void terms(const float (&f)[8], float4 (&pl)[2]) {
    note(f);
    split2(f, scale, pl);
  }
  __device__ __forceinline__ bool huge() const { return most >= F2_HUGE; }
  __device__ __forceinline__ bool misfit() const {      // (the scale's exponent taken off the bounds)
    const unsigned k = __float_as_uint(scale) - (127u << 23), lo = (127u - 12u) << 23, hi = 0x477de800u;      // 2^-12, 65000
    return most > hi - k || least < lo - k - 1u;
  }
};
// What a filter copy of this form ends with: 1 / (its scale), whether all of it fits, and whether three bf16 terms do not hold it either.
template <typename T>
__device__ __forceinline__ const float* f2_filter_end(const T* filt_mc, long long weights) {
  return reinterpret_cast<const float*>(reinterpret_cast<const char*>(filt_mc) + 8 * weights);
}
__device__ __forceinline__ void mma_f16(v16f& acc, const float4& a, const float4& b) {
  const v4f a4 = {a.x, a.y, a.z, a.w}, b4 = {b.x, b.y, b.z, b.w};
  acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(mie_f16x8, a4), __builtin_bit_cast(mie_f16x8, b4), acc, 0, 0, 0);
}
__device__ __forceinline__ void mma_unit2_f2(v16f& acc0, v16f& acc1, v16f& sm0, v16f& sm1, const float4 (&a0)[2], const float4 (&a1)[2],
                                             const float4 (&b)[2]) {
  mma_f16(acc0, a0[0], b[0]); mma_f16(acc1, a1[0], b[0]);
  mma_f16(sm0, a0[1], b[0]);  mma_f16(sm1, a1[1], b[0]);
  mma_f16(sm0, a0[0], b[1]);  mma_f16(sm1, a1[0], b[1]);
}

// One unit (16 input channels of a tap) of the X3 contraction for the two pixel blocks of a tile: six bf16 MFMAs
// per block.  The three large products (hi*hi, mid*hi, hi*mid) and the three small ones (lo*hi, mid*mid, hi*lo, 2^-16 of
// the first) go to accumulators of their own, added in the epilogue: four independent chains, so that no MFMA
// waits for the one issued just before it, and the small terms are summed among themselves.
__device__ __forceinline__ void mma_unit2_x3(v16f& acc0, v16f& acc1, v16f& sm0, v16f& sm1, const float4 (&a0)[3],
                                             const float4 (&a1)[3], const float4 (&b)[3]) {
  mma_unit(acc0, a0[0], b[0], mie_bf16()); mma_unit(acc1, a1[0], b[0], mie_bf16());
  mma_unit(sm0, a0[2], b[0], mie_bf16());  mma_unit(sm1, a1[2], b[0], mie_bf16());
  mma_unit(acc0, a0[1], b[0], mie_bf16()); mma_unit(acc1, a1[1], b[0], mie_bf16());
  mma_unit(sm0, a0[1], b[1], mie_bf16());  mma_unit(sm1, a1[1], b[1], mie_bf16());
  mma_unit(acc0, a0[0], b[1], mie_bf16()); mma_unit(acc1, a1[0], b[1], mie_bf16());
  mma_unit(sm0, a0[0], b[2], mie_bf16());  mma_unit(sm1, a1[0], b[2], mie_bf16());
}

// One 16-byte slot of delta elements <-> fp32 values (4 of them, or 8 for bf16).
__device__ __forceinline__ void slot_to_f32(const float4& raw, float (&f)[4], float) {
  f[0] = raw.x; f[1] = raw.y; f[2] = raw.z; f[3] = raw.w;
}
__device__ __forceinline__ void slot_to_f32(const float4& raw, float (&f)[8], mie_bf16) {
  const v4f r4 = {raw.x, raw.y, raw.z, raw.w};
  const mie_bf16x8 b = __builtin_bit_cast(mie_bf16x8, r4);
#pragma unroll
  for (int e = 0; e < 8; ++e) f[e] = (float)b[e];
}
__device__ __forceinline__ float4 f32_to_slot(const float (&f)[4], float) { return make_float4(f[0], f[1], f[2], f[3]); }
__device__ __forceinline__ float4 f32_to_slot(const float (&f)[8], mie_bf16) {
  mie_bf16x8 b;
#pragma unroll
  for (int e = 0; e < 8; ++e) b[e] = (mie_bf16)f[e];
  const v4f r4 = __builtin_bit_cast(v4f, b);
  return make_float4(r4[0], r4[1], r4[2], r4[3]);
}

// One item of a gates conv: a pixel and four adjacent hidden channels, whose state values start at element `ho` and whose 16
// gate columns start at element `go` of the gate reservoir.  What the gate chain reads (of an item that is not on: whatever
// lies first), as one batch ...
struct GateItem {
  float4 r[4], cp, cc, dp;
};
template <typename T>
__device__ __forceinline__ void conv_gates_load(const ConvArgsT<T>& a, bool on, bool has_cp, long long ho, long long go, GateItem& g) {
  const float4* gr = reinterpret_cast<const float4*>(a.res + (on ? go : 0));
#pragma unroll
  for (int j = 0; j < 4; ++j) g.r[j] = gr[j];
  g.cp = *reinterpret_cast<const float4*>(a.g_cpres + (on ? ho : 0));
  g.cc = *reinterpret_cast<const float4*>(a.g_cres + (on ? ho : 0));
  g.dp = make_float4(0.f, 0.f, 0.f, 0.f);
  if (a.g_cpd != nullptr) {
    const float4 d = mie_ld4(a.g_cpd, on ? ho : 0);
    g.dp = make_float4(has_cp ? d.x : 0.f, has_cp ? d.y : 0.f, has_cp ? d.z : 0.f, has_cp ? d.w : 0.f);
  }
}
// ... and the chain, given the conv sums dg of its columns: reservoirs updated, state deltas written (of an item that is not
// on: clean zeros).
template <typename T>
__device__ __forceinline__ void conv_gates_item(const ConvArgsT<T>& a, bool on, bool has_cp, long long ho, long long go, const float4 (&dg)[4],
                                                GateItem& g) {
  if (!on) {
    mie_st4(a.g_dh, ho, make_float4(0.f, 0.f, 0.f, 0.f));
    mie_st4(a.g_dc, ho, make_float4(0.f, 0.f, 0.f, 0.f));
    return;
  }
  float cp[4] = {g.cp.x, g.cp.y, g.cp.z, g.cp.w}, cc[4] = {g.cc.x, g.cc.y, g.cc.z, g.cc.w};
  const float dP[4] = {g.dp.x, g.dp.y, g.dp.z, g.dp.w};
  float dh[4], dc[4];
  float4* gr = reinterpret_cast<float4*>(a.res + go);
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    mie_lstm_gate_chain(g.r[j].x, g.r[j].y, g.r[j].z, g.r[j].w, dg[j].x, dg[j].y, dg[j].z, dg[j].w, cp[j], dP[j], cc[j],
                        dh[j], dc[j]);
    gr[j] = g.r[j];
  }
  if (has_cp) *reinterpret_cast<float4*>(a.g_cpres + ho) = make_float4(cp[0], cp[1], cp[2], cp[3]);
  *reinterpret_cast<float4*>(a.g_cres + ho) = make_float4(cc[0], cc[1], cc[2], cc[3]);
  mie_st4(a.g_dh, ho, make_float4(dh[0], dh[1], dh[2], dh[3]));
  mie_st4(a.g_dc, ho, make_float4(dc[0], dc[1], dc[2], dc[3]));
}

// The arguments of the running kernel, whose first and largest is a ConvArgsT<T>, where the launch put them.  To be inlined
// into the kernel itself: in a function that is called there is no such place.
template <typename T>
__device__ __forceinline__ const ConvArgsT<T>& conv_args_again() {
  uint64_t at = (uint64_t)(const void*)__builtin_amdgcn_kernarg_segment_ptr();
  asm("" : "+s"(at));
  return *(const ConvArgsT<T>*)at;
}

__device__ __forceinline__ bool finite4(const float4& v) {
  return isfinite(v.x) && isfinite(v.y) && isfinite(v.z) && isfinite(v.w);
}

// Four output channels of a conv in plain fp32, straight from the inputs and the plain filter, with the epilogue: what is
// done instead where a sum of the three-term form is not finite.  That form makes NaN of an infinite delta and of a finite
// one that rounds to an infinite bf16 term (3.39e38 and more); either leaves no finite sum, so the test of the sum finds all
// of them, and finite sums cost that test only.  For the 5x5 stride-2 convs of few tiles with a workspace, which ran on the
// fp32 instruction before and carried such values (the others do not: mie.h, MIE_DTYPE_F32_BF16X3).  It runs behind the
// ordinary stores, over the groups these left out: inside them the loops cost registers (1-2 us a launch).  Alone, without
// -> with: 32->64 at 64x96 10.9 -> 11.1 us, split 64->128 at 32x48 11.2 -> 11.3; on planes of many tiles it would be
// 24.4 -> 24.7 (64->128 at 132x176) and 25.8 -> 26.5 (128->256 at 66x88).
// (The arguments are read from memory anew, through conv_args_again: taken from the kernel's `a`, a dozen fields more stayed
// in registers through the contraction, whose scalar spills cost 0.5-1.1 us a launch.)
template <typename T, int K, int S>
__device__ void conv_quad_again(const ConvArgsT<T>& a, int n, int oy, int ox, int co) {
  float4 s = make_float4(0.f, 0.f, 0.f, 0.f);
  for (int t = 0; t < K * K; ++t) {
    const int iy = oy * S - a.pad + t / K, ix = ox * S - a.pad + t % K;
    if (iy < 0 || iy >= a.h_in || ix < 0 || ix >= a.w_in) continue;
    const long long pix = ((long long)n * a.h_in + iy) * a.w_in + ix;
    for (int in = 0; in < 2; ++in) {
      const T* x = in ? a.x2 : a.x;
      const uint8_t* m = in ? a.x2m : a.xm;
      const int c = in ? a.c2 : a.c1, ci0 = in ? a.c1 : 0;
      if (x == nullptr || (m != nullptr && m[pix] == 0)) continue;
      for (int ci = 0; ci < c; ++ci) {
        const float v = mie_ld(x, pix * c + ci);
        const float* w = a.filt + ((long long)(ci0 + ci) * (K * K) + t) * a.cout + co;
        s.x = fmaf(v, w[0], s.x); s.y = fmaf(v, w[1], s.y); s.z = fmaf(v, w[2], s.z); s.w = fmaf(v, w[3], s.w);
      }
    }
  }
  const long long off = (((long long)n * a.ts.h + oy) * a.ts.w + ox) * a.cout + co;
  conv_store(a, off, co, s.x); conv_store(a, off + 1, co + 1, s.y); conv_store(a, off + 2, co + 2, s.z); conv_store(a, off + 3, co + 3, s.w);
}

// (tile, slab, part) of a workgroup of a split launch, whose grid is (slab x part, tile).  A few per cent of such a launch are its
// filter's way into the L2s: a filter slice, of one slab and part, is fetched by every XCD that has one of its tiles.  The hardware
// deals workgroups out to the XCDs in launch order, x fastest, so that where the slices are a multiple of 8 all tiles of a slice are on
// one XCD, an eighth of the slices on each; of other numbers the tiles of a slice spread over 8 / gcd(8, slices) of them (4 slices,
// one slab in four parts: two).  Whole passes, (tile, slab, part) grid -> this: optical flow
// 1x256x256 366.7 -> 361.7 us (transposed convs), 467.9 -> 459.5 (up-sampling), e2depth 1x128x128 246.4 -> 243.8, 1x64x96 181.1 -> 180.6
// (two tiles: a slice was on two XCDs).
template <typename T>
__device__ __forceinline__ void split_order(const ConvArgsT<T>& a, int& bx, int& by, int& bz) {
  const int slice = bx, lp = a.xcd_fs;        // (of a split launch: log2 of the parts)
  bx = by;
  by = slice >> lp;
  bz = slice - (by << lp);
}

// UP: the conv input is up2x(x + x2), the bilinear x2 up-sampling of the sum of two deltas given at
// half resolution (x2 optional), and is never formed in memory: per chunk the 8x8 block of source
// pixels a tile's 12x12 input window blends is summed into LDS (fp32), and the staged tile is expanded
// from there.  5x5, stride 1, pad 2 only; a.h_in / a.w_in are the up-sampled size.
//
// SPLIT: launches with very few tiles (a 16x16 plane is 4 of them) leave most CUs idle.  The staged
// chunks of every (tile, slab) are then split over up to 8 workgroups; each writes its partial sums,
// fp32 and unactivated, into its own plane of the workspace (a.ws, laid out like the output), and
// k_conv_split_finish adds the planes in a fixed order and runs the epilogue.  Only the 32-channel
// slab kernels (WN = 1) have this form.
//
// X3 (fp32 deltas only): the contraction runs on the bf16 matrix-core instruction at fp32 accuracy.  Every staged
// input value and every filter value is split into three bf16 terms (split3; the filter once, by
// mie_pack_filter); the staged tile is three bf16 planes in LDS, a unit is 16 input channels of a tap, and
// its six significant term products are six v_mfma_f32_32x32x16_bf16 per pixel block -- 6 x 32 cycles for what
// eight v_mfma_f32_32x32x2_f32 take 8 x 64 cycles to do.  Chunks of 32 channels (two units per tap; stride 2, whose
// staged tile is four times the size: 16 channels, one unit per tap); where the k-split has more waves than a tap
// has units it is over (sub-chunk, tap class).  Global loads, masks, epilogue: fp32.
//
// ARITH: 1 is X3, 2 the form F2 above, 0 neither.
// AGAIN (X3 only): outputs whose sum is not finite are computed again in fp32 (conv_quad_again).
// GRU (with GATES): the gate math of a ConvGRU in place of the ConvLSTM's chain; eight columns, update and candidate, to four
// hidden channels.
// WIDE (F2): eight waves and chunks of twice the channels; f2_wide says where.
template <typename T, int K, int S, int WN, int NB, bool HALF, bool GATES = false, bool UP = false, bool SPLIT = false,
          int ARITH = 0, bool AGAIN = false, bool GRU = false, bool WIDE = false>
// (Build with -mllvm -pragma-unroll-threshold=65536: the unit loop of the 128-column 5x5 / 7x7 kernels is 100 / 196
// positions long, and where the compiler refuses to unroll it the operand ring is indexed at run time and lands in
// scratch memory -- a factor of three in time.)
__global__ __launch_bounds__(WIDE ? 512 : 256, conv_min_waves((int)sizeof(T), K, S, HALF, GATES, UP, SPLIT, ARITH != 0)) void k_conv_mfma(ConvArgsT<T> a) {
  constexpr bool X3 = ARITH != 0, F2 = ARITH == 2;           // values in terms; in two of them
  static_assert(!X3 || (sizeof(T) == 4 && !HALF && (K == 3 || K == 5)), "X3: fp32 deltas, 3x3 / 5x5");
  using TL = std::conditional_t<X3, mie_bf16, T>;            // element type in LDS and on the matrix cores
  constexpr int PL = F2 ? 2 : X3 ? 3 : 1;                    // operand planes (terms per value)
  constexpr int GPS = X3 ? 2 : 1;                            // 16-byte global loads per staging slot
  constexpr int TH = WIDE ? 512 : 256, WAVES = TH / 64;
  static_assert(!WIDE || (F2 && !UP && !SPLIT), "eight waves: two terms");
  constexpr int NBUF = X3 ? (((K == 3 && S == 1) || WIDE) ? 2 : 1) : stage_buffers(S, (int)sizeof(T));
  constexpr int EPS = 16 / (int)sizeof(TL);                  // elements per 16-byte slot (4 / 8)
  constexpr int SUB = 2 * EPS;                               // channels per unit (8 / 16)
  constexpr int WK = WAVES / WN;
  constexpr int IT = 7 * S + K;                              // input tile edge incl. halo
  constexpr int CC = X3 ? (S == 2 ? 16 : 32) * (WIDE ? 2 : 1) : stage_channels(K, S, HALF) * (4 / (int)sizeof(T));   // channels per LDS stage
  constexpr int LS = CC + EPS;                               // LDS elements per staged pixel
  constexpr int NPIX = IT * IT;
  constexpr int Q4 = CC / EPS;                               // 16-byte slots per pixel
  constexpr int NSLOT = NPIX * Q4;
  constexpr int NLD = (NSLOT + TH - 1) / TH;                   // staging slots per thread
  constexpr int RP = row_pitch_dw(IT, LS * (int)sizeof(TL) / 4, S) * 4 / (int)sizeof(TL);   // elements per tile row
  constexpr bool ROOM = RP - IT * LS >= EPS;                 // a slot fits into the padding of a row
  constexpr int STAGE = IT * RP + (WIDE && !ROOM ? 4 * EPS : 0);   // elements per plane of a staging buffer
  constexpr int NQ = CC / SUB;                               // sub-chunks (units per tap) per stage
  // k-split: over whole sub-chunks (every wave takes NQW of them, for every tap), or -- more waves than sub-chunks,
  // X3 only -- one sub-chunk and every TP-th tap per wave (the last position of a chunk is then empty for some waves)
  constexpr bool TPAR = WK > NQ;
  static_assert(TPAR ? (X3 && WK % NQ == 0) : (NQ % WK == 0), "the k-split is over whole sub-chunks, or over taps");
  constexpr int TP = TPAR ? WK / NQ : 1;                     // tap classes
  constexpr int NQW = TPAR ? 1 : NQ / WK;                    // sub-chunks per wave
  constexpr int UPC = TPAR ? pad_units((K * K + TP - 1) / TP) : K * K * NQW;   // unit positions per chunk and wave
  constexpr int RING = (X3 && ring_size(UPC) > 6) ? ring_size(UPC, 3) : ring_size(UPC);   // B operand ring (divides UPC)
  constexpr int PD = RING - 1;                               // prefetch distance in units
  constexpr int CO_BLK = 32 * NB * WN;
  constexpr int RED = WK * 64 * CO_BLK;                      // every wave parks its accumulators here for the epilogue
  constexpr int PLANES = F2 && NBUF == 1 ? 3 : NBUF * PL;    // (F2: one buffer of three planes for what does not fit)
  constexpr int STAGE_F = PLANES * STAGE * (int)sizeof(TL) / 4;     // the staging buffers, in floats
  constexpr int LOS = CC;                                    // floats per source pixel in LDS
  constexpr int LO_F = UP ? 64 * LOS : 0;                    // fp32 sums of the 8x8 source block, CC channels
  static_assert(!UP || (S == 1 && K == 5 && !GATES), "the up-sampling variant is the 5x5 stride-1 conv");
  // the k-split reduction of the epilogue reuses the staging buffers and the source block
  constexpr int SMEM = (STAGE_F + LO_F > RED) ? STAGE_F + LO_F : RED;
  static_assert(SMEM * 4 <= (WIDE ? 160 * 1024 : 65536), "LDS budget");
  __shared__ __attribute__((aligned(16))) float smem[SMEM];
  __shared__ float s_f2[F2 ? WAVES + 3 : 1];                         // largest values of the waves' first slots; whether a group of a chunk does
                                                                     // not fit, of every other one in the same place: a fast wave may be one ahead
  static_assert(!F2 || !AGAIN, "two terms: what is not finite is contracted in fp32");
  TL* const sbuf = reinterpret_cast<TL*>(smem);
  float* const s_lo = smem + STAGE_F;

  // (tile-list position, slab, part) of this workgroup.  Each of the 8 XCDs has an L2 of its own and the
  // hardware hands workgroups to the XCDs round robin in launch order (x fastest); with a.xcd_fs > 0 the
  // grid's x extent is a multiple of 8, so the XCD of a workgroup is blockIdx.x % 8, and the launch order
  // is permuted.  The slabs are cut into a.xcd_fs groups; a group's 8 / xcd_fs XCDs take its (tile, slab) pairs in the order
  // (tile, slab within the group), tiles in list order, i.e. along the rows of the image, each a contiguous
  // share.  A slab of the filter then reaches 8 / xcd_fs
  // L2s instead of all 8, an input tile about xcd_fs of them, once, for all slabs of the group at a
  // time, and neighbouring tiles, which share their halo, meet in one L2 (measured on the 5x5 256->128
  // conv at 66x88: 65 -> 31 MB fetched per launch).  Active and stale tiles are dealt out separately
  // (a stale tile costs next to nothing); the shares depend on their numbers, read from the tile set; the list's entry is asked for
  // together with these, as if every tile were active, and again where they are not.  Idle positions of the capacity-sized grid
  // fall off the end.
  const int entry_zero = conv_args_entry_zero(a);      // every line of the argument block, fetched in one batch
  MIE_STAMP(0);
  int bx = blockIdx.x + entry_zero, by = blockIdx.y;
  int bz = 0;
  if constexpr (SPLIT) split_order(a, bx, by, bz);
  int n, y0, x0, tk;
  if (!SPLIT && a.xcd_fs > 0) {
    const int cap = a.ts.n * a.ts.tiles_y * a.ts.tiles_x;
    const int lg = __builtin_ctz(a.xcd_fs), sh = 3 - lg, up = (1 << sh) - 1;      // groups, XCDs of a group
    const int spg = (a.cout / CO_BLK) >> lg;                 // slabs per group
    const int xcd = bx & 7, k = xcd & up;
    const int slot = by * (xcd_grid_x(cap) >> 3) + (bx >> 3);                     // launch order within the XCD
    const int guess = mie_tile_div(k * ((cap * spg + up) >> sh) + slot, spg, a.xcd_m);
    TileAsk ask = mie_tile_ask(a.ts, guess);
    asm("" : "+s"(ask.spec), "+s"(ask.n_active), "+s"(ask.n_stale));
    const int n_act = ask.n_active, n_st = ask.n_stale;
    if (n_act < 0 || n_st < 0 || n_act > cap || n_st > cap) return;
    const int c_act = (n_act * spg + up) >> sh, c_st = (n_st * spg + up) >> sh;   // a share
    const bool active = slot < c_act;
    const int u = active ? k * c_act + slot : k * c_st + (slot - c_act);
    if (u >= (active ? n_act : n_st) * spg || (!active && slot - c_act >= c_st)) return;
    const int t = mie_tile_div(u, spg, a.xcd_m);
    by = (xcd >> sh) * spg + (u - t * spg);
    bx = active ? t : n_act + t;
    if (active && t != guess) ask.spec = a.ts.tiles[t];
    tk = mie_pick_tile_loaded(a.ts, bx, ask.spec, n_act, n_st, n, y0, x0);
  } else {
    tk = mie_pick_tile(a.ts, bx, n, y0, x0);
  }
  if (tk == 0) return;
  MIE_STAMP(1);
  const int tid = threadIdx.x;
  // wave index as a scalar: everything derived from it (k-split, channel slab) stays in SGPRs
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int l32 = lane & 31, half = lane >> 5;
  const int wn = wave % WN, wk = wave / WN;
  const int co0 = by * CO_BLK;
  const int hout = a.ts.h, wout = a.ts.w;
  const int cout = a.cout;

  static_assert(!SPLIT || (WN == 1 && !GATES), "the split form is a 32-channel slab kernel (the gates conv splits as a plain conv)");
  if (SPLIT && tk == 2) return;      // stale tiles are zeroed by k_conv_split_finish
  if (GATES && tk == 2) {  // stale tile: zero the hidden / cell deltas of this workgroup's hidden channels
    constexpr int HG = CO_BLK / (GRU ? 8 : 16);          // groups of four hidden channels
    for (int idx = tid; idx < 64 * HG; idx += TH) {
      const int p = idx / HG, g4 = idx - p * HG;
      const int oy = y0 + (p >> 3), ox = x0 + (p & 7);
      if (oy < hout && ox < wout) {
        const long long o = (((long long)n * hout + oy) * wout + ox) * a.hid + co0 / (GRU ? 2 : 4) + 4 * g4;
        mie_st4(a.g_dh, o, make_float4(0.f, 0.f, 0.f, 0.f));
        if (!GRU) mie_st4(a.g_dc, o, make_float4(0.f, 0.f, 0.f, 0.f));
      }
    }
    return;
  }
  if (tk == 2) {  // stale tile: zero this workgroup's channel slab
    for (int idx = tid; idx < 16 * CO_BLK; idx += TH) {       // groups of four channels
      const int p = idx / (CO_BLK / 4), col = 4 * (idx - p * (CO_BLK / 4));
      const int oy = y0 + (p >> 3), ox = x0 + (p & 7);
      if (oy < hout && ox < wout)
        mie_st4(a.out, (((long long)n * hout + oy) * wout + ox) * cout + co0 + col, make_float4(0.f, 0.f, 0.f, 0.f));
    }
    return;
  }

  // Epilogue (all but the gate chain): every wave parks its accumulators in LDS, and a thread then owns groups of
  // four adjacent output channels of a pixel -- 16-byte reads of the k-split partial sums, 16-byte reservoir
  // accesses, 16- / 8-byte delta accesses.  A thread's share of the output is fixed by its index, so in the k-split
  // fp32 kernels the reservoir / addend values are fetched once the mask bytes are there and have the whole contraction to
  // arrive.
  constexpr int QPP = CO_BLK / 4;                            // groups of four channels per pixel
  constexpr int PER = GATES ? 1 : 64 * QPP / TH;            // groups per thread
  constexpr int PB = PER > 4 ? 4 : PER;                      // groups per pass of the epilogue (registers)
  long long e_off[PB];
  int e_co[PB];
  bool e_ok[PB], e_live[PB];
  float4 e_r0[PB], e_add[PB];
  // bit g: group g of this thread lies on a pixel of the output pixel mask.  Elsewhere in an active tile the sums are
  // exactly zero: no reservoir access, a zero delta.
  unsigned live_bits = 0u;
  // (bf16: a workgroup's contraction is too short to be worth the registers that hold these values
  // through it -- they cost a resident workgroup per CU -- so they are fetched after it instead; the same
  // holds for the 128-column slabs, whose threads own 8 groups.)
  constexpr bool EARLY = sizeof(T) == 4 && WK > 1 && !(X3 && K == 5);
  static_assert(!EARLY || PER == PB, "the early fetch covers a thread's whole share");
  auto epilogue_fetch = [&](int h0) {
#pragma unroll
    for (int i = 0; i < PB; ++i) {
      const int idx = tid + TH * (h0 + i);
      const int p = idx / QPP, col = 4 * (idx - p * QPP);
      const int oy = y0 + (p >> 3), ox = x0 + (p & 7);
      e_ok[i] = oy < hout && ox < wout;
      e_live[i] = SPLIT ? e_ok[i] : ((live_bits >> (h0 + i)) & 1u) != 0;
      e_off[i] = (((long long)n * hout + oy) * wout + ox) * a.cout + co0 + col;
      e_co[i] = co0 + col;
    }
    if (!SPLIT) conv_epilogue_load4<T, PB>(a, e_off, e_live, e_r0, e_add);
  };

  v16f acc[2][NB];
  v16f accs[X3 ? 2 : 1][X3 ? NB : 1];      // X3: the small term products
#pragma unroll
  for (int mb = 0; mb < 2; ++mb)
#pragma unroll
    for (int nb = 0; nb < NB; ++nb)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        acc[mb][nb][r] = 0.f;
        if (X3) accs[mb][nb][r] = 0.f;
      }

  // ---- per-thread staging plan: which pixels / float4 slots this thread copies -------------
  const int iy0 = y0 * S - a.pad, ix0 = x0 * S - a.pad;
  int st_po[NLD];       // linear input pixel index
  int st_lds[NLD];      // LDS element offset of the slot
  int st_c4[NLD];       // channel offset of the slot inside the chunk
  unsigned ok1 = 0u, ok2 = 0u;   // slot readable from x / x2 (inside the image, pixel mask set)
  unsigned inb = 0u;             // slot inside the image
#pragma unroll
  for (int i = 0; i < NLD; ++i) {
    const int slot = tid + TH * i;
    const int pix = slot / Q4, q4 = slot - pix * Q4;
    const int lrow = pix / IT;
    const int swz = (S == 2) ? ((lrow >> 1) & 1) : 0;
    st_lds[i] = lrow * RP + (pix - lrow * IT) * LS + EPS * (q4 ^ swz);
    st_c4[i] = EPS * q4;
    st_po[i] = 0;
    if (!UP && slot < NSLOT) {
      const int iy = iy0 + pix / IT, ix = ix0 + pix % IT;
      if (iy >= 0 && iy < a.h_in && ix >= 0 && ix < a.w_in) {
        st_po[i] = (n * a.h_in + iy) * a.w_in + ix;
        inb |= 1u << i;
      }
    }
  }
  const int nch1 = (a.c1 + CC - 1) / CC;
  const int nch = nch1 + ((!UP && a.x2 != nullptr) ? (a.c2 + CC - 1) / CC : 0);

  // UP: the source block.  Rows iy0 .. iy0+11 of the up-sampled image (iy0 even) blend source rows
  // iy0/2 - 1 .. iy0/2 + 6; one 16-byte slot per (source pixel, channel group) and tensor.
  constexpr int NLO = UP ? (64 * Q4 + TH - 1) / TH : 1;
  const int h_lo = a.h_in >> 1, w_lo = a.w_in >> 1;
  const int lo_y0 = (iy0 >> 1) - 1, lo_x0 = (ix0 >> 1) - 1;
  int lo_po[NLO];
  unsigned lo_ok1 = 0u, lo_ok2 = 0u, lo_inb = 0u;
  float4 lo_a[NLO][GPS], lo_b[NLO][GPS];
  if (UP) {
#pragma unroll
    for (int i = 0; i < NLO; ++i) {
      const int slot = tid + TH * i;
      const int lpix = slot / Q4;
      const int ly = lo_y0 + (lpix >> 3), lx = lo_x0 + (lpix & 7);
      lo_po[i] = 0;
      if (lpix < 64 && ly >= 0 && ly < h_lo && lx >= 0 && lx < w_lo) {
        lo_po[i] = (n * h_lo + ly) * w_lo + lx;
        lo_inb |= 1u << i;
      }
    }
  }

  // The pixel-mask bytes a workgroup needs are one more dependent round trip at its start (tile id -> mask
  // bytes -> input loads).  Where the contraction has at least four chunks, the loads of the FIRST chunk
  // therefore go out for every pixel inside the image, before the mask bytes are there (`first`), and the
  // masked pixels are zeroed when they are stored; from the second chunk on -- and in layers of fewer
  // chunks, where that would be a large share of the reads -- a masked pixel is not fetched at all.
  float4 st_reg[NLD][GPS];
  auto load_slots = [&](float4 (&regs)[NLD][GPS], int c, bool first) __attribute__((always_inline)) {
    const bool second = c >= nch1;
    const T* xin = second ? a.x2 : a.x;
    const int cs = second ? a.c2 : a.c1;
    const int ci0 = (second ? c - nch1 : c) * CC;
    const unsigned ok = first ? inb : (second ? ok2 : ok1);
    // The loads are unconditional in control flow (a branch around a load makes the compiler's
    // wait counters conservative: the first MFMAs of a chunk would then wait for the whole
    // global-memory latency of these loads).  Lanes whose pixel is masked or outside the image
    // all read one fixed, cache-resident address instead, and zeros are selected when the slot is stored,
    // so inactive pixels still cost no HBM traffic.
    const T* dummy = a.filt_mc;
#pragma unroll
    for (int i = 0; i < NLD; ++i) {
      const bool okb = (ok >> i) & 1u;
      const T* p = xin + (long long)st_po[i] * cs + ci0 + st_c4[i];
      p = okb ? p : dummy;
#pragma unroll
      for (int g = 0; g < GPS; ++g) {
        regs[i][g] = *reinterpret_cast<const float4*>(p + 4 * g);
      }
    }
  };
  auto stage_load = [&](int c, bool first = false) __attribute__((always_inline)) {
    if constexpr (UP) {
      const T* dummy = a.filt_mc;
#pragma unroll
      for (int i = 0; i < NLO; ++i) {
        const int q4 = (tid + TH * i) % Q4;
        const long long eo = (long long)lo_po[i] * a.c1 + c * CC + EPS * q4;
        const bool k1 = ((first ? lo_inb : lo_ok1) >> i) & 1u;
        const bool k2 = first ? (a.x2 != nullptr && ((lo_inb >> i) & 1u)) : ((lo_ok2 >> i) & 1u);
#pragma unroll
        for (int g = 0; g < GPS; ++g) {
          lo_a[i][g] = *reinterpret_cast<const float4*>(k1 ? a.x + eo + 4 * g : dummy);
          lo_b[i][g] = *reinterpret_cast<const float4*>(k2 ? a.x2 + eo + 4 * g : dummy);
        }
      }
      return;
    }
    load_slots(st_reg, c, first);
  };
  // one staged slot to LDS: as it is, or (X3) its eight fp32 values as three bf16 planes
  F2Groups groups;
  float filt_form = 1.f;                    // F2: 1 where the filter fits, -1 where not even three terms hold it
  auto store_slot = [&](TL* dst, const float4 (&raw)[GPS]) __attribute__((always_inline)) {
    if constexpr (F2) {
      const float f[8] = {raw[0].x, raw[0].y, raw[0].z, raw[0].w, raw[GPS - 1].x, raw[GPS - 1].y, raw[GPS - 1].z, raw[GPS - 1].w};
      float4 pl[2];
      groups.terms(f, pl);
#pragma unroll
      for (int q = 0; q < 2; ++q) *reinterpret_cast<float4*>(dst + q * STAGE) = pl[q];
    } else if constexpr (X3) {
      const float f[8] = {raw[0].x, raw[0].y, raw[0].z, raw[0].w, raw[1].x, raw[1].y, raw[1].z, raw[1].w};
      float4 pl[3];
      split3(f, pl);
#pragma unroll
      for (int q = 0; q < 3; ++q) *reinterpret_cast<float4*>(dst + q * STAGE) = pl[q];
    } else {
      *reinterpret_cast<float4*>(dst) = raw[0];
    }
  };
  // F2, what does not fit: in three terms (2), or as it is (0), the first four channels of a slot in one plane, the others in the next
  auto store_unfit = [&](TL* dst, const float4 (&raw)[GPS], auto form) __attribute__((always_inline)) {
    if constexpr (F2) {
      const float f[8] = {raw[0].x, raw[0].y, raw[0].z, raw[0].w, raw[GPS - 1].x, raw[GPS - 1].y, raw[GPS - 1].z, raw[GPS - 1].w};
      groups.note(f);
      float4 pl[3] = {raw[0], raw[GPS - 1], raw[0]};
      if constexpr (decltype(form)::value == 2) split3(f, pl);
#pragma unroll
      for (int q = 0; q < (decltype(form)::value == 2 ? 3 : 2); ++q) *reinterpret_cast<float4*>(dst + q * STAGE) = pl[q];
    }
  };
  auto kept = [](const float4& v, bool k) __attribute__((always_inline)) { return make_float4(k ? v.x : 0.f, k ? v.y : 0.f, k ? v.z : 0.f, k ? v.w : 0.f); };
  auto store_slots = [&](const float4 (&regs)[NLD][GPS], int buf, unsigned ok) __attribute__((always_inline)) {
    TL* dst = sbuf + buf * (PL * STAGE);
#pragma unroll
    for (int i = 0; i < NLD; ++i)
      if (tid + TH * i < NSLOT) {
        float4 r[GPS];
#pragma unroll
        for (int g = 0; g < GPS; ++g) r[g] = kept(regs[i][g], (ok >> i) & 1u);
        store_slot(dst + st_lds[i], r);
      }
  };
  // F2: the scale, from the first chunk's values (the sums of two, where they are added)
  auto scale_of = [&](float m) __attribute__((always_inline)) {
    m = f2_wave_max(m);
    if (lane == 0) s_f2[wave] = m;
    if (tid < 2) s_f2[F2 ? WAVES + tid : 0] = 0.f;
    __syncthreads();
    float w = s_f2[0];
#pragma unroll
    for (int i = 1; i < WAVES; ++i) w = __builtin_elementwise_maximum(w, s_f2[F2 ? i : 0]);
    groups.start(f2_scale(__int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(w)))));
  };
  auto slots_max = [&](const float4 (&regs)[NLD][GPS], unsigned ok) __attribute__((always_inline)) {
    float m = 0.f;
#pragma unroll
    for (int i = 0; i < NLD; ++i) {
      const float4 u = regs[i][0], v = regs[i][GPS - 1];
      const float f[8] = {u.x, u.y, u.z, u.w, v.x, v.y, v.z, v.w};
      const float g = f2_amax8(f);
      m = __builtin_elementwise_maximum(m, (ok >> i) & 1u ? g : 0.f);
    }
    return m;
  };
  // (c: the chunk in the registers; terms: 1 in terms, or a form of store_unfit; first: the first chunk, F2's scale from its sums)
  auto stage_store = [&](int buf, int c, auto terms, bool first = false) __attribute__((always_inline)) {
    constexpr bool TERMS = decltype(terms)::value == 1;
    TL* dst = sbuf + buf * (PL * STAGE);
    if constexpr (UP) {
      // x + x2 of the source block to LDS in fp32 (bit pattern zero = 0 in both element types) ...
      float lo_max = 0.f;
#pragma unroll
      for (int i = 0; i < NLO; ++i) {
        const int slot = tid + TH * i;
        const int lpix = slot / Q4, q4 = slot - lpix * Q4;
        float fa[EPS], fb[EPS];
        const bool k1 = (lo_ok1 >> i) & 1u, k2 = (lo_ok2 >> i) & 1u;
        const float4 a0 = kept(lo_a[i][0], k1), b0 = kept(lo_b[i][0], k2);
        if constexpr (X3) {
          const float4 a1 = kept(lo_a[i][1], k1), b1 = kept(lo_b[i][1], k2);
          const float ta[8] = {a0.x, a0.y, a0.z, a0.w, a1.x, a1.y, a1.z, a1.w};
          const float tb[8] = {b0.x, b0.y, b0.z, b0.w, b1.x, b1.y, b1.z, b1.w};
#pragma unroll
          for (int e = 0; e < 8; ++e) fa[e] = ta[e], fb[e] = tb[e];
        } else {
          slot_to_f32(a0, fa, T());
          slot_to_f32(b0, fb, T());
        }
        if (lpix < 64) {
#pragma unroll
          for (int e = 0; e < EPS; e += 4)
            *reinterpret_cast<float4*>(&s_lo[lpix * LOS + q4 * EPS + e]) =
                make_float4(fa[e] + fb[e], fa[e + 1] + fb[e + 1], fa[e + 2] + fb[e + 2], fa[e + 3] + fb[e + 3]);
          if constexpr (F2 && TERMS) {
            if (first) {
              float f[8];
#pragma unroll
              for (int e = 0; e < 8; ++e) f[e] = fa[e] + fb[e];
              lo_max = __builtin_elementwise_maximum(lo_max, f2_amax8(f));
            }
          }
        }
      }
      if constexpr (F2 && TERMS) {
        if (first) scale_of(lo_max);      // (with the barrier)
        else __syncthreads();
      } else {
        __syncthreads();
      }
      // ... and the staged tile blended from it; pixels outside the up-sampled image are the conv's zero padding.
      // The taps' LDS offsets and weights depend on the tile only, and the compiler computes them once
      // and keeps 40 registers alive through the contraction.  fp32 kernels have the registers to spare
      // (two workgroups per CU either way) and run 1.5 % faster for it; in the bf16 kernels they cost
      // one or two resident workgroups, so there an opaque zero makes them a per-chunk computation.  The three-term
      // kernels: the 32-column one would pass 256 registers and lose its second workgroup; the wider ones have the
      // room (252) and keep the values (decoder 0 of the 264x352 frame 73 -> 70 us).
      int opaque = 0;
      if (sizeof(T) == 2 || (X3 && WN == 1)) asm volatile("" : "+v"(opaque));
#pragma unroll
      for (int i = 0; i < NLD; ++i) {
        const int slot = tid + TH * i + opaque;
        if (slot >= NSLOT) continue;
        const int pix = slot / Q4, q4 = slot - pix * Q4;
        const int hy = iy0 + pix / IT, hx = ix0 + pix % IT;
        float o[EPS];
#pragma unroll
        for (int e = 0; e < EPS; ++e) o[e] = 0.f;
        if (hy >= 0 && hy < a.h_in && hx >= 0 && hx < a.w_in) {
          int r0, r1, q0, q1;
          float lr0, lr1, lq0, lq1;
          conv_up2x_coef(hy, h_lo, r0, r1, lr0, lr1);
          conv_up2x_coef(hx, w_lo, q0, q1, lq0, lq1);
          const float* v00 = s_lo + ((r0 - lo_y0) * 8 + (q0 - lo_x0)) * LOS + q4 * EPS;
          const float* v01 = s_lo + ((r0 - lo_y0) * 8 + (q1 - lo_x0)) * LOS + q4 * EPS;
          const float* v10 = s_lo + ((r1 - lo_y0) * 8 + (q0 - lo_x0)) * LOS + q4 * EPS;
          const float* v11 = s_lo + ((r1 - lo_y0) * 8 + (q1 - lo_x0)) * LOS + q4 * EPS;
#pragma unroll
          for (int e = 0; e < EPS; e += 4) {       // 16-byte LDS reads
            const float4 t00 = *reinterpret_cast<const float4*>(v00 + e), t01 = *reinterpret_cast<const float4*>(v01 + e);
            const float4 t10 = *reinterpret_cast<const float4*>(v10 + e), t11 = *reinterpret_cast<const float4*>(v11 + e);
            o[e] = conv_up2x_v(lr0, lr1, conv_up2x_h(lq0, lq1, t00.x, t01.x), conv_up2x_h(lq0, lq1, t10.x, t11.x));
            o[e + 1] = conv_up2x_v(lr0, lr1, conv_up2x_h(lq0, lq1, t00.y, t01.y), conv_up2x_h(lq0, lq1, t10.y, t11.y));
            o[e + 2] = conv_up2x_v(lr0, lr1, conv_up2x_h(lq0, lq1, t00.z, t01.z), conv_up2x_h(lq0, lq1, t10.z, t11.z));
            o[e + 3] = conv_up2x_v(lr0, lr1, conv_up2x_h(lq0, lq1, t00.w, t01.w), conv_up2x_h(lq0, lq1, t10.w, t11.w));
          }
        }
        const int lrow = pix / IT;
        TL* d = dst + lrow * RP + (pix - lrow * IT) * LS + EPS * q4;
        if constexpr (F2) {
          const float4 raw[GPS] = {make_float4(o[0], o[1], o[2], o[3]), make_float4(o[4], o[5], o[6], o[7])};
          if constexpr (TERMS) store_slot(d, raw);
          else store_unfit(d, raw, terms);
        } else if constexpr (X3) {
          float4 pl[3];
          split3(o, pl);
#pragma unroll
          for (int q = 0; q < 3; ++q) *reinterpret_cast<float4*>(d + q * STAGE) = pl[q];
        } else {
          *reinterpret_cast<float4*>(d) = f32_to_slot(o, T());
        }
      }
      return;
    }
    const unsigned ok = c >= nch1 ? ok2 : ok1;
    if constexpr (TERMS) {
      store_slots(st_reg, buf, ok);
    } else {
#pragma unroll
      for (int i = 0; i < NLD; ++i)
        if (tid + TH * i < NSLOT) {
          float4 r[GPS];
#pragma unroll
          for (int g = 0; g < GPS; ++g) r[g] = kept(st_reg[i][g], (ok >> i) & 1u);
          store_unfit(dst + st_lds[i], r, terms);
        }
    }
  };

  // ---- operand addressing ------------------------------------------------------------------------
  // This wave multiplies sub-chunks q = q0w .. q0w+NQW-1 of every chunk.  A unit is one tap of
  // one sub-chunk: 8 input channels, of which this lane's half handles 4 (channel pairing see
  // the header).  Everything that depends on the unit index is a compile-time constant times
  // cout (B) or a compile-time LDS offset (A); the lane-dependent parts are loop invariant.
  const int q0w = TPAR ? wk % NQ : wk * NQW;
  const int par = TPAR ? wk / NQ : 0;                          // tap class of this wave (scalar)
  // (tap, sub-chunk) of unit position `unit`; with the k-split over taps the tap depends on the wave and the last
  // position may hold no unit (tap >= K*K): it then multiplies nothing and prefetches the last tap once more
  auto unit_tap = [&](int unit) { return TPAR ? unit * TP + par : unit / NQW; };
  auto unit_sub = [&](int unit) { return TPAR ? 0 : unit % NQW; };
  const int cob0 = co0 + wn * (32 * NB);                       // first column of this wave
  const int b_lane = (half * cout + l32) * EPS;                // lane part of the packed filter index
  int a_lane[2], a_swap[2];                                    // lane part of the LDS index, what the other half adds to it
#pragma unroll
  for (int mb = 0; mb < 2; ++mb) {
    const int p = mb * 32 + l32;
    const int rowcol = ((p >> 3) * S) * RP + ((p & 7) * S) * LS + SUB * q0w;
    // stride 2: tile row r reads input row 2r + ky, whose halves are swapped iff (r + ky/2) is odd
    const int h0 = (S == 2) ? (half ^ ((p >> 3) & 1)) : half;
    a_lane[mb] = rowcol + EPS * h0;
    a_swap[mb] = EPS * (1 - 2 * h0);
  }
  // (where the tap depends on the wave, an index into the two would send them to LDS)
  auto swapped = [&](int mb, int ky) __attribute__((always_inline)) { return (S == 2 && ((ky >> 1) & 1) != 0) ? a_lane[mb] + a_swap[mb] : a_lane[mb]; };
  // filter row block of chunk c for this wave (c1 and c2 are multiples of CC: no partial chunks)
  auto chunk_b = [&](int c) __attribute__((always_inline)) -> const TL* {
    const bool second = c >= nch1;
    const int ci0 = (second ? c - nch1 : c) * CC;
    const int fb = second ? a.c1 : 0;
    return reinterpret_cast<const TL*>(a.filt_mc) +
           ((long long)((fb + ci0) / SUB + q0w) * (K * K) * (PL * 2) * cout + cob0) * EPS;
  };
  // Matrix-core filter copy: P[ci/8][tap][(ci%8)/4][co][ci%4] (fp32; 16 / 8 / 8 for bf16; X3: the bf16 layout with
  // the three term planes of a (block, tap) next to each other, P[ci/16][tap][term][(ci%16)/8][co][ci%8]).  The
  // k-steps of a unit are one 16-byte load per lane (and term), 512 contiguous bytes per half wave.
  float4 bring[RING][NB][PL];
  auto load_b = [&](const TL* ub, int unit, float4 (&bv)[NB][PL]) __attribute__((always_inline)) {
    if (TPAR && unit * TP >= K * K) return;          // padding position: no unit for any wave
    int tap = unit_tap(unit);                        // compile-time after unrolling, but for the k-split over taps
    const int qi = unit_sub(unit);
    if (TPAR && tap >= K * K) tap = K * K - 1;
#pragma unroll
    for (int nb = 0; nb < NB; ++nb)
#pragma unroll
      for (int q = 0; q < PL; ++q)
        bv[nb][q] = *reinterpret_cast<const float4*>(
            ub + ((long long)(((qi * (K * K) + tap) * PL + q) * 2) * cout + nb * 32) * EPS + b_lane);
  };

  // Three-term kernels with two buffers weave the staging of the next chunk into the MFMAs: a slot's split into terms (50
  // VALU instructions) and its LDS writes go between the MFMAs of a unit, one slot to a unit, then the loads of the chunk
  // after the next and its addresses between those of one more, all without a branch (a slot that does not exist is written
  // behind row 0), and the barrier sits between the last two units as in PIPE.  An MFMA takes 32 cycles, of which a wave's
  // own VALU instructions can use 28: measured, five of them between any two MFMAs cost nothing.  The slots of the next
  // chunk are loaded a whole chunk before they are stored, and in the prologue in front of the first B loads, because the
  // load counter is in order and takes the least of all paths: waiting for them must not mean waiting for the B loads
  // behind them.  (3x3 256->256: a chunk 1.55 -> 1.2 us in a launch of 16 workgroups, 18.3 -> 16.2 us together; at 33x44,
  // 240 workgroups, 20.0 -> 18.6; 512->512 at 8x12, unsplit, 30.7 -> 25.8.  On the full chip the matrix cores are held to
  // 1.6 .. 2.0 GHz by their power, and a launch that wastes less time runs at a lower clock.)
  const auto in_terms = std::integral_constant<int, 1>();
  constexpr bool WOVEN = X3 && NBUF == 2 && !UP && UPC >= NLD + 3;
  constexpr int TRASH = ROOM ? IT * LS : IT * RP;            // behind the pixels of row 0, or behind the rows: where slots that do not exist go
  static_assert(!WOVEN || TRASH + EPS <= STAGE, "room for a slot");
  int st_at[NLD];
#pragma unroll
  for (int i = 0; i < NLD; ++i) st_at[i] = tid + TH * i < NSLOT ? st_lds[i] : TRASH;
  unsigned ok_n = 0u;                                        // which slots of the chunk in st_reg count
  auto load_raw = [&](int c, bool first = false) __attribute__((always_inline)) {
    const bool second = c >= nch1;
    const T* xin = second ? a.x2 : a.x;
    const int cs = second ? a.c2 : a.c1;
    const int ci0 = (second ? c - nch1 : c) * CC;
    const T* dummy = a.filt_mc;
    ok_n = second ? ok2 : ok1;
#pragma unroll
    for (int i = 0; i < NLD; ++i) {
      const T* p = xin + (long long)st_po[i] * cs + ci0 + st_c4[i];
      p = (((first ? inb : ok_n) >> i) & 1u) ? p : dummy;
#pragma unroll
      for (int g = 0; g < GPS; ++g) st_reg[i][g] = *reinterpret_cast<const float4*>(p + 4 * g);
    }
  };
  auto store_one = [&](int i, TL* dst) __attribute__((always_inline)) {
    const bool k = (ok_n >> i) & 1u;
    const float4 u = st_reg[i][0], v = st_reg[i][GPS - 1];
    const float f[8] = {k ? u.x : 0.f, k ? u.y : 0.f, k ? u.z : 0.f, k ? u.w : 0.f, k ? v.x : 0.f, k ? v.y : 0.f, k ? v.z : 0.f, k ? v.w : 0.f};
    float4 pl[PL];
    if constexpr (F2) {
      groups.terms(f, pl);
    } else if constexpr (X3) {
      split3(f, pl);
    }
#pragma unroll
    for (int q = 0; q < PL; ++q) *reinterpret_cast<float4*>(dst + st_at[i] + q * STAGE) = pl[q];
  };
  float4 st_first[WOVEN ? NLD : 1][GPS];
  // All B loads below are unconditional: a conditional load would make the compiler's wait
  // counters conservative and collapse the prefetch distance.  After the last chunk the
  // "next chunk" pointer simply stays on the current one (a few redundant loads).
  // SPLIT: a part takes a contiguous range of the chunks (the host keeps the parts <= nch, so no range is empty)
  const int c_lo = SPLIT ? bz * nch >> a.xcd_fs : 0;
  const int c_hi = SPLIT ? (bz + 1) * nch >> a.xcd_fs : nch;
  const TL* ub_cur = chunk_b(c_lo);
  const TL* ub_next = ub_cur;
  // F2: the filter's scale and whether it fits, on their way from here on
  float filt_unscale = 1.f;
  if constexpr (F2) {
    const float* const end = f2_filter_end(a.filt_mc, (long long)a.cin_total * (K * K) * cout);
    filt_unscale = end[0];
    filt_form = end[1] - end[2];
  }
  int c_end = c_hi;                         // F2: where the contraction in two terms ends: in front of the first chunk that does not fit
  auto note_misfit = [&](int c) __attribute__((always_inline)) {      // in front of the barrier behind the stores of chunk c ...
    if constexpr (F2) {
      s_f2[groups.misfit() ? WAVES + ((c - c_lo) & 1) : WAVES + 2] = 1.f;      // (without a branch)
    }
  };
  // ... asked behind it whether some thread noted one, and looked at where chunk c would begin.  (As a part of the loop's own condition: a break of
  // its own costs twice as much, 0.3 us a launch)
  float stop = 0.f;
  auto ask_stop = [&](int c) __attribute__((always_inline)) {
    if constexpr (F2) stop = s_f2[WAVES + ((c - c_lo) & 1)];
  };
  auto stop_before = [&](int c) __attribute__((always_inline)) {
    if constexpr (F2) c_end = __builtin_amdgcn_readfirstlane(__float_as_int(stop)) != 0 && c < c_end ? c : c_end;
  };
  MIE_STAMP(2);
  const bool early = c_hi - c_lo >= 4;      // uniform over the workgroup
  if constexpr (WOVEN) {
    if (early) load_slots(st_first, c_lo, true);
  } else if (early) stage_load(c_lo, true);
  // F2, two inputs: the scale is for both, so it looks at the first chunk of the second one, too (a ConvLSTM's state deltas lie where the
  // events of earlier steps were: where the input is zero, nothing is known of them)
  const bool both = F2 && !UP && c_lo < nch1 && nch1 < c_hi;
  float4 st_two[F2 && !UP ? NLD : 1][GPS];
  if constexpr (F2 && !UP) {
    if (both) load_slots(st_two, nch1, true);
  }
  // the pixel-mask bytes, behind the first chunk's loads (pixel 0 stands in for slots outside the image, so that
  // these loads are unconditional too)
  {
    constexpr int NM = UP ? NLO : NLD;
    constexpr bool BOTH = NM <= 8;               // (with more slots the bytes of both cost registers: x2's follow, if there are any)
    const uint8_t* const x2m = a.x2 != nullptr ? a.x2m : nullptr;
    unsigned b1[NM], b2[NM];
    const auto& at = [&]() -> const int (&)[NM] { if constexpr (UP) return lo_po; else return st_po; }();
    const unsigned in = UP ? lo_inb : inb;
    unsigned k1, k2 = 0u;
    mie_mask_ask(a.xm, a.filt_mc, at, b1);
    if (BOTH) mie_mask_ask(x2m, a.filt_mc, at, b2);
    mie_mask_asked();
    k1 = mie_mask_take(a.xm, b1, in);
    if (BOTH) {
      k2 = mie_mask_take(x2m, b2, a.x2 != nullptr ? in : 0u);
    } else if (a.x2 != nullptr) {
      mie_mask_ask(x2m, a.filt_mc, at, b2);
      mie_mask_asked();
      k2 = mie_mask_take(x2m, b2, in);
    }
    if (UP) lo_ok1 = k1, lo_ok2 = k2;
    else ok1 = k1, ok2 = k2;
  }
  if constexpr (WOVEN) {
    if (!early) load_slots(st_first, c_lo, false);
    load_raw(c_lo + 1 < c_hi ? c_lo + 1 : c_lo, early);
  } else if (!early) stage_load(c_lo);
#pragma unroll
  for (int i = 0; i < (PD > 0 ? PD : 1); ++i) load_b(ub_cur, i, bring[i % RING]);
  // the output pixel mask of this thread's groups (or items of the gate chain, with their previous-cell masks): asked for
  // behind the first loads, taken behind their barrier
  constexpr int HG = CO_BLK / (GRU ? 8 : 16);                // groups of four hidden channels
  constexpr int PERG = (64 * HG + TH - 1) / TH;                // items per thread (the 32-column slab has 128: half the threads idle)
  constexpr int NLIVE = GATES ? PERG : PER;
  const uint8_t* const live_m = a.refresh ? nullptr : a.ts.pixmask;
  const uint8_t* const cp_m = GATES && !GRU && a.g_cpd != nullptr ? a.g_cpm : nullptr;
  unsigned live_in = 0u, live_b[NLIVE], cp_b[NLIVE];
  if (!SPLIT) {
    int at[NLIVE];
#pragma unroll
    for (int g = 0; g < NLIVE; ++g) {
      const int idx = tid + TH * g, p = GATES ? idx / HG : idx / QPP;
      const int oy = y0 + (p >> 3), ox = x0 + (p & 7);
      const bool k = p < 64 && oy < hout && ox < wout;
      at[g] = k ? (n * hout + oy) * wout + ox : 0;
      live_in |= (k ? 1u : 0u) << g;
    }
    mie_mask_ask(live_m, a.filt_mc, at, live_b);
    if (GATES && !GRU) mie_mask_ask(cp_m, a.filt_mc, at, cp_b);
    mie_mask_asked();
  }
  // (masked pixels that the first chunk's loads fetched are zeroed here)
  if constexpr (F2 && !UP) {
    float m;
    if constexpr (WOVEN) m = slots_max(st_first, c_lo >= nch1 ? ok2 : ok1);
    else m = slots_max(st_reg, c_lo >= nch1 ? ok2 : ok1);
    if (both) m = __builtin_elementwise_maximum(m, slots_max(st_two, ok2));
    scale_of(m);
  }
  if constexpr (WOVEN) store_slots(st_first, 0, c_lo >= nch1 ? ok2 : ok1);
  else stage_store(0, c_lo, in_terms, true);
  note_misfit(c_lo);
  __syncthreads();
  if (F2 && filt_form != 1.f) c_end = c_lo;
  ask_stop(c_lo);
  unsigned cp_bits = 0u;
  if (!SPLIT) live_bits = mie_mask_take(live_m, live_b, live_in);
  if (GATES && !GRU) cp_bits = mie_mask_take(cp_m, cp_b, a.g_cpd != nullptr ? live_bits : 0u);
  if (!GATES && !SPLIT && EARLY) epilogue_fetch(0);
  MIE_STAMP(3);

  // A operand of unit `unit` from the staged chunk at `sin` (one 16-byte LDS read per pixel block).
  auto load_a = [&](const TL* sin, int unit, float4 (&dst)[2][PL]) __attribute__((always_inline)) {
    if (TPAR && unit * TP >= K * K) return;
    int tap = unit_tap(unit);
    const int qi = unit_sub(unit);
    if (TPAR && tap >= K * K) tap = K * K - 1;
    const int ky = tap / K, kx = tap - ky * K;
#pragma unroll
    for (int mb = 0; mb < 2; ++mb)
#pragma unroll
      for (int q = 0; q < PL; ++q)
        dst[mb][q] = *reinterpret_cast<const float4*>(
            &sin[q * STAGE + swapped(mb, ky) + ky * RP + kx * LS + SUB * qi]);
  };
  // the MFMAs of one unit position
  auto mma = [&](int unit, const float4 (&av)[2][PL], const float4 (&bv)[NB][PL]) __attribute__((always_inline)) {
    if (TPAR && unit * TP >= K * K) return;
    if (TPAR && unit * TP + TP > K * K && unit_tap(unit) >= K * K) return;     // uniform over the wave
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
      if constexpr (F2) mma_unit2_f2(acc[0][nb], acc[1][nb], accs[0][nb], accs[1][nb], av[0], av[1], bv[nb]);
      else if constexpr (X3) mma_unit2_x3(acc[0][nb], acc[1][nb], accs[0][nb], accs[1][nb], av[0], av[1], bv[nb]);
      else mma_unit2(acc[0][nb], acc[1][nb], av[0][0], av[1][0], bv[nb][0], T());
    }
  };

  // Double-buffered kernels fold the chunk hand-over into the contraction, so that the matrix cores run
  // through it:
  //   * the next chunk's addresses are computed and its global loads issued right after the MFMAs of the
  //     first unit (an opaque copy of the chunk index keeps the compiler from hoisting the ~70 address
  //     instructions in front of them, where they ran with the matrix cores idle);
  //   * its LDS stores go out under the unit before the last but one;
  //   * the barrier sits between the last two units: by then every wave holds the A operands of its last
  //     unit in registers, so the barrier, and the LDS read of the next chunk's first operands (a register
  //     set of their own) behind it, pass under the last unit's MFMAs.
  // Measured on MI355X this ordering is worth under 1 % against "loads at the top of the chunk, stores and
  // barrier at its end": what a chunk loses against its MFMA time is not the hand-over (see the header).
  constexpr bool PIPE = MIE_PIPE && NBUF == 2 && !UP && UPC >= 8;
  if constexpr (WOVEN) {
    float4 av[2][2][PL], av0[2][PL];
    const TL* sin = sbuf;
    TL* snext = sbuf + PL * STAGE;
    load_a(sin, 0, av0);
    stop_before(c_lo);
    for (int c = c_lo; c < c_end; ++c) {
#pragma unroll
      for (int i = 0; i < UPC; ++i) {
        const int ip = i + PD;
        if (ip < UPC) load_b(ub_cur, ip, bring[ip % RING]);
        else load_b(ub_next, ip - UPC, bring[ip % RING]);
        if (i + 1 < UPC) load_a(sin, i + 1, av[(i + 1) & 1]);
        __builtin_amdgcn_sched_barrier(0);
        if (i == 0) mma(0, av0, bring[0]);
        else mma(i, av[i & 1], bring[i % RING]);
        if (i == 0) {
          int cn = __builtin_amdgcn_readfirstlane(c + 1 < c_hi ? c + 1 : c);
          asm volatile("" : "+s"(cn));
          ub_next = chunk_b(cn);
        }
        if (i < NLD) {
          store_one(i, snext);
        } else if (i == NLD) {
          note_misfit(c + 1);      // (well ahead of the barrier, which waits for what was written)
          int cn = __builtin_amdgcn_readfirstlane(c + 2 < c_hi ? c + 2 : c_hi - 1);
          asm volatile("" : "+s"(cn));
          load_raw(cn);
        }
        if (i <= NLD) {
#pragma unroll
          for (int j = 0; j < (F2 ? 6 : 12) * NB; ++j) {
            __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x2, F2 ? 8 : 5, 0);
            __builtin_amdgcn_sched_group_barrier(0x4, 3, 0);
          }
        }
        __builtin_amdgcn_sched_barrier(0);
        if (i == UPC - 2) {
          __syncthreads();
          load_a(snext, 0, av0);
          ask_stop(c + 1);
          __builtin_amdgcn_sched_barrier(0);
        }
      }
      ub_cur = ub_next;
      TL* const t = const_cast<TL*>(sin);
      sin = snext;
      snext = t;
      stop_before(c + 1);
      MIE_STAMP(4 + (c - c_lo));
    }
  } else if constexpr (PIPE) {
    float4 av[2][2][PL], av0[2][PL];
    load_a(sbuf, 0, av0);
    stop_before(c_lo);
    for (int c = c_lo; c < c_end; ++c) {
      const bool more = c + 1 < c_hi;
      const TL* sin = sbuf + ((c - c_lo) & 1) * (PL * STAGE);
      const TL* sin_next = sbuf + ((c - c_lo + 1) & 1) * (PL * STAGE);
#pragma unroll
      for (int i = 0; i < UPC; ++i) {
        if (PD > 0) {
          const int ip = i + PD;
          if (ip < UPC) load_b(ub_cur, ip, bring[ip % RING]);
          else load_b(ub_next, ip - UPC, bring[ip % RING]);
        }
        if (i + 1 < UPC) load_a(sin, i + 1, av[(i + 1) & 1]);
        __builtin_amdgcn_sched_barrier(0);
        if (i == 0) mma(0, av0, bring[0]);
        else mma(i, av[i & 1], bring[i % RING]);
        __builtin_amdgcn_sched_barrier(0);
        if (i == 0) {
          int cn = __builtin_amdgcn_readfirstlane(more ? c + 1 : c);      // after the last chunk: redundant re-load, never stored
          asm volatile("" : "+s"(cn));
          ub_next = chunk_b(cn);
          stage_load(cn);
          __builtin_amdgcn_sched_barrier(0);
        }
        if (i == UPC - 3) {
          if (more) stage_store((c - c_lo + 1) & 1, c + 1, in_terms);    // the other buffer: nobody reads it during this chunk
          __builtin_amdgcn_sched_barrier(0);
        }
        if (i == UPC - 2) {
          // every wave has its last operands of this chunk (the wait for them is part of the barrier)
          note_misfit(c + 1);
          __syncthreads();
          ask_stop(c + 1);
          load_a(sin_next, 0, av0);       // after the last chunk: read and dropped
          __builtin_amdgcn_sched_barrier(0);
        }
      }
      ub_cur = ub_next;
      stop_before(c + 1);
      MIE_STAMP(4 + (c - c_lo));
    }
    // (the epilogue reuses the staging buffers: every read of them that matters was waited for in front of the
    // last barrier; the operand read behind it returns whatever a faster wave has parked there, and is dropped)
  } else {
    stop_before(c_lo);
    for (int c = c_lo; c < c_end; ++c) {
      const bool more = c + 1 < c_hi;
      const int cn = more ? c + 1 : c;      // after the last chunk: redundant re-load, never stored
      ub_next = chunk_b(cn);
      stage_load(cn);
      const TL* sin = sbuf + ((c - c_lo) % NBUF) * (PL * STAGE);
      // A operands are read one unit ahead as well (two register sets); the scheduling barriers
      // pin "issue the loads for later units, then multiply this unit" so that the compiler can
      // neither sink the prefetches next to their uses nor hoist them all to the top.
      float4 av[2][2][PL];
      load_a(sin, 0, av[0]);
#pragma unroll
      for (int i = 0; i < UPC; ++i) {
        // B operands of the unit PD ahead (the first units of the next chunk at the end)
        if (PD > 0) {
          const int ip = i + PD;
          if (ip < UPC) load_b(ub_cur, ip, bring[ip % RING]);
          else load_b(ub_next, ip - UPC, bring[ip % RING]);
        }
        if (i + 1 < UPC) load_a(sin, i + 1, av[(i + 1) & 1]);
        __builtin_amdgcn_sched_barrier(0);
        mma(i, av[i & 1], bring[i % RING]);
        __builtin_amdgcn_sched_barrier(0);
        if (PD == 0) load_b(ub_next, 0, bring[0]);   // ring of one: reload right after use
      }
      if (NBUF == 1 && !UP) __syncthreads();   // every wave is done reading the only buffer (UP: stage_store syncs)
      if (more) stage_store((c - c_lo + 1) % NBUF, c + 1, in_terms);
      note_misfit(c + 1);
      __syncthreads();
      ask_stop(c + 1);
      stop_before(c + 1);
      ub_cur = ub_next;
      MIE_STAMP(4 + (c - c_lo));
    }
  }

  // ---- epilogue -----------------------------------------------------------------------------------
  // acc[mb][nb][r] of this lane is output pixel p = 32*mb + 8*(r/4) + 4*half + r%4,
  // channel column wn*32*NB + 32*nb + lane%32 of the workgroup's slab.
  if constexpr (F2) {
    const float c0 = f2_unscale(groups.scale) * filt_unscale, c1 = c0 * (1.f / F2_STEP);      // exactly: powers of two, 2^-143 at the least but for sums of zeros
#pragma unroll
    for (int mb = 0; mb < 2; ++mb)
#pragma unroll
      for (int nb = 0; nb < NB; ++nb)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[mb][nb][r] = fmaf(accs[mb][nb][r], c1, acc[mb][nb][r] * c0);
  } else if constexpr (X3) {
#pragma unroll
    for (int mb = 0; mb < 2; ++mb)
#pragma unroll
      for (int nb = 0; nb < NB; ++nb)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[mb][nb][r] += accs[mb][nb][r];
  }
  // F2, from the first chunk on that does not fit: three bf16 terms of the input and of the fp32 copy of the filter, as little code as
  // keeps the matrix cores busy (bound by the filter's 8 bytes a weight); where there are values that these do not hold, all of it on the
  // fp32 instruction.
  if constexpr (F2) {
    if (__builtin_expect(c_end < c_hi, 0)) {
      const long long fp32_at = 2LL * a.cin_total * (K * K) * cout;      // (in elements of two bytes: behind the terms)
      constexpr int R = 4;                                               // units of the filter in registers
      auto plainly = [&](int c_from, auto form) __attribute__((always_inline)) {
        constexpr bool THREE = decltype(form)::value == 2;
        constexpr int PA = THREE ? 3 : 2;
        for (int c = c_from; c < c_hi; ++c) {
          const TL* const ub = chunk_b(c) + fp32_at;
          float4 br[R][NB][PL];
          auto load = [&](int unit, float4 (&bv)[NB][PL]) __attribute__((always_inline)) {
            const int u = unit < UPC ? unit : UPC - 1, tap = unit_tap(u) < K * K ? unit_tap(u) : K * K - 1;
#pragma unroll
            for (int nb = 0; nb < NB; ++nb)
#pragma unroll
              for (int q = 0; q < PL; ++q)
                bv[nb][q] = *reinterpret_cast<const float4*>(ub + ((long long)(((unit_sub(u) * (K * K) + tap) * PL + q) * 2) * cout + nb * 32) * EPS + b_lane);
          };
          stage_load(c);
#pragma unroll
          for (int j = 0; j < R - 1; ++j) load(j, br[j]);
          __syncthreads();
          stage_store(0, c, form);
          __syncthreads();
          float4 av[2][2][PA];
          auto read = [&](int unit, float4 (&x)[2][PA]) __attribute__((always_inline)) {
            const int u = unit < UPC ? unit : UPC - 1, tap = unit_tap(u) < K * K ? unit_tap(u) : K * K - 1, ky = tap / K, kx = tap - ky * K;
#pragma unroll
            for (int mb = 0; mb < 2; ++mb)
#pragma unroll
              for (int q = 0; q < PA; ++q)
                x[mb][q] = *reinterpret_cast<const float4*>(&sbuf[q * STAGE + swapped(mb, ky) + ky * RP + kx * LS + SUB * unit_sub(u)]);
          };
          read(0, av[0]);
#pragma unroll 1
          for (int u0 = 0; u0 < UPC; u0 += R) {
#pragma unroll
            for (int j = 0; j < R; ++j) {
              const int u = u0 + j;
              load(u + R - 1, br[(j + R - 1) % R]);
              read(u + 1, av[(j + 1) & 1]);
              __builtin_amdgcn_sched_barrier(0);
              if (u >= UPC || unit_tap(u) >= K * K) continue;
              const auto& x = av[j & 1];
#pragma unroll
              for (int nb = 0; nb < NB; ++nb) {
                if constexpr (THREE) {
                  float4 b3[3];
                  split3_raw(br[j][nb], b3);
                  mma_unit2_x3(acc[0][nb], acc[1][nb], accs[0][nb], accs[1][nb], x[0], x[1], b3);
                } else {
#pragma unroll
                  for (int q = 0; q < PL; ++q) mma_unit2(acc[0][nb], acc[1][nb], x[0][q], x[1][q], br[j][nb][q], float());
                }
              }
            }
          }
        }
      };
      auto clear = [&](auto& v) __attribute__((always_inline)) {
#pragma unroll
        for (int mb = 0; mb < 2; ++mb)
#pragma unroll
          for (int nb = 0; nb < NB; ++nb)
#pragma unroll
            for (int r = 0; r < 16; ++r) v[mb][nb][r] = 0.f;
      };
      clear(accs);
      if (filt_form >= 0.f) plainly(c_end, std::integral_constant<int, 2>());
#pragma unroll
      for (int mb = 0; mb < 2; ++mb)
#pragma unroll
        for (int nb = 0; nb < NB; ++nb)
#pragma unroll
          for (int r = 0; r < 16; ++r) acc[mb][nb][r] += accs[mb][nb][r];
      __syncthreads();
      if (tid == 0) s_f2[WAVES] = filt_form < 0.f ? 1.f : 0.f;
      __syncthreads();
      if (groups.huge()) s_f2[WAVES] = 1.f;
      __syncthreads();
      if (__builtin_amdgcn_readfirstlane(__float_as_int(s_f2[WAVES])) != 0) {
        clear(acc);
        plainly(c_lo, std::integral_constant<int, 0>());
        __syncthreads();
      }
    }
  }
  // the wave's sums to LDS, where all of them meet behind a barrier
  auto meet = [&]() __attribute__((always_inline)) {
    float* red = smem + wk * (64 * CO_BLK);
#pragma unroll
    for (int mb = 0; mb < 2; ++mb)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int p = mb * 32 + 8 * (r >> 2) + 4 * half + (r & 3);
#pragma unroll
        for (int nb = 0; nb < NB; ++nb)
          red[p * CO_BLK + wn * (32 * NB) + nb * 32 + l32] = acc[mb][nb][r];
      }
    __syncthreads();
  };
  if constexpr (GRU) {
    // Gate math of a ConvGRU: column 8 * j + e is the update gate of hidden channel 4 * j + e (e < 4) or the candidate of 4 * j + e - 4.
    // An item is a pixel x four adjacent hidden channels: two 16-byte groups in LDS, 16 bytes of either reservoir, 16 (bf16: 8) of
    // the state delta.  Against a conv that stores the gates' deltas and a launch that reads them again, passes of optical flow at
    // 256x256, fp32 (four such layers; what goes is a launch and its trips to memory): 343.9 -> 326.4 and 434.8 -> 419.1 us.
    float4 ru[PERG], rc[PERG];
    long long ho[PERG];
#pragma unroll
    for (int i = 0; i < PERG; ++i) {
      const int idx = tid + TH * i, p = idx / HG, g4 = idx - p * HG;
      ho[i] = (((long long)n * hout + y0 + (p >> 3)) * wout + x0 + (p & 7)) * a.hid + co0 / 2 + 4 * g4;
      const long long at = ((live_bits >> i) & 1u) ? ho[i] : 0;
      ru[i] = *reinterpret_cast<const float4*>(a.res + at);
      rc[i] = *reinterpret_cast<const float4*>(a.g_cres + at);
    }
    meet();
#pragma unroll
    for (int i = 0; i < PERG; ++i) {
      if (!((live_in >> i) & 1u)) continue;
      if (!((live_bits >> i) & 1u)) {
        mie_st4(a.g_dh, ho[i], make_float4(0.f, 0.f, 0.f, 0.f));
        continue;
      }
      const int idx = tid + TH * i, p = idx / HG, g4 = idx - p * HG;
      float4 dg[2];
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        dg[j] = *reinterpret_cast<const float4*>(&smem[p * CO_BLK + 8 * g4 + 4 * j]);
#pragma unroll
        for (int k2 = 1; k2 < WK; ++k2) {
          const float4 part = *reinterpret_cast<const float4*>(&smem[k2 * (64 * CO_BLK) + p * CO_BLK + 8 * g4 + 4 * j]);
          dg[j].x += part.x; dg[j].y += part.y; dg[j].z += part.z; dg[j].w += part.w;
        }
      }
      const float4 h = mie_gru_gates4(ru[i], rc[i], dg[0], dg[1]);
      *reinterpret_cast<float4*>(a.res + ho[i]) = ru[i];
      *reinterpret_cast<float4*>(a.g_cres + ho[i]) = rc[i];
      mie_st4(a.g_dh, ho[i], h);
    }
  } else if constexpr (GATES) {
    // ConvLSTM gate chain as the epilogue.  The filter columns are interleaved by gate: column 4*hc + g is
    // gate g (in, remember, out, cell) of hidden channel hc, so a workgroup owns all four gates of its
    // CO_BLK/4 hidden channels.  Every wave parks its accumulators in LDS; a thread then sums the k-split
    // partials of the four gate columns of one (pixel, hidden channel) and runs the chain on the reservoirs.
    // An item is one pixel x four adjacent hidden channels: their 16 gate columns are four 16-byte groups in LDS
    // and 64 contiguous bytes of the gate reservoir, their cell / previous-cell reservoirs one 16-byte group each,
    // their state deltas 16 (fp32) or 8 (bf16) bytes.  The masks came with the first operands and the reservoirs are asked
    // for ahead of the exchange (both used to be asked for behind it, one after the other: bf16 8x480x640 pass, 20 % active,
    // 2558 -> 2495 us, 2x200x280 299 -> 297, fp32 1x64x96 185.5 -> 184.3).
    GateItem item[PERG];
    long long ho[PERG], go[PERG];
#pragma unroll
    for (int i = 0; i < PERG; ++i) {
      const int idx = tid + TH * i, p = idx / HG, g4 = idx - p * HG;
      const long long pix = ((long long)n * hout + y0 + (p >> 3)) * wout + x0 + (p & 7);
      ho[i] = pix * a.hid + co0 / 4 + 4 * g4;
      go[i] = pix * a.cout + co0 + 16 * g4;
      conv_gates_load<T>(a, (live_bits >> i) & 1u, (cp_bits >> i) & 1u, ho[i], go[i], item[i]);
    }
    meet();
#pragma unroll
    for (int i = 0; i < PERG; ++i) {
      if (!((live_in >> i) & 1u)) continue;
      const int idx = tid + TH * i, p = idx / HG, g4 = idx - p * HG;
      float4 dg[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        dg[j] = *reinterpret_cast<const float4*>(&smem[p * CO_BLK + 16 * g4 + 4 * j]);
#pragma unroll
        for (int k2 = 1; k2 < WK; ++k2) {
          const float4 part = *reinterpret_cast<const float4*>(&smem[k2 * (64 * CO_BLK) + p * CO_BLK + 16 * g4 + 4 * j]);
          dg[j].x += part.x; dg[j].y += part.y; dg[j].z += part.z; dg[j].w += part.w;
        }
      }
      conv_gates_item<T>(a, (live_bits >> i) & 1u, (cp_bits >> i) & 1u, ho[i], go[i], dg, item[i]);
    }
  } else {
    // the last barrier of the main loop has retired every read of the staging buffers that is used
    if (!EARLY && !SPLIT) epilogue_fetch(0);      // (ahead of the exchange: bf16 2x200x280 pass 298.8 -> 294.7 us with k_upconv2x's)
    meet();
    unsigned bad_bits = 0u;                      // groups whose sums are not finite (conv_quad_again)
#pragma unroll
    for (int h0 = 0; h0 < PER; h0 += PB) {       // the 128-column slabs in two passes of four groups per thread
      if (SPLIT || h0 > 0) epilogue_fetch(h0);
      float4 v[PB];
#pragma unroll
      for (int i = 0; i < PB; ++i) {
        const int idx = tid + TH * (h0 + i);      // group idx: pixel idx / QPP, channels 4 * (idx % QPP) ...
        float4 sum = *reinterpret_cast<const float4*>(&smem[4 * idx]);
#pragma unroll
        for (int k2 = 1; k2 < WK; ++k2) {
          const float4 part = *reinterpret_cast<const float4*>(&smem[k2 * (64 * CO_BLK) + 4 * idx]);
          sum.x += part.x; sum.y += part.y; sum.z += part.z; sum.w += part.w;
        }
        v[i] = sum;
      }
      if constexpr (SPLIT) {
        float* plane = a.ws + (long long)bz * a.ws_plane;
#pragma unroll
        for (int i = 0; i < PB; ++i)
          if (e_ok[i]) *reinterpret_cast<float4*>(plane + e_off[i]) = v[i];
      } else {
        if constexpr (AGAIN) {
#pragma unroll
          for (int i = 0; i < PB; ++i)
            if (e_ok[i] && !finite4(v[i])) {
              e_ok[i] = false;
              bad_bits |= 1u << (h0 + i);
            }
        }
        conv_epilogue_store4<T, PB>(a, e_off, e_co, e_ok, v, e_r0, e_add, e_live);
      }
    }
    if constexpr (AGAIN) {
      if (__builtin_expect(__ballot(bad_bits != 0u) != 0ull, 0))
        for (int g = 0; g < PER; ++g) {
          const int idx = tid + TH * g, p = idx / QPP, co = co0 + 4 * (idx - p * QPP);
          if ((bad_bits >> g) & 1u) conv_quad_again<T, K, S>(conv_args_again<T>(), n, y0 + (p >> 3), x0 + (p & 7), co);
        }
    }
  }
  MIE_STAMP(14);
}

// The partial sums of four channels (offset off), added in the order of the parts.  All of them are loaded before the first
// is added, for the counts a split makes (split_parts: 2, 4, 8): in a loop over the parts each load waited for the one
// before it, and these launches consist of little but that wait (8 parts, 256 channels at 8x12: 5.3 -> 4.1 us; a gates conv
// of 4 parts there 7.1 -> 5.6).
template <int PARTS>
__device__ __forceinline__ float4 split_sum_of(const float* ws, long long plane) {
  float4 v[PARTS];
#pragma unroll
  for (int q = 0; q < PARTS; ++q) v[q] = *reinterpret_cast<const float4*>(ws + q * plane);
#pragma unroll
  for (int q = 1; q < PARTS; ++q) {
    v[0].x += v[q].x; v[0].y += v[q].y; v[0].z += v[q].z; v[0].w += v[q].w;
  }
  return v[0];
}
__device__ __forceinline__ float4 split_sum(const float* ws, long long plane, int parts) {
  if (parts == 2) return split_sum_of<2>(ws, plane);
  if (parts == 4) return split_sum_of<4>(ws, plane);
  if (parts == 8) return split_sum_of<8>(ws, plane);
  float4 sum = *reinterpret_cast<const float4*>(ws);
  for (int q = 1; q < parts; ++q) {
    const float4 part = *reinterpret_cast<const float4*>(ws + q * plane);
    sum.x += part.x; sum.y += part.y; sum.z += part.z; sum.w += part.w;
  }
  return sum;
}

// The same for four such groups in a row, all loads before the first sum.
template <int PARTS>
__device__ __forceinline__ void split_sum4_of(const float* ws, long long plane, float4 (&sum)[4]) {
  float4 v[PARTS][4];
#pragma unroll
  for (int q = 0; q < PARTS; ++q)
#pragma unroll
    for (int j = 0; j < 4; ++j) v[q][j] = *reinterpret_cast<const float4*>(ws + q * plane + 4 * j);
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    sum[j] = v[0][j];
#pragma unroll
    for (int q = 1; q < PARTS; ++q) {
      sum[j].x += v[q][j].x; sum[j].y += v[q][j].y; sum[j].z += v[q][j].z; sum[j].w += v[q][j].w;
    }
  }
}
__device__ __forceinline__ void split_sum4(const float* ws, long long plane, int parts, float4 (&sum)[4]) {
  if (parts == 4) return split_sum4_of<4>(ws, plane, sum);
#pragma unroll
  for (int j = 0; j < 4; ++j) sum[j] = split_sum(ws + 4 * j, plane, parts);
}

// Second half of a SPLIT launch: per active tile the `parts` partial planes are added in order and
// the ordinary epilogue (addend, reservoir, activation) runs; stale tiles are zeroed.  One thread per
// (pixel, channel), channels fastest.
// K, S != 0: sums that are not finite are computed again in fp32 (conv_quad_again).
template <typename T, int K = 0, int S = 0>
__global__ __launch_bounds__(256) void k_conv_split_finish(ConvArgsT<T> a, int parts) {
  int n, y0, x0;
  const int tk = mie_pick_tile(a.ts, blockIdx.x + conv_args_entry_zero(a), n, y0, x0);
  if (tk == 0) return;
  const int hout = a.ts.h, wout = a.ts.w, cout = a.cout;
  const int cb = (((cout + (int)gridDim.y - 1) / (int)gridDim.y) + 3) & ~3;      // channels of this block (whole groups of four)
  const int c0 = (int)blockIdx.y * cb;
  const int cn = (cout - c0 < cb) ? cout - c0 : cb;
  const int qn = cn >> 2;                                             // groups of four adjacent channels
  const uint8_t* const live_m = a.refresh ? nullptr : a.ts.pixmask;
  bool bad = false;
  for (int idx = threadIdx.x; idx < 64 * qn; idx += 256) {
    const int p = idx / qn, co = c0 + 4 * (idx - p * qn);
    const int oy = y0 + (p >> 3), ox = x0 + (p & 7);
    if (oy >= hout || ox >= wout) continue;
    const long long off = (((long long)n * hout + oy) * wout + ox) * cout + co;
    if (tk == 2) {
      mie_st4(a.out, off, make_float4(0.f, 0.f, 0.f, 0.f));
      continue;
    }
    const long long offs[1] = {off};
    const int cos[1] = {co}, at[1] = {(n * hout + oy) * wout + ox};
    const bool oks[1] = {true};
    float4 r0[1], add[1];
    unsigned live_b[1];
    mie_mask_ask(live_m, a.ws, at, live_b);
    conv_epilogue_load4<T, 1>(a, offs, oks, r0, add);
    const float4 accs[1] = {split_sum(a.ws + off, a.ws_plane, parts)};
    if constexpr (K != 0) {
      if (!finite4(accs[0])) {
        bad = true;
        continue;
      }
    }
    const bool live[1] = {mie_mask_take(live_m, live_b, 1u) != 0u};
    conv_epilogue_store4<T, 1>(a, offs, cos, oks, accs, r0, add, live);
  }
  if constexpr (K != 0) {
    if (__builtin_expect(__ballot(bad) != 0ull, 0))
      for (int idx = threadIdx.x; idx < 64 * qn; idx += 256) {
        const int p = idx / qn, co = c0 + 4 * (idx - p * qn);
        const int oy = y0 + (p >> 3), ox = x0 + (p & 7);
        if (oy < hout && ox < wout && !finite4(split_sum(a.ws + (((long long)n * hout + oy) * wout + ox) * cout + co, a.ws_plane, parts)))
          conv_quad_again<T, K, S>(conv_args_again<T>(), n, oy, ox, co);
      }
  }
}

// Second half of a split gates conv: per active tile the partial planes of the 4 * hid gate columns are added in
// order and the ConvLSTM gate chain runs on the sums; stale tiles get zero state deltas.  One thread per (pixel, four
// adjacent hidden channels), blockIdx.y over groups of hidden channels.
template <typename T>
__global__ __launch_bounds__(256) void k_gates_split_finish(ConvArgsT<T> a, int parts) {
  int n, y0, x0;
  const int tk = mie_pick_tile(a.ts, blockIdx.x + conv_args_entry_zero(a), n, y0, x0);
  if (tk == 0) return;
  const int hout = a.ts.h, wout = a.ts.w, hid = a.hid;
  const int hg_all = hid / 4;                                         // groups of four hidden channels
  const int hgb = (hg_all + (int)gridDim.y - 1) / (int)gridDim.y;      // groups of this block
  const int g_lo = (int)blockIdx.y * hgb;
  const int gn = (hg_all - g_lo < hgb) ? hg_all - g_lo : hgb;
  const float4 zero4 = make_float4(0.f, 0.f, 0.f, 0.f);
  for (int idx = threadIdx.x; idx < 64 * gn; idx += 256) {
    const int p = idx / gn, g4 = g_lo + (idx - p * gn);
    const int oy = y0 + (p >> 3), ox = x0 + (p & 7);
    if (oy >= hout || ox >= wout) continue;
    const long long pix = ((long long)n * hout + oy) * wout + ox;
    const long long ho = pix * hid + 4 * g4, go = pix * a.cout + 16 * g4;
    if (tk == 2) {
      mie_st4(a.g_dh, ho, zero4);
      mie_st4(a.g_dc, ho, zero4);
      continue;
    }
    // masks, reservoirs and partial sums go out together
    const int at[1] = {(int)pix};
    const uint8_t* const cp_m = a.g_cpd != nullptr ? a.g_cpm : nullptr;
    unsigned live_b[1], cp_b[1];
    mie_mask_ask(a.ts.pixmask, a.filt_mc, at, live_b);
    mie_mask_ask(cp_m, a.filt_mc, at, cp_b);
    GateItem item;
    conv_gates_load<T>(a, true, true, ho, go, item);
    float4 dg[4];
    split_sum4(a.ws + go, a.ws_plane, parts, dg);
    const bool on = mie_mask_take(a.ts.pixmask, live_b, 1u) != 0u, has_cp = a.g_cpd != nullptr && mie_mask_take(cp_m, cp_b, 1u) != 0u;
    if (!has_cp) item.dp = zero4;
    conv_gates_item<T>(a, on, has_cp && on, ho, go, dg, item);
  }
}

// A launch is split when it has at most 128 workgroups, at least 4 staged chunks and a workspace:
// into the largest power of two of parts (up to 8) that keeps the launch at 256 workgroups or fewer (one
// per CU: measured on MI355X, a second workgroup per CU costs more in per-workgroup set-up than it gains),
// leaves every part a chunk, and fits the workspace.  Returns false when the launch is not split.
// Number of parts (0: the launch is not split) for `groups` (tile, slab) pairs of `nch` staged chunks each; sets the
// plane size of the workspace.
template <typename T>
int split_parts(ConvArgsT<T>& a, long long groups, int nch) {
  static const int max_groups = [] { const char* e = getenv("MIE_CONV_SPLIT_GROUPS"); return e ? atoi(e) : 128; }();
  static const int max_wgs = [] { const char* e = getenv("MIE_CONV_SPLIT_WGS"); return e ? atoi(e) : 256; }();
  static const int most = [] {      // MIE_CONV_SPLIT caps the number of parts (1: never split): a tuning knob, read once
    const char* e = getenv("MIE_CONV_SPLIT");
    return e ? atoi(e) : 8;
  }();
  if (a.ws == nullptr || groups > max_groups || nch < 4) return 0;
  a.ws_plane = (long long)a.ts.n * a.ts.h * a.ts.w * a.cout;
  int parts = 1;
  while (2 * parts <= most && 2 * parts <= nch && groups * (2 * parts) <= max_wgs && (long long)(2 * parts) * a.ws_plane <= a.ws_floats)
    parts *= 2;
  a.xcd_fs = __builtin_ctz(parts);
  return parts < 2 ? 0 : parts;
}

// Blocks of a tile: 1024 on the chip, but none of fewer than 16 channels, so that each has an item for every thread.  (Down
// to four channels, three of a block's four waves were there for nothing: 1x64x96 pass 183.5 -> 181.6 us, eight finishes,
// optical flow 1x256x256 389.6 -> 380.1 with transposed convs, 496.0 -> 487.4 with up-sampling.)
template <typename T, int K = 0, int S = 0>
void launch_split_finish(const ConvArgsT<T>& a, unsigned cap, int parts, hipStream_t st) {
  unsigned ny = (unsigned)((1024 + cap - 1) / cap);
  if (ny > (unsigned)(a.cout / 16)) ny = (unsigned)(a.cout / 16);
  if (ny < 1) ny = 1;
  hipLaunchKernelGGL((k_conv_split_finish<T, K, S>), dim3(cap, ny), dim3(256), 0, st, a, parts);
}

// The arguments of an F2 kernel: the filter copy from its fp16 terms on.
template <typename T>
ConvArgsT<T> f2_args(const ConvArgsT<T>& a0, int k) {
  ConvArgsT<T> a = a0;
  a.filt_mc = (const T*)((const char*)a0.filt_mc + 6LL * a0.cin_total * k * k * a0.cout);
  return a;
}

template <typename T, int K, int S>
bool launch_split(const ConvArgsT<T>& a0, unsigned cap, hipStream_t st) {
  constexpr bool HAS_X3 = sizeof(T) == 4 && (K == 5 || (K == 3 && S == 1));
  const bool x3 = HAS_X3 && a0.x3 != 0;
  const int CC = x3 && S == 2 ? 16 : stage_channels(K, S, false) * (4 / (int)sizeof(T));
  if (a0.ws == nullptr || a0.refresh || a0.cout % 32 != 0 || a0.c1 % CC != 0 || a0.c2 % CC != 0) return false;
  ConvArgsT<T> a = a0;
  const int parts = split_parts(a, (long long)cap * (a0.cout / 32), (a0.c1 + a0.c2) / CC);
  if (parts == 0) return false;
  const dim3 grid(a.cout / 32 * parts, cap);
  const std::lock_guard<std::mutex> pair(mie_split_launches());
  if (x3) {
    if constexpr (HAS_X3) {
      if (a.x3 == 2) hipLaunchKernelGGL((k_conv_mfma<T, K, S, 1, 1, false, false, false, true, 2>), grid, dim3(256), 0, st, f2_args(a, K));
      else hipLaunchKernelGGL((k_conv_mfma<T, K, S, 1, 1, false, false, false, true, 1>), grid, dim3(256), 0, st, a);
    }
  } else {
    hipLaunchKernelGGL((k_conv_mfma<T, K, S, 1, 1, false, false, false, true>), grid, dim3(256), 0, st, a);
  }
  if constexpr (HAS_X3 && S == 2) {
    if (a.x3 == 1) {
      launch_split_finish<T, K, S>(a, cap, parts, st);
      return true;
    }
  }
  launch_split_finish(a, cap, parts, st);
  return true;
}

// The split form of the 5x5 conv over up2x(x + x2): the chunks of the (summed) input split as above, the plain finish.
template <typename T>
bool launch_up_split(const ConvArgsT<T>& a0, unsigned cap, hipStream_t st) {
  constexpr int CC = stage_channels(5, 1, false) * (4 / (int)sizeof(T));
  static const bool on = [] { const char* e = getenv("MIE_CONV_SPLIT_UP"); return e == nullptr || atoi(e) != 0; }();   // tuning knob
  if (!on || a0.ws == nullptr || a0.cout % 32 != 0 || a0.c1 % CC != 0) return false;
  ConvArgsT<T> a = a0;
  const int parts = split_parts(a, (long long)cap * (a0.cout / 32), a0.c1 / CC);
  if (parts == 0) return false;
  bool x3 = false;
  if constexpr (sizeof(T) == 4) x3 = a.x3 != 0;
  const std::lock_guard<std::mutex> pair(mie_split_launches());
  if (x3) {
    if constexpr (sizeof(T) == 4) {
      const dim3 grid(a.cout / 32 * parts, cap);
      if (a.x3 == 2) hipLaunchKernelGGL((k_conv_mfma<T, 5, 1, 1, 1, false, false, true, true, 2>), grid, dim3(256), 0, st, f2_args(a, 5));
      else hipLaunchKernelGGL((k_conv_mfma<T, 5, 1, 1, 1, false, false, true, true, 1>), grid, dim3(256), 0, st, a);
    }
  } else {
    hipLaunchKernelGGL((k_conv_mfma<T, 5, 1, 1, 1, false, false, true, true>), dim3(a.cout / 32 * parts, cap), dim3(256), 0, st, a);
  }
  launch_split_finish(a, cap, parts, st);
  return true;
}

// The split form of a ConvLSTM's gates conv: the contraction as a plain split 3x3 conv of the two inputs (the partial
// sums of all 4 * hid gate columns go to the workspace), then the gate chain in the finish kernel.
template <typename T>
bool launch_gates_split(const ConvArgsT<T>& a0, unsigned cap, hipStream_t st) {
  constexpr int CC = stage_channels(3, 1, false) * (4 / (int)sizeof(T));
  static const bool on = [] { const char* e = getenv("MIE_CONV_SPLIT_GATES"); return e == nullptr || atoi(e) != 0; }();   // tuning knob
  if (!on || a0.ws == nullptr || a0.cout != 4 * a0.hid || a0.hid % 8 != 0 || a0.c1 % CC != 0 || a0.c2 % CC != 0) return false;
  ConvArgsT<T> a = a0;
  const int parts = split_parts(a, (long long)cap * (a0.cout / 32), (a0.c1 + a0.c2) / CC);
  // (two parts do not pay for the second launch: E2Depth-incr 128x128 frame 0.2685 -> 0.2699 ms, measured; four do)
  if (parts < 4) return false;
  bool x3 = false;
  if constexpr (sizeof(T) == 4) x3 = a.x3 != 0;
  const std::lock_guard<std::mutex> pair(mie_split_launches());
  if (x3) {
    if constexpr (sizeof(T) == 4) {
      const dim3 grid(a.cout / 32 * parts, cap);
      if (a.x3 == 2) hipLaunchKernelGGL((k_conv_mfma<T, 3, 1, 1, 1, false, false, false, true, 2>), grid, dim3(256), 0, st, f2_args(a, 3));
      else hipLaunchKernelGGL((k_conv_mfma<T, 3, 1, 1, 1, false, false, false, true, 1>), grid, dim3(256), 0, st, a);
    }
  } else {
    hipLaunchKernelGGL((k_conv_mfma<T, 3, 1, 1, 1, false, false, false, true>), dim3(a.cout / 32 * parts, cap), dim3(256), 0, st, a);
  }
  unsigned ny = (unsigned)((1024 + cap - 1) / cap);
  if (ny > (unsigned)(a.hid / 16)) ny = (unsigned)(a.hid / 16);
  if (ny < 1) ny = 1;
  hipLaunchKernelGGL(k_gates_split_finish<T>, dim3(cap, ny), dim3(256), 0, st, a, parts);
  return true;
}

// Output channels per workgroup (the slab 32*NB*WN) for a launch of `cap` tiles: the widest of
// 128 / 64 / 32 that still gives the chip at least 400 workgroups when every tile is active
// (256 CUs, up to 3 workgroups resident on each), else the narrowest the staging depth of this
// (K, S) allows.  Measured on MI355X over the layer shapes of both network sizes: wider slabs
// re-read less of the input tile but leave CUs idle on the small planes; the 256-wide variant
// (two 32-column blocks per wave) lost to the 128-wide one on every shape and is only taken
// when forced.  The environment
// variable MIE_CONV_SLAB (32, 64, 128 or 256) overrides the choice where the shape allows it --
// a tuning knob for measurements, read once.
int forced_slab() {
  static const int v = [] {
    const char* e = getenv("MIE_CONV_SLAB");
    return e ? atoi(e) : 0;
  }();
  return v;
}

template <int K, int S, bool HALF>
int pick_slab(int cout, unsigned cap) {
  constexpr int NQ = stage_channels(K, S, HALF) / 8;
  const bool ok128 = cout % 128 == 0, ok64 = NQ >= 2 && cout % 64 == 0;
  const bool ok32 = NQ >= 4 && cout % 32 == 0;
  const int f = forced_slab();
  if ((f == 128 && ok128) || (f == 64 && ok64) || (f == 32 && ok32)) return f;
  const long long want = 400;
  if (ok128 && ((long long)cap * (cout / 128) >= want || (!ok64 && !ok32))) return 128;
  if (ok64 && ((long long)cap * (cout / 64) >= want || !ok32)) return 64;
  if (ok32) return 32;
  return 0;
}

// XCD-aware launch order (see the kernel): chooses the number of slab groups a.xcd_fs in {1, 2, 4, 8}
// (a divisor of the slab count) that minimises what the 8 L2s fetch in total -- the filter 8 / xcd_fs
// times plus the input xcd_fs times -- and returns the grid's x extent (xcd_grid_x).  The
// environment variable MIE_CONV_XCD forces the number of groups (0: plain launch order, a.xcd_fs = 0) --
// a tuning knob for measurements, read once.
template <typename T>
unsigned xcd_plan(ConvArgsT<T>& a, unsigned cap, int nslabs, int k, bool up = false) {
  static const int forced = [] {
    const char* e = getenv("MIE_CONV_XCD");
    return e ? atoi(e) : -1;
  }();
  a.xcd_fs = 0;
  if (forced == 0) return cap;
  const double cin = (double)a.c1 + a.c2;
  const double filt = cin * k * k * a.cout;
  const double in = (double)a.ts.n * a.h_in * a.w_in * (up ? 0.5 * a.c1 : cin);
  int best = 1;
  double cost = 8 * filt + in;
  for (int fs = 2; fs <= 8; fs *= 2) {
    if (nslabs % fs != 0) break;
    const double c = (8 / fs) * filt + fs * in;
    if (c < cost) cost = c, best = fs;
  }
  if (forced > 0 && 8 % forced == 0 && nslabs % forced == 0) best = forced;
  a.xcd_fs = best;
  a.xcd_m = mie_tile_magic((long long)cap * (nslabs / best), nslabs / best);
  return (unsigned)xcd_grid_x((int)cap);
}

// X3 kernels (fp32 deltas, a.x3 set, the filter copy in the three-term layout): 3x3 / 5x5, stride 1, input channels in
// whole chunks of 32, output slabs of 128 / 64 / 32 columns by the same rule as above.
// Stride 1 first looks for the widest slab that makes the launch one round of more than half a chip of workgroups
// (129 .. 256): measured on MI355X, one workgroup per CU with twice the columns beats one and a half rounds of the
// narrow ones (5x5 256->128 at 66x88: 198 workgroups of 64 columns 61-65 us, 396 of 32 columns 71-74 us; 3x3 gates conv
// 256+256->1024 at 33x44: 240 of 128 columns 53 us, 480 of 64 columns 57 us); at stride 2, whose workgroups are short,
// it does not (28 vs 29 us).  (All in three terms; in two the same rule.)
inline int pick_slab_x3(int cout, unsigned cap, int s) {
  const bool ok128 = cout % 128 == 0, ok64 = cout % 64 == 0, ok32 = cout % 32 == 0;
  const int f = forced_slab();
  if ((f == 128 && ok128) || (f == 64 && ok64) || (f == 32 && ok32)) return f;
  if (s == 1) {
    const int widths[3] = {128, 64, 32};
    const bool oks[3] = {ok128, ok64, ok32};
    for (int i = 0; i < 3; ++i) {
      const long long wgs = (long long)cap * (cout / widths[i]);
      if (oks[i] && wgs > 128 && wgs <= 256) return widths[i];
    }
  }
  const long long want = 400;
  if (ok128 && ((long long)cap * (cout / 128) >= want || (!ok64 && !ok32))) return 128;
  if (ok64 && ((long long)cap * (cout / 64) >= want || !ok32)) return 64;
  if (ok32) return 32;
  return 0;
}
inline bool x3_takes(int k, int s, int c1, int c2, int cout) {
  // (3x3 stride 2 was measured too: no faster than the fp32 instruction, 15-29 us either way, and it has a split form)
  if (s == 2) return k == 5 && c1 % 16 == 0 && c2 % 16 == 0 && cout % 32 == 0;
  return (k == 3 || k == 5) && s == 1 && c1 % 32 == 0 && c2 % 32 == 0 && cout % 32 == 0;
}

// Two terms: eight waves a workgroup, chunks of twice the channels (WIDE).  Where the workgroups are one round of the chip, one a CU, a CU has one
// wave a SIMD with four, and nothing runs while it waits.  us, four waves -> eight, every tile active, filters cold: 3x3 256->256 at 33x44
// (240 workgroups) 12.4 -> 12.05, 256->512 there 17.3 -> 16.7; 5x5 stride 2 (which is then double-buffered, too) 128->256 at 66x88 18.4 -> 15.4,
// 64->128 at 80x100 11.6 -> 10.5.  Not for fewer channels: 3x3 64->64 at 66x88 6.9 and 7.2; nor for slabs of 128
// columns, whose four waves are busy as they are (gates of 256+256 at 33x44 31 and 33 in a trace, frames the same).  A second round of such workgroups is no better than
// two of four waves a CU side by side (5x5 stride 2 64->128 at 132x176, 64 columns wide so that it is one: 15.7 and 14.7 alone, a frame the same);
// the ConvGRU's gates, likewise, the same.  Frame of 264x352 342 -> 335 us, planned ahead 328 -> 320, refresh 386 -> 378.
inline bool f2_wide(const ConvArgsT<float>& a, unsigned cap, int slab, int s) {
  const int chunk = s == 2 ? 32 : 64;
  return (slab == 32 || slab == 64) && (long long)cap * (a.cout / slab) <= 256 && a.c1 % chunk == 0 && a.c2 % chunk == 0 && a.c1 + a.c2 >= (s == 2 ? 64 : 256);
}

template <int AR, int K, bool GATES, bool UP, int S>
bool launch_terms(const ConvArgsT<float>& a0, unsigned cap, hipStream_t st) {
  ConvArgsT<float> a = a0;
  const int cout = a.cout;
  if (!x3_takes(K, S, a.c1, UP ? 0 : a.c2, cout)) return false;
  if constexpr (S == 2 && AR == 1) {
    // few tiles and a workspace, but too few chunks to split (32->64 at 64x96): the same outputs as from the split form
    if (a.ws != nullptr && !a.refresh && (long long)cap * (cout / 32) <= 128) {
      hipLaunchKernelGGL((k_conv_mfma<float, K, S, 1, 1, false, GATES, UP, false, AR, true>), dim3(xcd_plan(a, cap, cout / 32, K, UP), cout / 32), dim3(256), 0, st, a);
      return true;
    }
  }
  const int slab = pick_slab_x3(cout, cap, S);
  if constexpr (AR == 2 && !UP && (K == 3 || S == 2)) {
    if (f2_wide(a, cap, slab, S)) {
      const dim3 grid(xcd_plan(a, cap, cout / slab, K, UP), cout / slab);
      if (slab == 64) hipLaunchKernelGGL((k_conv_mfma<float, K, S, 2, 1, false, GATES, UP, false, AR, false, false, true>), grid, dim3(512), 0, st, a);
      else hipLaunchKernelGGL((k_conv_mfma<float, K, S, 1, 1, false, GATES, UP, false, AR, false, false, true>), grid, dim3(512), 0, st, a);
      return true;
    }
  }
  switch (slab) {
    case 128:
      hipLaunchKernelGGL((k_conv_mfma<float, K, S, 4, 1, false, GATES, UP, false, AR>), dim3(xcd_plan(a, cap, cout / 128, K, UP), cout / 128), dim3(256), 0, st, a);
      return true;
    case 64:
      hipLaunchKernelGGL((k_conv_mfma<float, K, S, 2, 1, false, GATES, UP, false, AR>), dim3(xcd_plan(a, cap, cout / 64, K, UP), cout / 64), dim3(256), 0, st, a);
      return true;
    case 32:
      hipLaunchKernelGGL((k_conv_mfma<float, K, S, 1, 1, false, GATES, UP, false, AR>), dim3(xcd_plan(a, cap, cout / 32, K, UP), cout / 32), dim3(256), 0, st, a);
      return true;
    default:
      return false;
  }
}
template <int K, bool GATES, bool UP, int S = 1>
bool launch_x3(const ConvArgsT<float>& a, unsigned cap, hipStream_t st) {
  return a.x3 == 2 ? launch_terms<2, K, GATES, UP, S>(f2_args(a, K), cap, st) : launch_terms<1, K, GATES, UP, S>(a, cap, st);
}

template <typename T, int K, int S, bool HALF>
bool launch_depth(const ConvArgsT<T>& a0, unsigned cap, hipStream_t st) {
  constexpr int NQ = stage_channels(K, S, HALF) / 8;
  ConvArgsT<T> a = a0;
  const int cout = a.cout;
  switch (pick_slab<K, S, HALF>(cout, cap)) {
    case 128:
      hipLaunchKernelGGL((k_conv_mfma<T, K, S, 4, 1, HALF>), dim3(xcd_plan(a, cap, cout / 128, K), cout / 128), dim3(256), 0, st, a);
      return true;
    case 64:
      if constexpr (NQ >= 2) {
        hipLaunchKernelGGL((k_conv_mfma<T, K, S, 2, 1, HALF>), dim3(xcd_plan(a, cap, cout / 64, K), cout / 64), dim3(256), 0, st, a);
        return true;
      }
      return false;
    case 32:
      if constexpr (NQ >= 4) {
        hipLaunchKernelGGL((k_conv_mfma<T, K, S, 1, 1, HALF>), dim3(xcd_plan(a, cap, cout / 32, K), cout / 32), dim3(256), 0, st, a);
        return true;
      }
      return false;
    default:
      return false;
  }
}

// The 5x5 stride-1 conv over up2x(x + x2): full staging depth only.
template <typename T>
bool launch_up(const ConvArgsT<T>& a0, unsigned cap, hipStream_t st) {
  if (launch_up_split<T>(a0, cap, st)) return true;
  if constexpr (sizeof(T) == 4) {
    if (a0.x3) return launch_x3<5, false, true>(a0, cap, st);
  }
  constexpr int FULL = stage_channels(5, 1) * (4 / (int)sizeof(T));
  if (a0.c1 % FULL != 0) return false;
  ConvArgsT<T> a = a0;
  const int cout = a.cout;
  switch (pick_slab<5, 1, false>(cout, cap)) {
    case 128:
      hipLaunchKernelGGL((k_conv_mfma<T, 5, 1, 4, 1, false, false, true>), dim3(xcd_plan(a, cap, cout / 128, 5, true), cout / 128), dim3(256), 0, st, a);
      return true;
    case 64:
      hipLaunchKernelGGL((k_conv_mfma<T, 5, 1, 2, 1, false, false, true>), dim3(xcd_plan(a, cap, cout / 64, 5, true), cout / 64), dim3(256), 0, st, a);
      return true;
    case 32:
      hipLaunchKernelGGL((k_conv_mfma<T, 5, 1, 1, 1, false, false, true>), dim3(xcd_plan(a, cap, cout / 32, 5, true), cout / 32), dim3(256), 0, st, a);
      return true;
    default:
      return false;
  }
}

// The gates conv of a ConvLSTM: 3x3, stride 1, full staging depth, gate chain in the epilogue.
template <typename T>
bool launch_gates(const ConvArgsT<T>& a0, unsigned cap, hipStream_t st) {
  if (launch_gates_split<T>(a0, cap, st)) return true;
  if constexpr (sizeof(T) == 4) {
    if (a0.x3) return a0.cout == 4 * a0.hid && a0.hid % 8 == 0 && launch_x3<3, true, false>(a0, cap, st);
  }
  constexpr int FULL = stage_channels(3, 1) * (4 / (int)sizeof(T));
  if (a0.c1 % FULL != 0 || a0.c2 % FULL != 0 || a0.cout != 4 * a0.hid || a0.hid % 8 != 0) return false;
  ConvArgsT<T> a = a0;
  const int cout = a.cout;
  switch (pick_slab<3, 1, false>(cout, cap)) {
    case 128:
      hipLaunchKernelGGL((k_conv_mfma<T, 3, 1, 4, 1, false, true>), dim3(xcd_plan(a, cap, cout / 128, 3), cout / 128), dim3(256), 0, st, a);
      return true;
    case 64:
      hipLaunchKernelGGL((k_conv_mfma<T, 3, 1, 2, 1, false, true>), dim3(xcd_plan(a, cap, cout / 64, 3), cout / 64), dim3(256), 0, st, a);
      return true;
    case 32:
      hipLaunchKernelGGL((k_conv_mfma<T, 3, 1, 1, 1, false, true>), dim3(xcd_plan(a, cap, cout / 32, 3), cout / 32), dim3(256), 0, st, a);
      return true;
    default:
      return false;
  }
}

// The stacked gates conv of a ConvGRU, gate math in the epilogue.
template <typename T, int AR>
bool launch_gru_as(const ConvArgsT<T>& a0, unsigned cap, hipStream_t st) {
  ConvArgsT<T> a = a0;
  const int cout = a.cout;
  switch (AR != 0 ? pick_slab_x3(cout, cap, 1) : pick_slab<3, 1, false>(cout, cap)) {
    case 128:
      hipLaunchKernelGGL((k_conv_mfma<T, 3, 1, 4, 1, false, true, false, false, AR, false, true>), dim3(xcd_plan(a, cap, cout / 128, 3), cout / 128), dim3(256), 0, st, a);
      return true;
    case 64:
      hipLaunchKernelGGL((k_conv_mfma<T, 3, 1, 2, 1, false, true, false, false, AR, false, true>), dim3(xcd_plan(a, cap, cout / 64, 3), cout / 64), dim3(256), 0, st, a);
      return true;
    case 32:
      hipLaunchKernelGGL((k_conv_mfma<T, 3, 1, 1, 1, false, true, false, false, AR, false, true>), dim3(xcd_plan(a, cap, cout / 32, 3), cout / 32), dim3(256), 0, st, a);
      return true;
    default:
      return false;
  }
}
template <typename T>
bool launch_gru(const ConvArgsT<T>& a, unsigned cap, hipStream_t st) {
  constexpr bool X3 = sizeof(T) == 4;
  constexpr int CC = X3 ? 32 : 64;
  if ((X3 && !a.x3) || a.c1 % CC != 0 || a.c2 % CC != 0 || a.cout != 2 * a.hid || a.cout % 32 != 0) return false;
  if constexpr (X3) return a.x3 == 2 ? launch_gru_as<T, 2>(f2_args(a, 3), cap, st) : launch_gru_as<T, 1>(a, cap, st);
  else return launch_gru_as<T, 0>(a, cap, st);
}

// Staging depth: the full one when both inputs' channel counts are multiples of it, else
// (stride 2 only) the half one.
template <typename T, int K, int S>
bool launch_ks(const ConvArgsT<T>& a, unsigned cap, hipStream_t st) {
  constexpr int MULT = 4 / (int)sizeof(T);
  constexpr int FULL = stage_channels(K, S) * MULT;
  if (a.c1 % FULL == 0 && a.c2 % FULL == 0 && pick_slab<K, S, false>(a.cout, cap) != 0)
    return launch_depth<T, K, S, false>(a, cap, st);
  if constexpr (S == 2) {
    constexpr int HALFC = stage_channels(K, S, true) * MULT;
    if (a.c1 % HALFC == 0 && a.c2 % HALFC == 0) return launch_depth<T, K, S, true>(a, cap, st);
  }
  return false;
}

}  // namespace

namespace {
template <typename T>
bool launch_any(const ConvArgsT<T>& a, int k, int s, unsigned cap, hipStream_t st) {
  if constexpr (sizeof(T) == 4) {
    if (a.x3) {
      if (k == 3 && s == 1) return launch_split<T, 3, 1>(a, cap, st) || launch_x3<3, false, false>(a, cap, st);
      if (k == 5 && s == 1) return launch_split<T, 5, 1>(a, cap, st) || launch_x3<5, false, false>(a, cap, st);
      // (5x5 stride 2 on planes of few tiles, the fp32 instruction's split form -> this: 64->128 at 32x48 20.8 -> 12.1 us,
      // 128->256 at 16x24 16.5 -> 13.1, at 32x32 16.8 -> 14.0; 32->64 at 64x96, two chunks and not split, 14.7 -> 12.3)
      if (k == 5 && s == 2) return launch_split<T, 5, 2>(a, cap, st) || launch_x3<5, false, false, 2>(a, cap, st);
      return false;
    }
  }
  switch (k * 10 + s) {
    case 11: return launch_ks<T, 1, 1>(a, cap, st);
    case 12: return launch_ks<T, 1, 2>(a, cap, st);
    case 31: return launch_split<T, 3, 1>(a, cap, st) || launch_ks<T, 3, 1>(a, cap, st);
    case 32: return launch_split<T, 3, 2>(a, cap, st) || launch_ks<T, 3, 2>(a, cap, st);
    case 51: return launch_split<T, 5, 1>(a, cap, st) || launch_ks<T, 5, 1>(a, cap, st);
    case 52: return launch_split<T, 5, 2>(a, cap, st) || launch_ks<T, 5, 2>(a, cap, st);
    case 71: return launch_ks<T, 7, 1>(a, cap, st);
    case 72: return launch_ks<T, 7, 2>(a, cap, st);
    default: return false;
  }
}
}  // namespace

