// Masked 3x3 stride-1 conv on planes of few tiles: the whole contraction of an output inside one workgroup, one launch.
//
// What bounds these layers (256 channels at 8x12 .. 32x32) is neither memory nor the matrix cores but the trips to memory one after
// the other in a launch -- arguments, tile list, masks and pixels, sums -- and the launches themselves: the split form of
// k_conv_mfma fills the chip with parts of the contraction and pays a second launch and a trip through memory for it.  Here
// a workgroup is small in outputs instead: DEEP_COLS channels of ROWS rows of a tile, and its DEEP_WAVES waves share the contraction,
// 32 channels (a chunk) a wave, with 64 or 128 channels some of the taps of a chunk.
//   * Nothing is shared before the sums: a wave stages the window of its own chunk in its own part of the LDS, so there is no
//     barrier until the partial sums meet there.  The window's pixels are asked for beside their mask bytes.
//   * The filter of a wave's first chunk depends on the workgroup's number alone: it is asked for at the very start, into registers
//     (9 taps x 3 terms x 16 bytes a lane), and arrives while the tile list, masks and pixels are on their way.  A later
//     chunk's follow as the registers fall free.
//   * The filter is the first operand of v_mfma_f32_16x16x32_bf16, so that a lane ends with four adjacent channels of a pixel.
//   * fp32 deltas as three bf16 terms (split3), the products by size in three accumulators, so that the large ones are added up
//     among themselves: chains of 9 sums a chunk.  Error of the sums against fp64, relative 2-norm, split form -> this:
//     256->256 1.20e-7 -> 1.07e-7, 512->512 1.90e-7 -> 1.44e-7, 64->64 1.4e-7 -> 0.8e-7.  bf16: three accumulators in turn.
// Measured, back to back on one plane with all pixels active, split form (two launches) -> this: fp32 256->256 at 8x12 9.95 ->
// 6.5 us, at 16x16 11.8 -> 7.5, at 16x24 11.8 -> 8.8, 512->512 at 16x16 15.9 -> 12.4, 128->128 9.2 -> 5.4, 64->64 at 16x24
// 8.0 -> 4.7; bf16 8.0 -> 4.4, 8.8 -> 4.5, 9.2 -> 4.9, 11.4 -> 6.5, 6.4 -> 4.3, 5.7 -> 3.9.  The pass over several chunks is bound by the filter's
// way from L2 (442 KB a workgroup for 512 fp32 channels).
#include "mie_conv_mfma_impl.h"

namespace {

typedef float v4acc __attribute__((ext_vector_type(4)));

__device__ __forceinline__ void mma16(v4acc& acc, const float4& w, const float4& x) {
  const v4f w4 = {w.x, w.y, w.z, w.w}, x4 = {x.x, x.y, x.z, x.w};
  acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(mie_bf16x8, w4), __builtin_bit_cast(mie_bf16x8, x4), acc, 0, 0, 0);
}

constexpr int DEEP_WAVES = 8, DEEP_COLS = 16;

// TPC: the waves a chunk's taps are dealt out to.  ROWS: rows of the workgroup's outputs.
template <typename T, int TPC, int ROWS>
__global__ __launch_bounds__(64 * DEEP_WAVES) void k_conv_deep(ConvArgsT<T> a) {
  constexpr bool X3 = sizeof(T) == 4;
  constexpr int K = 3, PL = X3 ? 3 : 1, GPS = X3 ? 2 : 1;
  constexpr int CC = 32, EPS = 8, Q4 = CC / EPS, LS = CC + EPS;
  constexpr int WX = 7 + K, WY = ROWS - 1 + K, NPIX = WX * WY;
  constexpr int RP = row_pitch_dw(WX, LS / 2, 1) * 2, STAGE = WY * RP;      // elements: row, term plane
  constexpr int NSLOT = NPIX * Q4, NLD = (NSLOT + 63) / 64;
  constexpr int NCW = DEEP_WAVES / TPC, NT = (K * K + TPC - 1) / TPC;
  constexpr int MB = ROWS * 8 / 16;
  constexpr int OS = DEEP_COLS + 4;                                        // floats per pixel of a wave's parked sums
  static_assert(OS * ROWS * 8 * 4 <= PL * STAGE * 2, "the sums fit where the pixels were");
  __shared__ __attribute__((aligned(16))) mie_bf16 smem[DEEP_WAVES * PL * STAGE];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int kg = lane >> 4, l16 = lane & 15;
  const int by = blockIdx.x + conv_args_entry_zero(a), bx = blockIdx.y;
  const int co0 = by * DEEP_COLS, cout = a.cout;

  const int cg = wave % NCW, tc = wave / NCW;
  const int nch1 = a.c1 / CC, nch = nch1 + (a.x2 != nullptr ? a.c2 / CC : 0);

  // filter of chunk c, this lane's part
  const int w_lane = (((kg >> 1) * (K * K * PL * 2) + (kg & 1)) * cout + co0 + l16) * EPS;
  auto chunk_w = [&](int c) -> const mie_bf16* {
    return reinterpret_cast<const mie_bf16*>(a.filt_mc) + (long long)(c * (CC / 16)) * (K * K * PL * 2) * cout * EPS;
  };
  float4 w[NT][PL];
  auto load_w = [&](const mie_bf16* p, int i) {
    int tap = tc + TPC * i;
    if (TPC > 1 && tap >= K * K) tap = K * K - 1;
#pragma unroll
    for (int q = 0; q < PL; ++q) w[i][q] = *reinterpret_cast<const float4*>(p + (long long)((tap * PL + q) * 2) * cout * EPS + w_lane);
  };
  if (cg < nch) {
    const mie_bf16* p = chunk_w(cg);
#pragma unroll
    for (int i = 0; i < NT; ++i) load_w(p, i);
  }

  int n, y0, x0;
  const int tk = mie_pick_tile(a.ts, bx / (8 / ROWS), n, y0, x0);
  y0 += ROWS * (bx % (8 / ROWS));
  const int hout = a.ts.h, wout = a.ts.w;
  if (tk == 0 || y0 >= hout) return;

  // the outputs of this thread: pixel it >> 2, channels 4 * (it & 3) ... of the slab (threads of a higher number: the same again)
  const int it = tid & (ROWS * 8 * 4 - 1);
  const int oy = y0 + (it >> 5), ox = x0 + ((it >> 2) & 7), co = co0 + 4 * (it & 3);
  const bool mine = tid < ROWS * 8 * 4 && oy < hout && ox < wout;
  const int opix = (oy < hout && ox < wout) ? (n * hout + oy) * wout + ox : 0;
  const long long off = (long long)opix * cout + co;
  if (tk == 2) {
    if (mine) mie_st4(a.out, off, make_float4(0.f, 0.f, 0.f, 0.f));
    return;
  }

  // ---- the window's pixels, CC channels of them, for this wave alone
  mie_bf16* const sw = smem + wave * (PL * STAGE);
  int st_po[NLD], st_lds[NLD];
  unsigned inb = 0u;
  const int q8 = EPS * (lane & (Q4 - 1));
#pragma unroll
  for (int i = 0; i < NLD; ++i) {
    const int pix = (lane + 64 * i) / Q4, ly = pix / WX, lx = pix - ly * WX;
    const int iy = y0 - a.pad + ly, ix = x0 - a.pad + lx;
    const bool k = pix < NPIX && iy >= 0 && iy < a.h_in && ix >= 0 && ix < a.w_in;
    st_po[i] = k ? (n * a.h_in + iy) * a.w_in + ix : 0;
    st_lds[i] = ly * RP + lx * LS + q8;
    inb |= (k ? 1u : 0u) << i;
  }
  float4 xr[NLD][GPS];
  auto load_x = [&](int c) {
    const bool second = c >= nch1;
    const T* p = second ? a.x2 : a.x;
    const int cs = second ? a.c2 : a.c1, ci0 = (second ? c - nch1 : c) * CC + q8;
#pragma unroll
    for (int i = 0; i < NLD; ++i)
#pragma unroll
      for (int g = 0; g < GPS; ++g) xr[i][g] = *reinterpret_cast<const float4*>(p + (long long)st_po[i] * cs + ci0 + 4 * g);
  };
  auto store_x = [&](unsigned ok) {
#pragma unroll
    for (int i = 0; i < NLD; ++i) {
      if (64 * i + 63 >= NSLOT && lane + 64 * i >= NSLOT) continue;
      const bool k = (ok >> i) & 1u;
      float4 pl[3];
      const float4 u = make_float4(k ? xr[i][0].x : 0.f, k ? xr[i][0].y : 0.f, k ? xr[i][0].z : 0.f, k ? xr[i][0].w : 0.f);
      if constexpr (X3) {
        const float4 v = make_float4(k ? xr[i][GPS - 1].x : 0.f, k ? xr[i][GPS - 1].y : 0.f, k ? xr[i][GPS - 1].z : 0.f, k ? xr[i][GPS - 1].w : 0.f);
        const float f[8] = {u.x, u.y, u.z, u.w, v.x, v.y, v.z, v.w};
        split3(f, pl);
      } else {
        pl[0] = u;
      }
#pragma unroll
      for (int q = 0; q < PL; ++q) *reinterpret_cast<float4*>(sw + q * STAGE + st_lds[i]) = pl[q];
    }
  };
  unsigned ok1 = 0u, ok2 = 0u;
  const uint8_t* const live_m = a.refresh ? nullptr : a.ts.pixmask;
  const long long offs[1] = {off};
  const int cos[1] = {co}, at[1] = {opix};
  const bool oks[1] = {true};
  float4 r0[1], add[1];
  unsigned live_b[1];
  {
    unsigned b1[NLD], b2[NLD];
    load_x(cg < nch ? cg : 0);
    mie_mask_ask(a.xm, a.filt_mc, st_po, b1);
    mie_mask_ask(a.x2 != nullptr ? a.x2m : nullptr, a.filt_mc, st_po, b2);
    mie_mask_ask(live_m, a.filt_mc, at, live_b);
    conv_epilogue_load4<T, 1>(a, offs, oks, r0, add);
    mie_mask_asked();
    ok1 = mie_mask_take(a.xm, b1, inb);
    ok2 = mie_mask_take(a.x2 != nullptr ? a.x2m : nullptr, b2, inb);
  }

  // ---- contraction
  v4acc acc[MB], sm[MB], sl[MB];      // fp32: products of 1, 2^-8 and 2^-16 of the largest
#pragma unroll
  for (int b = 0; b < MB; ++b) acc[b] = v4acc{0.f, 0.f, 0.f, 0.f}, sm[b] = sl[b] = v4acc{0.f, 0.f, 0.f, 0.f};
  const int x_lane = (l16 >> 3) * RP + (l16 & 7) * LS + EPS * kg;
  auto chunk = [&](int c, auto more) {
    constexpr bool MORE = decltype(more)::value;
    store_x(c >= nch1 ? ok2 : ok1);
    __builtin_amdgcn_wave_barrier();
    const mie_bf16* p = nullptr;
    if constexpr (MORE) {
      load_x(c + NCW);
      p = chunk_w(c + NCW);
    }
#pragma unroll
    for (int i = 0; i < NT; ++i) {
      const int tap = tc + TPC * i;
      if (TPC == 1 || TPC * i + TPC <= K * K || tap < K * K) {
        const int ky = tap / K, kx = tap - ky * K;
        float4 xv[MB][PL];
#pragma unroll
        for (int b = 0; b < MB; ++b)
#pragma unroll
          for (int q = 0; q < PL; ++q) xv[b][q] = *reinterpret_cast<const float4*>(sw + q * STAGE + x_lane + (2 * b + ky) * RP + kx * LS);
        if constexpr (X3) {
          auto term = [&](v4acc (&s)[MB], int tw, int tx) {
#pragma unroll
            for (int b = 0; b < MB; ++b) mma16(s[b], w[i][tw], xv[b][tx]);
          };
          term(acc, 0, 0); term(sl, 0, 2); term(sm, 0, 1);
          term(sl, 1, 1); term(sm, 1, 0); term(sl, 2, 0);
        } else {
#pragma unroll
          for (int b = 0; b < MB; ++b) mma16(i % 3 == 0 ? acc[b] : i % 3 == 1 ? sm[b] : sl[b], w[i][0], xv[b][0]);
        }
      }
      if constexpr (MORE) load_w(p, i);
    }
    __builtin_amdgcn_wave_barrier();
  };
  int c = cg;
  for (; c + NCW < nch; c += NCW) chunk(c, std::true_type());
  if (c < nch) chunk(c, std::false_type());

  // ---- the waves' sums meet in LDS, each in its wave's own part: pixel 16 * b + l16, channels 4 * kg ...
  float* const park = reinterpret_cast<float*>(sw);
#pragma unroll
  for (int b = 0; b < MB; ++b) {
    const v4acc s = acc[b] + (sm[b] + sl[b]);
    *reinterpret_cast<float4*>(park + (16 * b + l16) * OS + 4 * kg) = make_float4(s[0], s[1], s[2], s[3]);
  }
  __syncthreads();
  if (!mine) return;
  float4 part[DEEP_WAVES];
#pragma unroll
  for (int k = 0; k < DEEP_WAVES; ++k)
    part[k] = *reinterpret_cast<const float4*>(reinterpret_cast<const float*>(smem + k * (PL * STAGE)) + (it >> 2) * OS + 4 * (it & 3));
#pragma unroll
  for (int k = 1; k < DEEP_WAVES; ++k) {
    part[0].x += part[k].x; part[0].y += part[k].y; part[0].z += part[k].z; part[0].w += part[k].w;
  }
  const float4 sums[1] = {part[0]};
  const bool live[1] = {mie_mask_take(live_m, live_b, 1u) != 0u};
  conv_epilogue_store4<T, 1>(a, offs, cos, oks, sums, r0, add, live);
}

template <typename T, int ROWS>
void launch_rows(const ConvArgsT<T>& a, unsigned cap, hipStream_t st) {
  const dim3 grid(a.cout / DEEP_COLS, 8 / ROWS * cap), block(64 * DEEP_WAVES);
  const int nch = (a.c1 + a.c2) / 32;
  if (nch >= 8) hipLaunchKernelGGL((k_conv_deep<T, 1, ROWS>), grid, block, 0, st, a);
  else if (nch >= 4) hipLaunchKernelGGL((k_conv_deep<T, 2, ROWS>), grid, block, 0, st, a);
  else hipLaunchKernelGGL((k_conv_deep<T, 4, ROWS>), grid, block, 0, st, a);
}

// Two rows a workgroup while that makes one workgroup a CU at most (the filter is read twice as often: fp32 256->256 at 8x12 7.55
// with four -> 6.50 us with two, at 16x16, 256 workgroups, 8.7 -> 7.5, at 16x24, 384, 8.8 -> 12.5).
template <typename T>
bool launch_deep(const ConvArgsT<T>& a, int k, int s, unsigned cap, hipStream_t st) {
  const int dtype = sizeof(T) == 2 ? MIE_DTYPE_BF16 : a.x3 ? MIE_DTYPE_F32_BF16X3 : MIE_DTYPE_F32;
  if (a.ws != nullptr || !mie_conv_deep_form(k, s, a.c1, a.c2, a.cout, cap, dtype)) return false;
  if (8 / 2 * (long long)cap * (a.cout / DEEP_COLS) <= 256) launch_rows<T, 2>(a, cap, st);
  else launch_rows<T, 4>(a, cap, st);
  return true;
}

}  // namespace

// From two chunks on, while the workgroups are one round of the chip: one a CU with the three terms' 129 KB of LDS and 208
// registers, two in bf16.  (fp32 256->256 at 24x24, 288 workgroups: 14.0 us in the form of 64 columns, 15.1 in this; 128->512 at 16x24,
// 384, 11.9 and 11.6; 256->512 at 32x32, 1024, 18.0 and 30.2.  bf16 128->256 at 32x32, 512 workgroups, 6.6 and 6.0; 256->256 at
// 33x44, 960, 8.7 and 11.2.)
bool mie_conv_deep_form(int k, int s, int c1, int c2, int cout, long long tiles, int dtype) {
  if (k != 3 || s != 1 || (dtype != MIE_DTYPE_BF16 && dtype != MIE_DTYPE_F32_BF16X3)) return false;
  if (c1 % 32 != 0 || c2 % 32 != 0 || c1 + c2 < 64 || cout % DEEP_COLS != 0) return false;
  return 2 * tiles * (cout / DEEP_COLS) <= (dtype == MIE_DTYPE_BF16 ? 512 : 256);
}

bool mie_launch_conv_deep(const ConvArgsT<float>& a, int k, int s, unsigned cap, hipStream_t st) { return launch_deep(a, k, s, cap, st); }
bool mie_launch_conv_deep(const ConvArgsT<mie_bf16>& a, int k, int s, unsigned cap, hipStream_t st) { return launch_deep(a, k, s, cap, st); }
