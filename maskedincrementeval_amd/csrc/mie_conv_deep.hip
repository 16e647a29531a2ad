// Masked convs on planes of few tiles -- 3x3 stride 1, also with the gate chain of a ConvLSTM or ConvGRU as its epilogue, 3x3 and 5x5
// stride 2, 5x5 over an up-sampled sum, the 3x3 transposed conv -- with the whole contraction of an output inside one workgroup, in one launch.
//
// What bounds these layers (256 channels at 8x12 .. 32x32) is neither memory nor the matrix cores but the trips to memory one after
// the other in a launch -- arguments, tile list, masks and pixels, sums -- and the launches themselves: the split form of
// k_conv_mfma fills the chip with parts of the contraction and pays a second launch and a trip through memory for it.  Here
// a workgroup is small in outputs instead: DEEP_COLS channels of ROWS rows of a tile, and its DEEP_WAVES waves share the contraction:
// NCW chunks of 32 input channels are in LDS at a time, and the taps of each are dealt out to DEEP_WAVES / NCW waves.
//   * The filter of a wave's first chunk depends on the workgroup's number alone: it is asked for at the very start, into registers,
//     behind the tile list's words, and arrives while list, masks and pixels are on their way.  A later chunk's follows as
//     the registers fall free.  A workgroup's 16 columns come through a 64-byte path to its CU, 221 KB of them for 256 fp32 channels: 1.4 us.
//   * The window's pixels are asked for beside their mask bytes.  With 8 chunks at a time a wave stages the one it multiplies
//     itself (OWN), and nothing is shared before the sums; with fewer all waves stage, and meet.
//   * Few chunks at a time mean few taps a wave: little filter in registers (48 of them for a 5x5 chunk dealt out to 8 waves), short code that
//     every launch fetches anew, a second workgroup on the CU.  fp32 5x5 128->256 at 8x12 with 1, 2, 4 chunks at a time 9.7, 10.1, 15.9 us; 3x3
//     256->256 8.0 with 2, 7.5 with 4, 6.9 with 8 of their own; at 64 channels 2 (4.5) beat 1 (4.8).
//   * The filter is the first operand of v_mfma_f32_16x16x32_bf16, so that a lane ends with four adjacent channels of a pixel, or the
//     four gates of a hidden channel: the gate chain runs on four times the threads it has in k_conv_mfma.
//   * fp32 deltas as three bf16 terms (split3), the products by size in three accumulators, so that the large ones are added up
//     among themselves: chains of 9 sums a chunk.  Error of the sums against fp64, relative 2-norm, split form -> this:
//     256->256 1.20e-7 -> 1.07e-7, 512->512 1.90e-7 -> 1.44e-7, 64->64 1.4e-7 -> 0.8e-7.  bf16: three accumulators in turn.
//     (For MIE_DTYPE_F32_F16X2 too, but for the 3x3 convs of many channels: DEEP_F2_FROM.)
//   * In two fp16 terms (F2) the scale is a pass's, a wave's own with OWN: every DEEP_BL taps the leading products are folded into the total at
//     its true size, with what that rounds off carried on among the small ones (deep_fold), and chunks of any size add up.
//   * Up-sampling: the sums of the source pixels in LDS, the window blended from them, as in k_conv_mfma.  fp32 layers of 256 channels are
//     not taken: 25 taps of filter, 614 KB a workgroup, take as long as the split form (256->128 at 16x24 16.4 us, 14.6).
// Measured back to back on one plane with all pixels active, the filter another each time, split form -> this, us:
//                     fp32                                                    bf16
//   3x3 256->256      8x12 15.8 -> 6.9, 16x16 15.9 -> 7.4, 24x24 14.3 -> 11.5   8.1 -> 4.5, 8.1 -> 4.6, 8.2 -> 6.2
//   3x3 512->512      16x16 26.4 -> 14.9                                       11.3 -> 6.3
//   3x3 64->64        32x32 8.2 -> 4.4, 64x64 8.7 -> 6.6                        5.9 -> 4.0, 6.1 -> 5.0
//   gates 256         8x12 13.2 -> 9.7, two inputs at 16x16 28.1 -> 23.0        10.0 -> 5.0, 12.2 -> 10.0
//   gates 128, 64     16x24 11.1 -> 8.5, 32x32 8.6 -> 6.7                       6.8 -> 5.3, 6.2 -> 5.1
//   5x5 s2 32->64     32x48 10.3 -> 5.7, 64x64 10.9 -> 7.5                      8.1 -> 4.4, 8.2 -> 5.3
//   5x5 s2 128->256   8x12 11.2 -> 8.6, 16x16 13.1 -> 9.8                       9.5 -> 5.2, 9.5 -> 5.5
//   3x3 s2 64->128    32x32 11.6 -> 5.9 (from the fp32 instruction)              7.0 -> 4.6
//   3x3 s2 256->512   16x16 16.1 -> 12.0                                       10.7 -> 6.1
//   up 128->64, 64->32  32x48 13.5 -> 11.4, 64x64 15.9 -> 7.8                   11.9 -> 6.8, 8.5 -> 5.4
// Whole passes: fp32 1x64x96 163.1 -> 147 us, 1x128x128 231 -> 215.
// With more input channels than these the split form is the faster one (mie_conv_deep_faster).  Counters (256->256 at 8x12, fp32): matrix
// cores busy 12 % of a CU's time, 250 KB a workgroup through its path to the L2s (1.6 of 7.7 us), 47 % of the LDS cycles bank conflicts.
// The fp32 gates forms of eight rows are at 256 registers and keep 20 (ConvLSTM) and 12 (ConvGRU) bytes a lane in scratch memory.
#include "mie_conv_mfma_impl.h"

namespace {

typedef float v4acc __attribute__((ext_vector_type(4)));

__device__ __forceinline__ void mma16(v4acc& acc, const float4& w, const float4& x) {
  const v4f w4 = {w.x, w.y, w.z, w.w}, x4 = {x.x, x.y, x.z, x.w};
  acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(mie_bf16x8, w4), __builtin_bit_cast(mie_bf16x8, x4), acc, 0, 0, 0);
}

// A place in global memory by its type: behind an asm the compiler no longer sees where a plain pointer came from and makes flat loads
// of it, which a wait for LDS waits for too.
typedef const __attribute__((address_space(1))) char* GlobalBytes;
__device__ __forceinline__ float4 global_ld4(GlobalBytes p) {
  const v4f v = *(const __attribute__((address_space(1))) v4f*)p;
  return make_float4(v[0], v[1], v[2], v[3]);
}

constexpr int DEEP_BL = 3;
constexpr int DEEP_WAVES = 8, DEEP_COLS = 16, DEEP_THREADS = 64 * DEEP_WAVES, DEEP_WGS = 256;
enum { DEEP_PLAIN = 0, DEEP_GATES = 1, DEEP_UP = 2, DEEP_GRU = 3 };

__device__ __forceinline__ void mma16_f16(v4acc& acc, const float4& w, const float4& x) {
  const v4f w4 = {w.x, w.y, w.z, w.w}, x4 = {x.x, x.y, x.z, x.w};
  acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(mie_f16x8, w4), __builtin_bit_cast(mie_f16x8, x4), acc, 0, 0, 0);
}
// Four of a lane's eight channels on the fp32 instruction, from fp32 copies laid out as the terms are (the first four in plane 0).
__device__ __forceinline__ void mma16_f32(v4acc& acc, const float4& w, const float4& x) {
  acc = __builtin_amdgcn_mfma_f32_16x16x4f32(w.x, x.x, acc, 0, 0, 0);
  acc = __builtin_amdgcn_mfma_f32_16x16x4f32(w.y, x.y, acc, 0, 0, 0);
  acc = __builtin_amdgcn_mfma_f32_16x16x4f32(w.z, x.z, acc, 0, 0, 0);
  acc = __builtin_amdgcn_mfma_f32_16x16x4f32(w.w, x.w, acc, 0, 0, 0);
}
// Two terms: the products so far (acc, at the scales that c0 takes off) to the total, what the addition rounds off to the small ones.
__device__ __forceinline__ void deep_fold(v4acc& tot, v4acc& low, v4acc& acc, float c0) {
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const float t = tot[r], u = fmaf(acc[r], c0, t);
    low[r] += fmaf(acc[r], c0, t - u);
    tot[r] = u;
    acc[r] = 0.f;
  }
}

// Sizes of a form; NCW: chunks of 32 channels in LDS at a time, ROWS: output rows of a tile, AR: 0 bf16, 1 fp32 in three bf16 terms, 2 in
// two fp16 terms.
template <int AR, int K, int S, int NCW, int ROWS, int KIND>
struct Deep {
  static constexpr bool X3 = AR != 0;
  static constexpr int PL = AR == 2 ? 2 : X3 ? 3 : 1, GPS = X3 ? 2 : 1;      // term planes; 16-byte loads of 8 channels
  static constexpr int CC = 32, EPS = 8, LS = CC + EPS;        // LDS elements per staged pixel of a chunk
  static constexpr int TPC = DEEP_WAVES / NCW, NT = (K * K + TPC - 1) / TPC;
  static constexpr int WX = 7 * S + K, WY = (ROWS - 1) * S + K, NPIX = WX * WY;
  static constexpr int RP = row_pitch_dw(WX, LS / 2, S) * 2, STAGE = WY * RP;      // elements: row, term plane
  static constexpr bool OWN = NCW == DEEP_WAVES && KIND != DEEP_UP;               // a wave stages its chunk itself, for itself
  static constexpr int SPP = (OWN ? 1 : NCW) * (CC / EPS), STEP = (OWN ? 64 : DEEP_THREADS) / SPP;   // slots of 8 channels a pixel, pixels a round
  static constexpr int NLD = (NPIX + STEP - 1) / STEP;
  static constexpr int MB = ROWS * 8 / 16;
  static constexpr int OS = DEEP_COLS + 4;                     // floats per pixel of a wave's parked sums
  static constexpr int PARK = OWN ? PL * STAGE / 2 : ROWS * 8 * OS;                // floats from wave to wave (OWN: where its pixels were)
  static_assert(PARK >= ROWS * 8 * OS, "the sums fit where the pixels were");
  static constexpr bool UP = KIND == DEEP_UP;
  static constexpr int SX = 8, SY = UP ? WY / 2 + 2 : 0, NLO = UP ? (SX * SY + STEP - 1) / STEP : 1;   // source pixels of a window
  static constexpr int LOS = NCW * CC + 4;                     // floats per source pixel
  static constexpr int WIN_B = NCW * PL * STAGE * 2, LO_B = SX * SY * LOS * 4, PARK_B = DEEP_WAVES * PARK * 4;
  static constexpr int BYTES = WIN_B + LO_B > PARK_B ? WIN_B + LO_B : PARK_B;
};

template <typename T, int AR, int K, int S, int NCW, int ROWS, int KIND>
__global__ __launch_bounds__(DEEP_THREADS) void k_conv_deep(ConvArgsT<T> a) {
  typedef Deep<AR, K, S, NCW, ROWS, KIND> D;
  static_assert((AR != 0) == (sizeof(T) == 4), "fp32 deltas in terms, bf16 as they are");
  constexpr bool X3 = D::X3, F2 = AR == 2, UP = D::UP, GATES = KIND == DEEP_GATES, GRU = KIND == DEEP_GRU, AGAIN = AR == 1 && S == 2;
  constexpr int PL = D::PL, GPS = D::GPS, CC = D::CC, EPS = D::EPS, LS = D::LS, TPC = D::TPC, NT = D::NT;
  constexpr int WX = D::WX, NPIX = D::NPIX, RP = D::RP, STAGE = D::STAGE, SPP = D::SPP, STEP = D::STEP, NLD = D::NLD;
  constexpr bool OWN = D::OWN;
  constexpr int MB = D::MB, OS = D::OS, NLO = D::NLO, LOS = D::LOS;
  static_assert(D::BYTES <= 160 * 1024, "LDS of a CU");
  static_assert(!UP || (K == 5 && S == 1), "the up-sampling variant is the 5x5 stride-1 conv");
  static_assert(!F2 || (K == 3 && S == 1 && !UP), "two terms: the 3x3 convs");
  __shared__ __attribute__((aligned(16))) char smem[D::BYTES];
  __shared__ float s_f2[F2 && !OWN ? DEEP_WAVES + 2 : 1];      // largest values of the waves' slots; whether a group of a pass does not fit, of
                                                               // every other one in the same place
  mie_bf16* const win = reinterpret_cast<mie_bf16*>(smem);
  float* const s_lo = reinterpret_cast<float*>(smem + D::WIN_B);
  float* const park = reinterpret_cast<float*>(smem);

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int kg = lane >> 4, l16 = lane & 15;
  // the slabs are dealt out to the XCDs in eighths: a filter slab is fetched by one of the L2s, and lines that neighbouring slabs
  // share (a pixel's 16 channels are 32 or 64 bytes, of a gates conv 8 or 16) are written by one
  const int slabs = a.cout / DEEP_COLS, bx = blockIdx.y;
  int by = blockIdx.x + conv_args_entry_zero(a);
  if ((slabs & 7) == 0) by = (by & 7) * (slabs >> 3) + (by >> 3);
  const int co0 = by * DEEP_COLS, cout = a.cout;

  const int cg = wave % NCW, tc = wave / NCW;
  const int nch1 = a.c1 / CC, nch = nch1 + (!UP && a.x2 != nullptr ? a.c2 / CC : 0);

  // Filter: where this wave's taps of chunk c start, and a lane's place in a term of a tap, in bytes.  Tap i of the wave to
  // registers.
  const unsigned w_step = 2u * cout * (2 * EPS);                // from term to term, and from the last of a tap to the next tap
  const unsigned w_lane = (((kg >> 1) * (K * K * PL * 2) + (kg & 1)) * cout + co0 + l16) * (2 * EPS);
  auto chunk_w = [&](int c) -> const char* {
    return reinterpret_cast<const char*>(a.filt_mc) + ((long long)(c * (CC / 16)) * (K * K) + tc) * PL * w_step;
  };
  float4 w[NT][PL];
  // (The first chunk's taps from one base by a place that a lane works out for each; the later ones' bases by scalar sums, beside
  // the matrix instructions.  The asm keeps the compiler from taking the one for the other.  fp32 256->256 at 8x12, one chunk a wave,
  // 6.9 us, by scalar sums 7.3; 512->512 at 16x16, two, 14.8, by places of a lane 16.3.)
  auto load_w = [&](const char* p, int i, auto first) {
    const bool none = TPC > 1 && TPC * i + TPC > K * K && tc + TPC * i >= K * K;      // (no such tap: the last one again)
    const unsigned at = (none ? K * K - 1 - tc : TPC * i) * PL * w_step;
#pragma unroll
    for (int q = 0; q < PL; ++q) {
      if constexpr (decltype(first)::value) {
        w[i][q] = *reinterpret_cast<const float4*>(p + (w_lane + at + q * w_step));
      } else {
        GlobalBytes t = (GlobalBytes)p + (at + q * w_step);
        asm("" : "+s"(t));
        w[i][q] = global_ld4(t + w_lane);
      }
    }
  };
  const int pos = bx / (8 / ROWS);
  TileAsk ask = mie_tile_ask(a.ts, pos);
  __builtin_amdgcn_sched_barrier(0);
  {
    const char* p = chunk_w(cg < nch ? cg : 0);
#pragma unroll
    for (int i = 0; i < NT; ++i) load_w(p, i, std::true_type());
  }

  int n, y0, x0;
  const int tk = mie_tile_take(a.ts, pos, ask, n, y0, x0);
  y0 += ROWS * (bx % (8 / ROWS));
  const int hout = a.ts.h, wout = a.ts.w;
  if (tk == 0 || y0 >= hout) return;

  // the outputs of this thread: pixel it >> 2, channels 4 * (it & 3) ... of the slab, with GATES the four gates of one hidden
  // channel (threads of a higher number: the same again)
  const int it = tid & (ROWS * 8 * 4 - 1);
  const int oy = y0 + (it >> 5), ox = x0 + ((it >> 2) & 7), co = co0 + 4 * (it & 3);
  const bool mine = tid < ROWS * 8 * 4 && oy < hout && ox < wout;
  const int opix = (oy < hout && ox < wout) ? (n * hout + oy) * wout + ox : 0;
  const long long off = (long long)opix * cout + co;
  // (GRU: the first groups of four of every eight columns, update gates, work for the second, candidates, too)
  const bool idle = GRU && (it & 1) != 0;
  const long long ho = GATES ? (long long)opix * a.hid + co / 4 : GRU ? (long long)opix * a.hid + (co & ~7) / 2 : 0;
  if (tk == 2) {
    if (!mine || idle) return;
    if constexpr (GRU) {
      mie_st4(a.g_dh, ho, make_float4(0.f, 0.f, 0.f, 0.f));
    } else if constexpr (GATES) {
      mie_st(a.g_dh, ho, 0.f);
      mie_st(a.g_dc, ho, 0.f);
    } else {
      mie_st4(a.out, off, make_float4(0.f, 0.f, 0.f, 0.f));
    }
    return;
  }

  // ---- the window's pixels, NCW * CC channels of them at a time; UP: of the source block they are blended from
  const int sq = (OWN ? lane : tid) % SPP, p0 = (OWN ? lane : tid) / SPP;
  const int ck = OWN ? cg : sq / (CC / EPS), q8 = EPS * (sq % (CC / EPS));      // chunk of those in LDS and channel this thread stages
  const int iy0 = y0 * S - a.pad, ix0 = x0 * S - a.pad;
  const int h_lo = a.h_in >> 1, w_lo = a.w_in >> 1;
  const int lo_y0 = (iy0 >> 1) - 1, lo_x0 = (ix0 >> 1) - 1;
  constexpr int NL = UP ? NLO : NLD;
  int st_po[NL];
  unsigned inb = 0u;
#pragma unroll
  for (int i = 0; i < NL; ++i) {
    const int pix = p0 + STEP * i;
    const int ly = UP ? pix / D::SX : pix / WX, lx = UP ? pix % D::SX : pix - ly * WX;
    const int iy = (UP ? lo_y0 : iy0) + ly, ix = (UP ? lo_x0 : ix0) + lx;
    const int h = UP ? h_lo : a.h_in, wd = UP ? w_lo : a.w_in;
    const bool k = pix < (UP ? D::SX * D::SY : NPIX) && iy >= 0 && iy < h && ix >= 0 && ix < wd;
    st_po[i] = k ? (n * h + iy) * wd + ix : 0;
    inb |= (k ? 1u : 0u) << i;
  }
  float4 xr[NL][GPS], xb[UP ? NL : 1][GPS];
  auto load_x = [&](int pass) {
    int c = pass * NCW + ck;
    if (c >= nch) c = 0;
    const bool second = !UP && c >= nch1;
    const T* p = second ? a.x2 : a.x;
    const int cs = second ? a.c2 : a.c1, ci0 = (second ? c - nch1 : c) * CC + q8;
#pragma unroll
    for (int i = 0; i < NL; ++i)
#pragma unroll
      for (int g = 0; g < GPS; ++g) xr[i][g] = *reinterpret_cast<const float4*>(p + (long long)st_po[i] * cs + ci0 + 4 * g);
    if constexpr (UP) {
      const T* pb = a.x2 != nullptr ? a.x2 : a.x;
#pragma unroll
      for (int i = 0; i < NL; ++i)
#pragma unroll
        for (int g = 0; g < GPS; ++g) xb[i][g] = *reinterpret_cast<const float4*>(pb + (long long)st_po[i] * cs + ci0 + 4 * g);
    }
  };
  auto kept = [](const float4& v, bool k) { return make_float4(k ? v.x : 0.f, k ? v.y : 0.f, k ? v.z : 0.f, k ? v.w : 0.f); };
  F2Groups groups;
  auto put = [&](int at, const float (&f)[8], auto terms) {
    if constexpr (F2) {
      float4 pl[2] = {make_float4(f[0], f[1], f[2], f[3]), make_float4(f[4], f[5], f[6], f[7])};
      if constexpr (decltype(terms)::value) groups.terms(f, pl);
#pragma unroll
      for (int q = 0; q < PL; ++q) *reinterpret_cast<float4*>(win + q * STAGE + at) = pl[q];
    } else if constexpr (X3) {
      float4 pl[3];
      split3(f, pl);
#pragma unroll
      for (int q = 0; q < PL; ++q) *reinterpret_cast<float4*>(win + q * STAGE + at) = pl[q];
    } else {
      *reinterpret_cast<float4*>(win + at) = f32_to_slot(f, T());
    }
  };
  unsigned ok1 = 0u, ok2 = 0u;
  const int st_c = ck * (PL * STAGE) + q8;      // this thread's place in a staged pixel
  // F2: the scale of a pass, a wave's own (OWN) or the workgroup's
  auto scale_of = [&](int pass, float m) {
    m = f2_wave_max(m);
    if constexpr (!OWN) {
      if (lane == 0) s_f2[wave] = m;
      if (pass == 0 && tid < 2) s_f2[DEEP_WAVES + tid] = 0.f;
      __syncthreads();
      m = f2_wave_max(s_f2[lane & (DEEP_WAVES - 1)]);
    }
    groups.start(f2_scale(m));
  };
  // (terms: in terms, or F2's fp32 form)
  auto store_x = [&](int pass, auto terms) {
    const int c = pass * NCW + ck;
    if constexpr (UP) {
#pragma unroll
      for (int i = 0; i < NL; ++i) {
        const int pix = p0 + STEP * i;
        if (pix >= D::SX * D::SY) continue;
        const bool k1 = (ok1 >> i) & 1u, k2 = (ok2 >> i) & 1u;
        float fa[8], fb[8];
        const float4 a0 = kept(xr[i][0], k1), b0 = kept(xb[i][0], k2);
        if constexpr (X3) {
          const float4 a1 = kept(xr[i][GPS - 1], k1), b1 = kept(xb[i][GPS - 1], k2);
          const float ta[8] = {a0.x, a0.y, a0.z, a0.w, a1.x, a1.y, a1.z, a1.w}, tb[8] = {b0.x, b0.y, b0.z, b0.w, b1.x, b1.y, b1.z, b1.w};
#pragma unroll
          for (int e = 0; e < 8; ++e) fa[e] = ta[e], fb[e] = tb[e];
        } else {
          slot_to_f32(a0, fa, T());
          slot_to_f32(b0, fb, T());
        }
        float* const d = s_lo + pix * LOS + 8 * sq;
        *reinterpret_cast<float4*>(d) = make_float4(fa[0] + fb[0], fa[1] + fb[1], fa[2] + fb[2], fa[3] + fb[3]);
        *reinterpret_cast<float4*>(d + 4) = make_float4(fa[4] + fb[4], fa[5] + fb[5], fa[6] + fb[6], fa[7] + fb[7]);
      }
      __syncthreads();
#pragma unroll
      for (int i = 0; i < NLD; ++i) {
        const int pix = p0 + STEP * i, ly = pix / WX, lx = pix - ly * WX;
        if (pix >= NPIX) continue;
        const int hy = iy0 + ly, hx = ix0 + lx;
        float o[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
        if (hy >= 0 && hy < a.h_in && hx >= 0 && hx < a.w_in) {
          int r0, r1, q0, q1;
          float lr0, lr1, lq0, lq1;
          conv_up2x_coef(hy, h_lo, r0, r1, lr0, lr1);
          conv_up2x_coef(hx, w_lo, q0, q1, lq0, lq1);
          const float* v00 = s_lo + ((r0 - lo_y0) * D::SX + (q0 - lo_x0)) * LOS + 8 * sq;
          const float* v01 = s_lo + ((r0 - lo_y0) * D::SX + (q1 - lo_x0)) * LOS + 8 * sq;
          const float* v10 = s_lo + ((r1 - lo_y0) * D::SX + (q0 - lo_x0)) * LOS + 8 * sq;
          const float* v11 = s_lo + ((r1 - lo_y0) * D::SX + (q1 - lo_x0)) * LOS + 8 * sq;
#pragma unroll
          for (int e = 0; e < 8; e += 4) {
            const float4 t00 = *reinterpret_cast<const float4*>(v00 + e), t01 = *reinterpret_cast<const float4*>(v01 + e);
            const float4 t10 = *reinterpret_cast<const float4*>(v10 + e), t11 = *reinterpret_cast<const float4*>(v11 + e);
            o[e] = conv_up2x_v(lr0, lr1, conv_up2x_h(lq0, lq1, t00.x, t01.x), conv_up2x_h(lq0, lq1, t10.x, t11.x));
            o[e + 1] = conv_up2x_v(lr0, lr1, conv_up2x_h(lq0, lq1, t00.y, t01.y), conv_up2x_h(lq0, lq1, t10.y, t11.y));
            o[e + 2] = conv_up2x_v(lr0, lr1, conv_up2x_h(lq0, lq1, t00.z, t01.z), conv_up2x_h(lq0, lq1, t10.z, t11.z));
            o[e + 3] = conv_up2x_v(lr0, lr1, conv_up2x_h(lq0, lq1, t00.w, t01.w), conv_up2x_h(lq0, lq1, t10.w, t11.w));
          }
        }
        put(st_c + ly * RP + lx * LS, o, terms);
      }
    } else {
      const unsigned ok = c >= nch ? 0u : c >= nch1 ? ok2 : ok1;
      if constexpr (F2 && decltype(terms)::value) {
        float m = 0.f;
#pragma unroll
        for (int i = 0; i < NL; ++i) {
          const float4 u = xr[i][0], v = xr[i][GPS - 1];
          const float f[8] = {u.x, u.y, u.z, u.w, v.x, v.y, v.z, v.w};
          m = __builtin_elementwise_maximum(m, (ok >> i) & 1u ? f2_amax8(f) : 0.f);
        }
        scale_of(pass, m);
      }
#pragma unroll
      for (int i = 0; i < NL; ++i) {
        const int pix = p0 + STEP * i, ly = pix / WX, lx = pix - ly * WX;
        if (STEP * i + STEP > NPIX && pix >= NPIX) continue;
        const bool k = (ok >> i) & 1u;
        const float4 u = kept(xr[i][0], k);
        if constexpr (X3) {
          const float4 v = kept(xr[i][GPS - 1], k);
          const float f[8] = {u.x, u.y, u.z, u.w, v.x, v.y, v.z, v.w};
          put(st_c + ly * RP + lx * LS, f, terms);
        } else {
          *reinterpret_cast<float4*>(win + st_c + ly * RP + lx * LS) = u;
        }
      }
    }
  };
  const uint8_t* const live_m = a.refresh ? nullptr : a.ts.pixmask;
  const uint8_t* const x2m = a.x2 != nullptr ? a.x2m : nullptr;
  const uint8_t* const cp_m = GATES && a.g_cpd != nullptr ? a.g_cpm : nullptr;
  const long long offs[1] = {off};
  const int cos[1] = {co}, at[1] = {opix};
  float4 r0[1], add[1];
  float g_cp = 0.f, g_cc = 0.f, g_dp = 0.f;
  unsigned live_b[1], cp_b[1];
  {
    unsigned b1[NL], b2[NL];
    load_x(0);
    mie_mask_ask(a.xm, a.filt_mc, st_po, b1);
    mie_mask_ask(x2m, a.filt_mc, st_po, b2);
    mie_mask_ask(live_m, a.filt_mc, at, live_b);
    if constexpr (GATES) {
      mie_mask_ask(cp_m, a.filt_mc, at, cp_b);
      r0[0] = *reinterpret_cast<const float4*>(a.res + off);
      g_cp = a.g_cpres[ho];
      g_cc = a.g_cres[ho];
      if (a.g_cpd != nullptr) g_dp = mie_ld(a.g_cpd, ho);
    } else if constexpr (GRU) {
      r0[0] = *reinterpret_cast<const float4*>(a.res + ho);
      add[0] = *reinterpret_cast<const float4*>(a.g_cres + ho);
    } else {
      const bool oks[1] = {true};
      conv_epilogue_load4<T, 1>(a, offs, oks, r0, add);
    }
    mie_mask_asked();
    ok1 = mie_mask_take(a.xm, b1, inb);
    ok2 = mie_mask_take(x2m, b2, a.x2 != nullptr ? inb : 0u);
  }

  // ---- contraction
  v4acc acc[MB], sm[MB], sl[MB];      // fp32: products of 1, 2^-8 and 2^-16 of the largest; F2: of 1 and 2^-11, and the totals' small part
  v4acc tot[F2 ? MB : 1];
  float c0 = 1.f, filt_unscale = 1.f;
  bool unfit = false;
  const long long weights = (long long)a.cin_total * (K * K) * cout;
  if constexpr (F2) {
    const float* const end = f2_filter_end(a.filt_mc, weights);
    filt_unscale = end[0];
    unfit = end[1] != 1.f;
#pragma unroll
    for (int b = 0; b < MB; ++b) tot[b] = v4acc{0.f, 0.f, 0.f, 0.f};
  }
#pragma unroll
  for (int b = 0; b < MB; ++b) acc[b] = v4acc{0.f, 0.f, 0.f, 0.f}, sm[b] = sl[b] = v4acc{0.f, 0.f, 0.f, 0.f};
  const mie_bf16* const x_lane = win + cg * (PL * STAGE) + (l16 >> 3) * S * RP + (l16 & 7) * S * LS + EPS * kg;
  auto chunk = [&](const char* next, auto more) {
    constexpr bool MORE = decltype(more)::value;
#pragma unroll
    for (int i = 0; i < NT; ++i) {
      const int tap = tc + TPC * i;
      if (TPC == 1 || TPC * i + TPC <= K * K || tap < K * K) {
        const int ky = tap / K, kx = tap - ky * K;
        float4 xv[MB][PL];
#pragma unroll
        for (int b = 0; b < MB; ++b)
#pragma unroll
          for (int q = 0; q < PL; ++q) xv[b][q] = *reinterpret_cast<const float4*>(x_lane + q * STAGE + (2 * S * b + ky) * RP + kx * LS);
        if constexpr (F2) {
#pragma unroll
          for (int b = 0; b < MB; ++b) mma16_f16(acc[b], w[i][0], xv[b][0]);
#pragma unroll
          for (int b = 0; b < MB; ++b) mma16_f16(sm[b], w[i][0], xv[b][1]);
#pragma unroll
          for (int b = 0; b < MB; ++b) mma16_f16(sm[b], w[i][1], xv[b][0]);
          if (i % DEEP_BL == DEEP_BL - 1 || i == NT - 1) {
#pragma unroll
            for (int b = 0; b < MB; ++b) deep_fold(tot[b], sl[b], acc[b], c0);
          }
        } else if constexpr (X3) {
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
      if constexpr (MORE) load_w(next, i, std::false_type());
    }
    if constexpr (F2) {      // (the rest of a wave whose last tap is none; the small products at this chunk's scale)
      const float c1 = c0 * (1.f / F2_STEP);
#pragma unroll
      for (int b = 0; b < MB; ++b) {
        if (TPC > 1) deep_fold(tot[b], sl[b], acc[b], c0);
#pragma unroll
        for (int r = 0; r < 4; ++r) sl[b][r] = fmaf(sm[b][r], c1, sl[b][r]), sm[b][r] = 0.f;
      }
    }
  };
  int unfit_pass = unfit ? 0 : nch;      // F2: the first pass that does not fit
  for (int pass = 0, c = cg; pass * NCW < nch; ++pass, c += NCW) {
    if (!OWN && pass > 0) __syncthreads();
    store_x(pass, std::true_type());
    if constexpr (F2) {
      if constexpr (OWN) unfit_pass = __ballot(groups.misfit()) != 0ull && pass < unfit_pass ? pass : unfit_pass;
      else if (groups.misfit()) s_f2[DEEP_WAVES + (pass & 1)] = 1.f;
      c0 = f2_unscale(groups.scale) * filt_unscale;
    }
    if constexpr (OWN) mie_wave_order();
    else __syncthreads();
    if constexpr (F2) {
      if (!OWN && __builtin_amdgcn_readfirstlane(__float_as_int(s_f2[F2 && !OWN ? DEEP_WAVES + (pass & 1) : 0])) != 0) unfit_pass = pass < unfit_pass ? pass : unfit_pass;
      if (__builtin_expect(unfit_pass <= pass, 0)) break;
    }
    if ((pass + 1) * NCW < nch) load_x(pass + 1);
    if (c + NCW < nch) chunk(chunk_w(c + NCW), std::true_type());
    else if (c < nch) chunk(nullptr, std::false_type());
    if constexpr (OWN) mie_wave_order();
  }
  if constexpr (F2) {
    // from the first pass on that does not fit, of the wave (OWN) or the workgroup: on the fp32 instruction from the fp32 copy of the filter behind
    // the terms (512->512 at 16x16 10.7 us, no pass fits 19; at 8x8 7.9 and 12.1)
    if (__builtin_expect(unfit_pass < nch, 0)) {
      for (int pass = __builtin_amdgcn_readfirstlane(unfit_pass), c = cg + NCW * pass; pass * NCW < nch; ++pass, c += NCW) {
        load_x(pass);
        if (c < nch)
#pragma unroll
          for (int i = 0; i < NT; ++i) load_w(chunk_w(c) + 4 * weights, i, std::false_type());
        if constexpr (OWN) mie_wave_order();
        else __syncthreads();
        store_x(pass, std::false_type());
        if constexpr (OWN) mie_wave_order();
        else __syncthreads();
        if (c >= nch) continue;
#pragma unroll
        for (int i = 0; i < NT; ++i) {
          const int tap = tc + TPC * i;
          if (TPC == 1 || TPC * i + TPC <= K * K || tap < K * K) {
            const int ky = tap / K, kx = tap - ky * K;
#pragma unroll
            for (int q = 0; q < PL; ++q)
#pragma unroll
              for (int b = 0; b < MB; ++b) mma16_f32(tot[b], w[i][q], *reinterpret_cast<const float4*>(x_lane + q * STAGE + (2 * S * b + ky) * RP + kx * LS));
            __builtin_amdgcn_sched_barrier(0);
          }
        }
      }
      if constexpr (OWN) mie_wave_order();
    }
  }
  if constexpr (!OWN) __syncthreads();

  // ---- the waves' sums meet in LDS: pixel 16 * b + l16, channels 4 * kg ...
#pragma unroll
  for (int b = 0; b < MB; ++b) {
    const v4acc s = F2 ? tot[b < (F2 ? MB : 1) ? b : 0] + sl[b] : acc[b] + (sm[b] + sl[b]);
    *reinterpret_cast<float4*>(park + wave * D::PARK + (16 * b + l16) * OS + 4 * kg) = make_float4(s[0], s[1], s[2], s[3]);
  }
  __syncthreads();
  if (!mine || idle) return;
  float4 part[DEEP_WAVES];
#pragma unroll
  for (int k = 0; k < DEEP_WAVES; ++k) part[k] = *reinterpret_cast<const float4*>(park + k * D::PARK + (it >> 2) * OS + 4 * (it & 3));
#pragma unroll
  for (int k = 1; k < DEEP_WAVES; ++k) {
    part[0].x += part[k].x; part[0].y += part[k].y; part[0].z += part[k].z; part[0].w += part[k].w;
  }
  const bool on = mie_mask_take(live_m, live_b, 1u) != 0u;
  if constexpr (GRU) {
    float4 dc = *reinterpret_cast<const float4*>(park + (it >> 2) * OS + 4 * (it & 3) + 4);
#pragma unroll
    for (int k = 1; k < DEEP_WAVES; ++k) {
      const float4 v = *reinterpret_cast<const float4*>(park + k * D::PARK + (it >> 2) * OS + 4 * (it & 3) + 4);
      dc.x += v.x; dc.y += v.y; dc.z += v.z; dc.w += v.w;
    }
    float4 h = make_float4(0.f, 0.f, 0.f, 0.f);
    if (on) {
      h = mie_gru_gates4(r0[0], add[0], part[0], dc);
      *reinterpret_cast<float4*>(a.res + ho) = r0[0];
      *reinterpret_cast<float4*>(a.g_cres + ho) = add[0];
    }
    mie_st4(a.g_dh, ho, h);
  } else if constexpr (GATES) {
    const bool has_cp = a.g_cpd != nullptr && mie_mask_take(cp_m, cp_b, 1u) != 0u;
    float dh = 0.f, dc = 0.f;
    if (on) {
      mie_lstm_gate_chain(r0[0].x, r0[0].y, r0[0].z, r0[0].w, part[0].x, part[0].y, part[0].z, part[0].w, g_cp, has_cp ? g_dp : 0.f, g_cc,
                          dh, dc);
      *reinterpret_cast<float4*>(a.res + off) = r0[0];
      if (has_cp) a.g_cpres[ho] = g_cp;
      a.g_cres[ho] = g_cc;
    }
    mie_st(a.g_dh, ho, dh);
    mie_st(a.g_dc, ho, dc);
  } else {
    const float4 sums[1] = {part[0]};
    const bool live[1] = {on};
    const bool oks[1] = {!AGAIN || finite4(part[0])};
    conv_epilogue_store4<T, 1>(a, offs, cos, oks, sums, r0, add, live);
    if constexpr (AGAIN) {
      if (__builtin_expect(__ballot(!oks[0]) != 0ull, 0))
        if (!oks[0]) conv_quad_again<T, K, S>(conv_args_again<T>(), n, oy, ox, co);
    }
  }
}

// Two terms for MIE_DTYPE_F32_F16X2: 3x3 convs of this many input channels and more.  Their error hardly grows with the channels (1.14 .. 1.19e-7
// of the output against fp64; a third as many sums between folds would make it 1.05 .. 1.09e-7, and a chunk 7 % longer), that of three
// terms does: 256 channels 1.07e-7, 512 1.43e-7.  us: 512->512 at 16x16 12.8 -> 11.1, at 8x8 9.0 -> 8.3, gates of 256+256 at 16x16 22.3 -> 19.7, of a
// ConvGRU of 512 there 22.6 -> 20.3.  (Below: 256->256 at 8x12 6.7 and 6.1, 64->64 at 32x32 4.0 and 4.4; stride 2 of 128 channels at
// 16x24 8.2 and 9.4, whose waves share their pixels and meet once more over the scale.)
constexpr int DEEP_F2_FROM = 512;

template <typename T, int K, int S, int NCW, int ROWS, int KIND>
void launch_form(const ConvArgsT<T>& a, unsigned cap, hipStream_t st) {
  const dim3 grid(a.cout / DEEP_COLS, 8 / ROWS * cap);
  if constexpr (sizeof(T) == 4 && K == 3 && S == 1 && KIND != DEEP_UP) {
    if (a.x3 == 2 && a.c1 + a.c2 >= DEEP_F2_FROM) {
      hipLaunchKernelGGL((k_conv_deep<T, 2, K, S, NCW, ROWS, KIND>), grid, dim3(DEEP_THREADS), 0, st, f2_args(a, K));
      return;
    }
  }
  hipLaunchKernelGGL((k_conv_deep<T, sizeof(T) == 4 ? 1 : 0, K, S, NCW, ROWS, KIND>), grid, dim3(DEEP_THREADS), 0, st, a);
}

// Chunks in LDS at a time.
template <typename T, int K, int S, int ROWS, int KIND>
void launch_chunks(const ConvArgsT<T>& a, unsigned cap, hipStream_t st) {
  const int nch = (a.c1 + (KIND == DEEP_UP ? 0 : a.c2)) / 32;
  if constexpr (KIND == DEEP_UP) {
    if constexpr (sizeof(T) == 4) launch_form<T, K, S, 1, ROWS, KIND>(a, cap, st);
    else if (ROWS < 8 && nch >= 4) launch_form<T, K, S, 4, ROWS < 8 ? ROWS : 4, KIND>(a, cap, st);
    else launch_form<T, K, S, 2, ROWS, KIND>(a, cap, st);
  } else if constexpr (S == 2 && K == 3) {
    // (fp32 128->256 at 16x16 with 1, 2, 4: 6.7, 6.1, 6.4 us, 256->512 13.8, 12.0, 12.0; bf16 4.9, 4.7, 4.3 and 7.3, 6.5, 6.1)
    if (sizeof(T) == 4 || nch < 4) launch_form<T, K, S, 2, ROWS, KIND>(a, cap, st);
    else launch_form<T, K, S, sizeof(T) == 4 ? 2 : 4, ROWS, KIND>(a, cap, st);
  } else if constexpr (S == 2) {
    launch_form<T, K, S, 1, ROWS, KIND>(a, cap, st);
  } else {
    if (ROWS < 8 && nch >= 8) launch_form<T, K, S, 8, ROWS < 8 ? ROWS : 4, KIND>(a, cap, st);
    else if (nch > 2) launch_form<T, K, S, 4, ROWS, KIND>(a, cap, st);
    else launch_form<T, K, S, 2, ROWS, KIND>(a, cap, st);
  }
}

// ---- the stride-2 transposed conv (3x3, pad 1, the output twice the input; phases and block tile set as in mie_tconv_mfma.hip) ----
// A workgroup takes ROWS x 8 input positions of a block, i.e. 2 * ROWS x 16 output pixels, times 16 columns; each of the waves a
// chunk of 32 channels in eight, which it stages itself, all nine taps: a tap's phase is then known at compile time, and a staged
// pixel is read once for each of the four shifts instead of for nine taps.  Bound by the serial trips and by the filter, which
// every workgroup of a slab fetches for itself.  In place of a split launch and its finish, us per layer (graph of 24, filters cold):
//                                   fp32             bf16
//   256+256->256 from 16x16      16.4 -> 10.4     13.5 -> 5.2
//   128+128->128 from 32x32      16.1 -> 9.0      13.4 -> 6.2
//   128+128->64 from 64x64       20.7 -> 17.0     14.9 -> 10.4   (two rounds of the chip)
// Whole pass of optical flow, 1x256x256 fp32, transposed decoder: 334.0 -> 314.3 us, with the two-round shapes 312.1.
template <typename T, int ROWS>
__global__ __launch_bounds__(DEEP_THREADS) void k_tconv_deep(ConvArgsT<T> a, TileSetDev pts) {
  constexpr bool X3 = sizeof(T) == 4;
  constexpr int PL = X3 ? 3 : 1, GPS = X3 ? 2 : 1, CC = 32, EPS = 8, LS = CC + EPS;
  constexpr int WX = 9, WY = ROWS + 1, NPIX = WX * WY, RP = row_pitch_dw(WX, LS / 2, 1) * 2, STAGE = WY * RP;
  constexpr int SPP = CC / EPS, STEP = 64 / SPP, NLD = (NPIX + STEP - 1) / STEP, MB = ROWS / 2, OS = DEEP_COLS + 4;
  constexpr int SUMS = 4 * ROWS * 8 * OS, OWN = PL * STAGE / 2 > SUMS ? PL * STAGE / 2 : SUMS;      // floats of a wave: its pixels, then its sums
  constexpr int ITEMS = 4 * ROWS * 8 * (DEEP_COLS / 4);
  static_assert(OWN * 4 * DEEP_WAVES <= 160 * 1024 && ITEMS <= DEEP_THREADS && OWN % 4 == 0, "LDS of a CU, an item a thread");
  __shared__ __attribute__((aligned(16))) float smem[OWN * DEEP_WAVES];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int kg = lane >> 4, l16 = lane & 15;
  mie_bf16* const win = reinterpret_cast<mie_bf16*>(smem + wave * OWN);
  const int slabs = a.cout / DEEP_COLS, bx = blockIdx.y;
  int by = blockIdx.x + conv_args_entry_zero(a);
  if ((slabs & 7) == 0) by = (by & 7) * (slabs >> 3) + (by >> 3);      // (as in k_conv_deep)
  const int co0 = by * DEEP_COLS, cout = a.cout;
  const int nch1 = a.c1 / CC, nch = nch1 + (a.x2 != nullptr ? a.c2 / CC : 0);

  const unsigned w_step = 2u * cout * (2 * EPS);
  const unsigned w_lane = (((kg >> 1) * (9 * PL * 2) + (kg & 1)) * cout + co0 + l16) * (2 * EPS);
  auto chunk_w = [&](int c) -> const char* { return reinterpret_cast<const char*>(a.filt_mc) + (long long)(c * (CC / 16)) * 9 * PL * w_step; };
  // Taps in the order of their shifts (a direction's tap 0: phase 1 from the next pixel, 1: phase 0, 2: phase 1).  fp32 of four rows
  // has registers for RING of them beside its sums (with all nine it kept 130 in scratch memory).
  constexpr int RING = X3 && ROWS == 4 ? 3 : 9;
  constexpr int TAPS[9] = {0, 1, 2, 3, 6, 4, 5, 7, 8};
  float4 w[RING][PL];
  auto load_w = [&](const char* p, int j, auto first) {      // (first chunk, later ones: as in k_conv_deep)
#pragma unroll
    for (int q = 0; q < PL; ++q) {
      if constexpr (decltype(first)::value) {
        w[j % RING][q] = *reinterpret_cast<const float4*>(p + (w_lane + (TAPS[j] * PL + q) * w_step));
      } else {
        GlobalBytes t = (GlobalBytes)p + (TAPS[j] * PL + q) * w_step;
        asm("" : "+s"(t));
        w[j % RING][q] = global_ld4(t + w_lane);
      }
    }
  };
  const int pos = bx / (8 / ROWS);
  TileAsk ask = mie_tile_ask(pts, pos);
  __builtin_amdgcn_sched_barrier(0);
  {
    const char* p = chunk_w(wave < nch ? wave : 0);
#pragma unroll
    for (int i = 0; i < RING; ++i) load_w(p, i, std::true_type());
  }
  int n, y0, x0;      // in input pixels
  const int tk = mie_tile_take(pts, pos, ask, n, y0, x0);
  y0 += ROWS * (bx % (8 / ROWS));
  const int hout = a.ts.h, wout = a.ts.w;
  if (tk == 0 || y0 >= a.h_in) return;

  // the output of this thread: pixel it >> 2 of the 2 * ROWS x 16, channels 4 * (it & 3) ... of the slab
  const int it = tid & (ITEMS - 1), ly = it >> 6, lx = (it >> 2) & 15;
  const int oy = 2 * y0 + ly, ox = 2 * x0 + lx, co = co0 + 4 * (it & 3);
  const bool in = oy < hout && ox < wout, mine = tid < ITEMS && in;
  const int opix = in ? (n * hout + oy) * wout + ox : 0;
  const long long off = (long long)opix * cout + co;
  if (tk == 2) {
    if (mine) mie_st4(a.out, off, make_float4(0.f, 0.f, 0.f, 0.f));
    return;
  }

  const int q8 = EPS * (lane % SPP), p0 = lane / SPP;
  int st_po[NLD];
  unsigned inb = 0u;
#pragma unroll
  for (int i = 0; i < NLD; ++i) {
    const int pix = p0 + STEP * i, py = pix / WX, iy = y0 + py, ix = x0 + pix - py * WX;
    const bool k = pix < NPIX && iy < a.h_in && ix < a.w_in;
    st_po[i] = k ? (n * a.h_in + iy) * a.w_in + ix : 0;
    inb |= (k ? 1u : 0u) << i;
  }
  float4 xr[NLD][GPS];
  auto load_x = [&](int c) {
    if (c >= nch) c = 0;
    const bool second = c >= nch1;
    const T* p = second ? a.x2 : a.x;
    const int cs = second ? a.c2 : a.c1, ci0 = (second ? c - nch1 : c) * CC + q8;
#pragma unroll
    for (int i = 0; i < NLD; ++i)
#pragma unroll
      for (int g = 0; g < GPS; ++g) xr[i][g] = *reinterpret_cast<const float4*>(p + (long long)st_po[i] * cs + ci0 + 4 * g);
  };
  auto kept = [](const float4& v, bool k) { return make_float4(k ? v.x : 0.f, k ? v.y : 0.f, k ? v.z : 0.f, k ? v.w : 0.f); };
  const uint8_t* const live_m = a.refresh ? nullptr : a.ts.pixmask;
  const uint8_t* const x2m = a.x2 != nullptr ? a.x2m : nullptr;
  const long long offs[1] = {off};
  const int cos[1] = {co}, at[1] = {opix};
  const bool oks[1] = {true};
  float4 r0[1], add[1];
  unsigned live_b[1], ok1, ok2;
  {
    unsigned b1[NLD], b2[NLD];
    load_x(wave);
    mie_mask_ask(a.xm, a.filt_mc, st_po, b1);
    mie_mask_ask(x2m, a.filt_mc, st_po, b2);
    mie_mask_ask(live_m, a.filt_mc, at, live_b);
    conv_epilogue_load4<T, 1>(a, offs, oks, r0, add);
    mie_mask_asked();
    ok1 = mie_mask_take(a.xm, b1, inb);
    ok2 = mie_mask_take(x2m, b2, a.x2 != nullptr ? inb : 0u);
  }
  auto store_x = [&](int c) {
    const unsigned ok = c >= nch1 ? ok2 : ok1;
#pragma unroll
    for (int i = 0; i < NLD; ++i) {
      const int pix = p0 + STEP * i, py = pix / WX;
      if (STEP * i + STEP > NPIX && pix >= NPIX) continue;
      const bool k = (ok >> i) & 1u;
      mie_bf16* const d = win + py * RP + (pix - py * WX) * LS + q8;
      const float4 u = kept(xr[i][0], k);
      if constexpr (X3) {
        const float4 v = kept(xr[i][GPS - 1], k);
        const float f[8] = {u.x, u.y, u.z, u.w, v.x, v.y, v.z, v.w};
        float4 pl[3];
        split3(f, pl);
#pragma unroll
        for (int q = 0; q < PL; ++q) *reinterpret_cast<float4*>(d + q * STAGE) = pl[q];
      } else {
        *reinterpret_cast<float4*>(d) = u;
      }
    }
  };

  v4acc acc[4][MB], sm[X3 ? 4 : 1][MB];      // by phase; fp32: products of the first terms, and the smaller ones
#pragma unroll
  for (int b = 0; b < MB; ++b) {
#pragma unroll
    for (int ph = 0; ph < 4; ++ph) acc[ph][b] = v4acc{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int ph = 0; ph < (X3 ? 4 : 1); ++ph) sm[ph][b] = v4acc{0.f, 0.f, 0.f, 0.f};
  }
  const mie_bf16* const x_lane = win + (l16 >> 3) * RP + (l16 & 7) * LS + EPS * kg;
  auto chunk = [&](const char* cur, const char* next, auto more) {
    float4 xv[MB][PL];
#pragma unroll
    for (int j = 0; j < 9; ++j) {
      const int ky = TAPS[j] / 3, kx = TAPS[j] % 3, ph = (ky == 1 ? 0 : 2) + (kx == 1 ? 0 : 1);
      if (j == 0 || j == 1 || j == 3 || j == 5) {      // another shift
#pragma unroll
        for (int b = 0; b < MB; ++b)
#pragma unroll
          for (int q = 0; q < PL; ++q)
            xv[b][q] = *reinterpret_cast<const float4*>(x_lane + q * STAGE + (2 * b + (ky == 0)) * RP + (kx == 0) * LS);
      }
      if constexpr (X3) {
        auto term = [&](v4acc (&t)[MB], int tw, int tx) {
#pragma unroll
          for (int b = 0; b < MB; ++b) mma16(t[b], w[j % RING][tw], xv[b][tx]);
        };
        term(sm[ph], 0, 2); term(acc[ph], 0, 0); term(sm[ph], 1, 1);
        term(sm[ph], 2, 0); term(sm[ph], 0, 1); term(sm[ph], 1, 0);
      } else {
#pragma unroll
        for (int b = 0; b < MB; ++b) mma16(acc[ph][b], w[j % RING][0], xv[b][0]);
      }
      if (RING < 9 && j + RING < 9) load_w(cur, j + RING, std::false_type());
      else if (decltype(more)::value) load_w(next, (j + RING) % 9, std::false_type());
      if constexpr (RING < 9) __builtin_amdgcn_sched_barrier(0);
    }
  };
  for (int c = wave; c < nch; c += DEEP_WAVES) {
    store_x(c);
    mie_wave_order();
    if (RING < 9 || c + DEEP_WAVES < nch) {      // (RING < 9: the chunk after the last is the first again, one form of the loop)
      load_x(c + DEEP_WAVES);
      chunk(chunk_w(c), chunk_w(c + DEEP_WAVES < nch ? c + DEEP_WAVES : 0), std::true_type());
    } else {
      chunk(chunk_w(c), nullptr, std::false_type());
    }
    mie_wave_order();
  }

  // ---- two more input channels (a.g_cpd with its mask a.g_cpm, plain filter rows a.g_cpres), in fp32: an output pixel sees the one, two or
  // four taps of its phase.  Asked for here, where the filter's registers are free, and added behind the sums.  (As a launch of their
  // own and an addend, optical flow with transposed decoders, two such layers: 312.4 -> 304.9 us a pass, a third in k_tconv_mfma -> 300.3.)
  float2 lx2[4];
  float4 lf[4][2];
  unsigned lead_b[4], lead_in = 0u;
  const bool lead = a.g_cpd != nullptr;
  if (lead) {
    int lat[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int r = q >> 1, c = q & 1, iy = y0 + (ly >> 1) + r, ix = x0 + (lx >> 1) + c;
      const bool k = in && (r == 0 || (ly & 1)) && (c == 0 || (lx & 1)) && iy < a.h_in && ix < a.w_in;
      const int ky = r != 0 ? 0 : (ly & 1) ? 2 : 1, kx = c != 0 ? 0 : (lx & 1) ? 2 : 1;
      lat[q] = k ? (n * a.h_in + iy) * a.w_in + ix : 0;
      lead_in |= (k ? 1u : 0u) << q;
      if constexpr (X3) {
        lx2[q] = *reinterpret_cast<const float2*>(a.g_cpd + 2LL * lat[q]);
      } else {
        const uint32_t v = *reinterpret_cast<const uint32_t*>(a.g_cpd + 2LL * lat[q]);
        lx2[q] = make_float2(__uint_as_float(v << 16), __uint_as_float(v & 0xffff0000u));
      }
#pragma unroll
      for (int i = 0; i < 2; ++i) lf[q][i] = *reinterpret_cast<const float4*>(a.g_cpres + (long long)(9 * i + 3 * ky + kx) * cout + co);
    }
    mie_mask_ask(a.g_cpm, a.filt_mc, lat, lead_b);
  }

  // ---- the waves' sums meet in LDS: phase, position 16 * b + l16, channels 4 * kg ... (each where its own pixels were)
#pragma unroll
  for (int ph = 0; ph < 4; ++ph)
#pragma unroll
    for (int b = 0; b < MB; ++b) {
      v4acc s = acc[ph][b];
      if constexpr (X3) s += sm[ph][b];
      *reinterpret_cast<float4*>(smem + wave * OWN + ((ph * MB + b) * 16 + l16) * OS + 4 * kg) = make_float4(s[0], s[1], s[2], s[3]);
    }
  __syncthreads();
  if (!mine) return;
  const int from = ((2 * (ly & 1) + (lx & 1)) * (ROWS * 8) + (ly >> 1) * 8 + (lx >> 1)) * OS + 4 * (it & 3);
  float4 part[DEEP_WAVES];
#pragma unroll
  for (int k = 0; k < DEEP_WAVES; ++k) part[k] = *reinterpret_cast<const float4*>(smem + k * OWN + from);
#pragma unroll
  for (int k = 1; k < DEEP_WAVES; ++k) {
    part[0].x += part[k].x; part[0].y += part[k].y; part[0].z += part[k].z; part[0].w += part[k].w;
  }
  if (lead) {
    const unsigned k = mie_mask_take(a.g_cpm, lead_b, lead_in);
    float4 s = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const float u = (k >> q) & 1u ? lx2[q].x : 0.f, v = (k >> q) & 1u ? lx2[q].y : 0.f;
      s.x += u * lf[q][0].x + v * lf[q][1].x; s.y += u * lf[q][0].y + v * lf[q][1].y;
      s.z += u * lf[q][0].z + v * lf[q][1].z; s.w += u * lf[q][0].w + v * lf[q][1].w;
    }
    part[0].x += s.x; part[0].y += s.y; part[0].z += s.z; part[0].w += s.w;
  }
  const float4 sums[1] = {part[0]};
  const bool live[1] = {mie_mask_take(live_m, live_b, 1u) != 0u};
  conv_epilogue_store4<T, 1>(a, offs, cos, oks, sums, r0, add, live);
}

long long deep_slabs(long long tiles, int cout) { return tiles * (cout / DEEP_COLS); }
int deep_rows(long long slabs) { return 4 * slabs <= DEEP_WGS ? 2 : 2 * slabs <= DEEP_WGS ? 4 : 8; }      // (launch_deep)
template <typename T>
int deep_dtype(const ConvArgsT<T>& a) { return sizeof(T) == 2 ? MIE_DTYPE_BF16 : a.x3 ? MIE_DTYPE_F32_BF16X3 : MIE_DTYPE_F32; }

// Two rows of input positions a workgroup while that is one round of the chip, else four: in one round or in two (fp32 and bf16, two
// rounds against the split form: 512->256 from 24x32 24.3 -> 21.4 and 14.9 -> 10.4 us, 64+64->64 from 64x64 16.8 -> 12.6 and 12.1 -> 9.2).
template <typename T>
bool deep_tconv(const ConvArgsT<T>& a, const TileSetDev& pts, hipStream_t st) {
  const long long cap = (long long)pts.n * pts.tiles_y * pts.tiles_x, slabs = deep_slabs(cap, a.cout);
  if ((sizeof(T) == 4 && !a.x3) || a.c1 % 32 != 0 || a.c2 % 32 != 0 || a.c1 + a.c2 < 128 || a.cout % DEEP_COLS != 0 || slabs > DEEP_WGS) return false;
  if (4 * slabs <= DEEP_WGS)
    hipLaunchKernelGGL((k_tconv_deep<T, 2>), dim3(a.cout / DEEP_COLS, 4 * (unsigned)cap), dim3(DEEP_THREADS), 0, st, a, pts);
  else
    hipLaunchKernelGGL((k_tconv_deep<T, 4>), dim3(a.cout / DEEP_COLS, 2 * (unsigned)cap), dim3(DEEP_THREADS), 0, st, a, pts);
  return true;
}

// Workgroups of whole tiles.  The form is taken while they are one round of the chip, one a CU, and with as few rows as keep it that: two
// beat four and these eight while there are CUs for them (fp32 256->256 at 8x12 7.4, 8.8, 11.7 us, bf16 5.2, 5.5, 6.6), and a second
// round costs more than anything (at 16x24, 96 slabs: four rows 9.3, two 11.2; at 33x44, 480 slabs: 24.7 us, k_conv_mfma 20.7; a gates conv
// of 64 channels at 32x48, 384: 12.1 and 8.9; 5x5 64->128 at 48x48, 288: 19.5 and 16.1).
template <typename T, int K, int S, int KIND>
void launch_deep(const ConvArgsT<T>& a, unsigned cap, hipStream_t st) {
  const int rows = deep_rows(deep_slabs(cap, a.cout));
  if (rows == 2) launch_chunks<T, K, S, 2, KIND>(a, cap, st);
  else if (rows == 4) launch_chunks<T, K, S, 4, KIND>(a, cap, st);
  else if constexpr (!(sizeof(T) == 4 && KIND == DEEP_UP)) launch_chunks<T, K, S, 8, KIND>(a, cap, st);      // (mie_upconv_deep_form: not fp32)
}

template <typename T>
bool deep_plain(const ConvArgsT<T>& a, int k, int s, unsigned cap, hipStream_t st) {
  if (a.ws != nullptr || !mie_conv_deep_form(k, s, a.c1, a.c2, a.cout, cap, deep_dtype(a))) return false;
  if (k == 5) launch_deep<T, 5, 2, DEEP_PLAIN>(a, cap, st);
  else if (s == 2) launch_deep<T, 3, 2, DEEP_PLAIN>(a, cap, st);
  else launch_deep<T, 3, 1, DEEP_PLAIN>(a, cap, st);
  return true;
}
template <typename T>
bool deep_gates(const ConvArgsT<T>& a, unsigned cap, hipStream_t st) {
  if (a.ws != nullptr || a.cout != 4 * a.hid || !mie_conv_deep_form(3, 1, a.c1, a.c2, a.cout, cap, deep_dtype(a))) return false;
  launch_deep<T, 3, 1, DEEP_GATES>(a, cap, st);
  return true;
}
template <typename T>
bool deep_gru(const ConvArgsT<T>& a, unsigned cap, hipStream_t st) {
  if (a.cout != 2 * a.hid || !mie_conv_deep_form(3, 1, a.c1, a.c2, a.cout, cap, deep_dtype(a))) return false;
  launch_deep<T, 3, 1, DEEP_GRU>(a, cap, st);
  return true;
}
template <typename T>
bool deep_up(const ConvArgsT<T>& a, unsigned cap, hipStream_t st) {
  if (a.ws != nullptr || !mie_upconv_deep_form(a.c1, a.cout, cap, deep_dtype(a))) return false;
  launch_deep<T, 5, 1, DEEP_UP>(a, cap, st);
  return true;
}

}  // namespace

bool mie_conv_deep_form(int k, int s, int c1, int c2, int cout, long long tiles, int dtype) {
  if (dtype == MIE_DTYPE_F32_F16X2) dtype = MIE_DTYPE_F32_BF16X3;      // (what this form multiplies for it)
  if (c1 <= 0 || c2 < 0 || cout <= 0 || tiles <= 0) return false;
  if (!((k == 3 && (s == 1 || s == 2)) || (k == 5 && s == 2))) return false;
  // what comes to the matrix cores at all (the queries must not name other layers: they run on the VALU); 3x3 stride 2 in three terms
  // does in this form only
  if (dtype == MIE_DTYPE_BF16 ? !mie_conv_mfma_takes(k, s, dtype, c1, c2, cout)
                              : dtype != MIE_DTYPE_F32_BF16X3 || !((k == 3 && s == 2) || mie_conv_x3_takes(k, s, c1, c2, cout))) return false;
  if (c1 % 32 != 0 || c2 % 32 != 0 || c1 + c2 < (k == 3 ? 64 : 32) || cout % DEEP_COLS != 0) return false;
  // (fp32 of eight rows a workgroup splits its pixels into terms for 16 columns only, one pass of chunks behind the other: with more than
  // 512 channels the split form is faster.  512+512->512 at 16x32 39.1 us, 34.5 there, ->256 at 32x32 38.3, 34.6;
  // the other way 512->512 at 16x32 22.3 and 23.4, 256+256->256 at 32x32 21.4 and 22.4.  Optical flow, up-sampling decoder, 433.1 -> 428.2)
  if (dtype == MIE_DTYPE_F32_BF16X3 && k == 3 && s == 1 && 2 * deep_slabs(tiles, cout) > DEEP_WGS && c1 + c2 > 512) return false;
  return deep_slabs(tiles, cout) <= DEEP_WGS;
}
// (fp32 of eight rows a workgroup: 128->64 at 64x64 17.8 us, k_upconv2x 16.1)
bool mie_upconv_deep_form(int c, int cout, long long tiles, int dtype) {
  if (dtype == MIE_DTYPE_F32_F16X2) dtype = MIE_DTYPE_F32_BF16X3;
  if ((dtype != MIE_DTYPE_BF16 && dtype != MIE_DTYPE_F32_BF16X3) || c <= 0 || cout <= 0 || tiles <= 0) return false;
  if (c % (dtype == MIE_DTYPE_BF16 ? 64 : 32) != 0 || cout % 32 != 0) return false;      // (other layers are refused)
  return dtype == MIE_DTYPE_BF16 ? deep_slabs(tiles, cout) <= DEEP_WGS : 2 * deep_slabs(tiles, cout) <= DEEP_WGS && c <= 128;
}

// Whether the one-launch form is the faster one where the caller has a workspace for the split form.  A workgroup here has the
// whole contraction, a few chunks at a time, and takes as long as there are channels; the split form has an eighth of it behind a
// fixed cost of a second launch.  So the line is a number of input channels, and hardly depends on anything but the kind of
// layer, the type and the rows a workgroup (2, 4, 8: how many columns and tiles there are).  One launch over split, median of 5 to 20
// layers of other sizes and densities each, at the line and at the next count that was measured above it:
//                  fp32, two rows     four               eight              bf16, two           four                eight
//   3x3           512 .98, 640 1.05  576 .99, 640 1.03  256 .89, 320 1.05  1536 .97, 2048 1.2  1536 .91            1024 .96, 1280 1.04
//   3x3 s2        448 .98, 512 1.05  640 .98, 768 1.02  1024 .97, 1280 1.02  896 .99, 1024 1.08  896 .96, 1536 1.2  576 1.0, 704 1.06
//   5x5 s2        160 .96, 192 1.04  160 .91, 256 1.10  256 .98, 320 1.01  448 .99, 512 1.4    384 .98, 448 1.09   320 .92, 384 1.07
//   gates         640 .91, 768 1.02  1024 .93, 1536 1.07  512 .76          2048 .94, 2560 1.04  3072 .83           3072 .73
//   up            128 .84            128 .89            (none)             448 .97, 512 1.28   384 .87, 448 1.01   512 .99, 768 1.07
// (3x3 fp32 of eight rows: 384 and 512, which fill its passes of four chunks, .98 and 1.01; 448 1.05.)
// The fp32 lines are of three terms in both forms.  With MIE_DTYPE_F32_F16X2, whose split form runs in two, medians of four layers a cell: 3x3 of
// two rows 448 .99, 512 and more (in two terms here, too) .87 to 1.01, four 256 .89, 320 1.03, 448 1.04, 512 .89, eight 128 .85, 192 1.05, 256 1.01, 384 1.12,
// 512 1.15; 5x5 s2 160 .97, 128 .99 and 160 1.04, 96 .99, 128 1.07 and 256 1.25; gates 1024 .97, 1024 1.01, 256 .98, 512 1.04; up 128 .93.  So
// with it 5x5 s2 and 3x3 of eight rows would go to the split form earlier.  Far above it, 5x5 stride 2
// of 512 / 1024 channels: fp32 1.6 / 2.1, up to 2.9 times as long, bf16 1.4 / 2.0.
bool mie_conv_deep_faster(int k, int s, int c1, int c2, int cout, long long tiles, int dtype, bool gates) {
  if (!mie_conv_deep_form(k, s, c1, c2, cout, tiles, dtype)) return false;
  static const int most[4][2][3] = {{{512, 576, 256}, {1536, 1536, 1024}}, {{448, 640, 1024}, {896, 896, 576}}, {{160, 160, 256}, {448, 384, 320}},
                                    {{640, 1024, 512}, {2048, 3072, 3072}}};
  const int kind = gates ? 3 : k == 5 ? 2 : s - 1, bf = dtype == MIE_DTYPE_BF16 ? 1 : 0, rows = deep_rows(deep_slabs(tiles, cout)), c = c1 + c2;
  return c <= most[kind][bf][rows / 4] || (kind == 0 && bf == 0 && rows == 8 && c % 128 == 0);
}
bool mie_upconv_deep_faster(int c, int cout, long long tiles, int dtype) {
  if (!mie_upconv_deep_form(c, cout, tiles, dtype)) return false;
  static const int most[3] = {448, 384, 512};
  return dtype != MIE_DTYPE_BF16 || c <= most[deep_rows(deep_slabs(tiles, cout)) / 4];
}

bool mie_launch_conv_deep(const ConvArgsT<float>& a, int k, int s, unsigned cap, hipStream_t st) { return deep_plain(a, k, s, cap, st); }
bool mie_launch_conv_deep(const ConvArgsT<mie_bf16>& a, int k, int s, unsigned cap, hipStream_t st) { return deep_plain(a, k, s, cap, st); }
bool mie_launch_gates_deep(const ConvArgsT<float>& a, unsigned cap, hipStream_t st) { return deep_gates(a, cap, st); }
bool mie_launch_gates_deep(const ConvArgsT<mie_bf16>& a, unsigned cap, hipStream_t st) { return deep_gates(a, cap, st); }
bool mie_launch_gru_deep(const ConvArgsT<float>& a, unsigned cap, hipStream_t st) { return deep_gru(a, cap, st); }
bool mie_launch_gru_deep(const ConvArgsT<mie_bf16>& a, unsigned cap, hipStream_t st) { return deep_gru(a, cap, st); }
bool mie_launch_upconv_deep(const ConvArgsT<float>& a, unsigned cap, hipStream_t st) { return deep_up(a, cap, st); }
bool mie_launch_upconv_deep(const ConvArgsT<mie_bf16>& a, unsigned cap, hipStream_t st) { return deep_up(a, cap, st); }
bool mie_launch_tconv_deep(const ConvArgsT<float>& a, const TileSetDev& blocks, hipStream_t st) { return deep_tconv(a, blocks, st); }
bool mie_launch_tconv_deep(const ConvArgsT<mie_bf16>& a, const TileSetDev& blocks, hipStream_t st) { return deep_tconv(a, blocks, st); }
