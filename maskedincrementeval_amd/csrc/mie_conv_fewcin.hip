// Masked conv on the matrix cores for layers with very few input channels: the network heads (5 or 4
// event bins -> 32 / 64 channels, 5x5 or 3x3).  Their contraction, K*K*Cin = 36 .. 125, is too short for
// the staged implicit GEMM of mie_conv_mfma_impl.h (whole chunks of 32 channels, 16-byte channel slots),
// and on the VALU path they run at a tenth of the vector peak.  Here the whole problem of a workgroup
// fits LDS at once:
//   * one 256-thread workgroup = one active 8x8 output tile x 32 output channels;
//   * the input tile plus halo is staged in fp32, channels padded to 8 (pixel stride 9 floats), zeros for inactive
//     pixels (what is fetched of them is dropped); bf16 deltas are widened while staging, so one kernel body
//     (v_mfma_f32_32x32x2_f32) serves both element types -- products of bf16 values are exact in fp32;
//   * the filter slab [tap][8 channels][32 columns] is staged from the plain fp32 filter, zero rows for
//     the padding channels;
//   * k = (tap, channel pair); wave w multiplies the 32-pixel block w & 1 (tile rows 0-3 / 4-7) for the
//     taps of parity w >> 1, only the ceil(Cin / 2) channel pairs that exist; the two tap halves meet in
//     LDS and are added in a fixed order; epilogue as everywhere (addend, reservoir, activation, refresh).
// One input only (x2 unsupported), stride 1 or 2, K = 3 or 5, Cout % 32 == 0.
// UP: the input is up2x(x), the bilinear x2 up-sampling of a delta given at half resolution (a.h_in / a.w_in are
// the up-sampled size): the source pixels are staged first and every staged pixel is blended from four of them, the
// up-sampled tensor is never formed (the 2-channel flow estimate in front of an EVFlowNet decoder).  Stride 1 only.
#include "mie_conv.h"

namespace {

typedef float v16f __attribute__((ext_vector_type(16)));

constexpr int FC_CH = 8;     // staged channels per pixel
constexpr int FC_PS = 9;     // LDS floats per staged pixel (odd: the 32 pixels of a block fall on distinct banks)

// Waves a SIMD: as many workgroups a CU as the LDS has room for (3x3 at stride 2: as many as without spills).  Without a bound the
// compiler gives the accumulators registers of their own and a CU holds one to four fewer: 8x480x640, every pixel active, 4->64
// 3x3 stride 2 139 -> 128 us, 5->32 5x5 stride 2 125 -> 115, 4->32 3x3 205 -> 189.
constexpr int fc_waves(int k, int s, bool up) { return k == 3 ? (s == 2 ? 5 : 8) : s == 2 ? 4 : up ? 5 : 1; }

template <typename T, int K, int S, bool UP = false>
__global__ __launch_bounds__(256, fc_waves(K, S, UP)) void k_conv_fewcin(ConvArgsT<T> a) {
  static_assert(!UP || S == 1, "the up-sampling form is stride 1");
  constexpr int IT = 7 * S + K;                  // input tile edge incl. halo
  constexpr int NPIX = IT * IT;
  constexpr int IN_F = NPIX * FC_PS;
  constexpr int W_F = K * K * FC_CH * 32;
  constexpr int RED_F = 2 * 64 * 32;             // the accumulators of the two tap halves, parked for the epilogue
  constexpr int NIN = (NPIX * FC_CH + 255) / 256;
  constexpr int LO = UP ? (K == 5 ? 8 : 6) : IT; // edge of what is loaded: source pixels, or the staged ones themselves
  constexpr int NLD = (LO * LO * FC_CH + 255) / 256;
  constexpr int SMEM_F = (IN_F + W_F > RED_F) ? IN_F + W_F : RED_F;      // (they reuse the staging area)
  // the source pixels lie behind the filter, or (5x5, five workgroups a CU) where its last taps go afterwards
  constexpr int LATE = UP && IN_F + W_F + LO * LO * FC_PS > SMEM_F ? 3 : 0;
  constexpr int LO_AT = IN_F + W_F - LATE * FC_CH * 32;
  static_assert(!UP || LO_AT + LO * LO * FC_PS <= SMEM_F, "room for the source pixels");
  __shared__ float smem[SMEM_F];
  float* const s_in = smem;
  float* const s_w = smem + IN_F;

  int n, y0, x0;
  const int tk = mie_pick_tile(a.ts, blockIdx.x + conv_args_entry_zero(a), n, y0, x0);
  if (tk == 0) return;
  const int tid = threadIdx.x;
  const int hout = a.ts.h, wout = a.ts.w, cout = a.cout, cin = a.c1;
  const int co0 = blockIdx.y * 32;
  if (tk == 2) {   // stale tile: zero this workgroup's channel slab
    for (int idx = tid; idx < 64 * 8; idx += 256) {        // groups of four channels
      const int p = idx >> 3, col = 4 * (idx & 7);
      const int oy = y0 + (p >> 3), ox = x0 + (p & 7);
      if (oy < hout && ox < wout)
        mie_st4(a.out, (((long long)n * hout + oy) * wout + ox) * cout + co0 + col, make_float4(0.f, 0.f, 0.f, 0.f));
    }
    return;
  }

  // pixels of this thread's two epilogue groups that lie in the output pixel mask (elsewhere the sums are exactly
  // zero: no reservoir access, a zero delta); the bytes are asked for before the staging loads
  int live_at[2];
  unsigned live_in = 0u;
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int p = (tid + 256 * i) >> 3;
    const int oy = y0 + (p >> 3), ox = x0 + (p & 7);
    const bool k = oy < hout && ox < wout;
    live_at[i] = k ? (n * hout + oy) * wout + ox : 0;
    live_in |= (k ? 1u : 0u) << i;
  }
  const uint8_t* const live_m = a.refresh ? nullptr : a.ts.pixmask;
  unsigned live_b[2];
  mie_mask_ask(live_m, a.filt, live_at, live_b);

  // ---- stage the input tile (fp32, 8 channels per pixel) and the filter slab ---------------------
  // Every global load of the thread is issued before the first LDS store (compile-time trip counts, fully
  // unrolled): one memory round trip for the whole staging instead of one per loop iteration.
  const int iy0 = y0 * S - a.pad, ix0 = x0 * S - a.pad;
  float vw[K * K];
  {
    const int col = tid & 31, ch = (tid >> 5) & 7;           // filter: thread = (channel, column), one load per tap
    const float* wp = a.filt + (long long)ch * (K * K) * cout + co0 + col;
#pragma unroll
    for (int tap = 0; tap < K * K; ++tap) vw[tap] = (ch < cin) ? wp[(long long)tap * cout] : 0.f;
  }
  // (the values of masked pixels too, which the mask bytes, loaded beside them, drop)
  // UP: what is loaded are the LO x LO source pixels under the staged tile; the staged pixels are blended from LDS.  (Four loads
  // and four mask bytes for each staged pixel took 156 registers and two workgroups a CU instead of five: 2->32 5x5, every pixel
  // active, 1x256x256 21.1 us, this way 13.9; 8x240x320 159 -> 76; 2->256 at 1x32x32 9.4 -> 8.6.)
  const int ch = tid & 7, h_src = UP ? a.h_in >> 1 : a.h_in, w_src = UP ? a.w_in >> 1 : a.w_in;
  const int sy0 = UP ? ((iy0 + 1) >> 1) - 1 : iy0, sx0 = UP ? ((ix0 + 1) >> 1) - 1 : ix0;
  int src[NLD];
  unsigned in = 0u;
#pragma unroll
  for (int i = 0; i < NLD; ++i) {
    const int pix = (tid + 256 * i) >> 3;
    const int sy = sy0 + pix / LO, sx = sx0 + pix % LO;
    const bool k = pix < LO * LO && ch < cin && sy >= 0 && sy < h_src && sx >= 0 && sx < w_src;
    src[i] = k ? (n * h_src + sy) * w_src + sx : 0;
    in |= (k ? 1u : 0u) << i;
  }
  static_assert(NLD <= 32, "a bit for each");
  float vin[NLD];
#pragma unroll
  for (int i = 0; i < NLD; ++i) vin[i] = mie_ld(a.x, (long long)src[i] * cin + (ch < cin ? ch : 0));
  unsigned b[NLD];
  mie_mask_ask(a.xm, a.filt, src, b);
  mie_mask_asked();
  const unsigned on = mie_mask_take(a.xm, b, in), live_bits = mie_mask_take(live_m, live_b, live_in);
  const bool live[2] = {(live_bits & 1u) != 0u, (live_bits & 2u) != 0u};
  // the reservoir and addend values of the epilogue have the contraction to arrive
  long long off[2];
  int co[2];
  bool ok[2];
  float4 r0[2], add[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int idx = tid + 256 * i;
    const int p = idx >> 3, col = 4 * (idx & 7);
    const int oy = y0 + (p >> 3), ox = x0 + (p & 7);
    ok[i] = oy < hout && ox < wout;
    off[i] = (((long long)n * hout + oy) * wout + ox) * cout + co0 + col;
    co[i] = co0 + col;
  }
  conv_epilogue_load4<T, 2>(a, off, live, r0, add);
  float* const s_src = UP ? smem + LO_AT : s_in;
#pragma unroll
  for (int tap = 0; tap < K * K - LATE; ++tap) s_w[tap * 256 + tid] = vw[tap];
#pragma unroll
  for (int i = 0; i < NLD; ++i) {
    const int idx = tid + 256 * i;
    if ((idx >> 3) < LO * LO) s_src[(idx >> 3) * FC_PS + (idx & 7)] = ((on >> i) & 1u) ? vin[i] : 0.f;
  }
  __syncthreads();
  if constexpr (UP) {
#pragma unroll
    for (int i = 0; i < NIN; ++i) {
      const int pix = (tid + 256 * i) >> 3;
      const int iy = iy0 + pix / IT, ix = ix0 + pix % IT;
      float v = 0.f;
      if (iy >= 0 && iy < a.h_in && ix >= 0 && ix < a.w_in) {
        int r[2], q[2];
        float lr[2], lq[2];
        conv_up2x_coef(iy, h_src, r[0], r[1], lr[0], lr[1]);
        conv_up2x_coef(ix, w_src, q[0], q[1], lq[0], lq[1]);
#pragma unroll
        for (int j = 0; j < 4; ++j)
          if (pix < NPIX) v += lr[j >> 1] * lq[j & 1] * s_src[((r[j >> 1] - sy0) * LO + (q[j & 1] - sx0)) * FC_PS + ch];
      }
      if (pix < NPIX) s_in[pix * FC_PS + ch] = v;
    }
    __syncthreads();
    if (LATE > 0) {
#pragma unroll
      for (int tap = K * K - LATE; tap < K * K; ++tap) s_w[tap * 256 + tid] = vw[tap];
      __syncthreads();
    }
  }

  // ---- contraction ---------------------------------------------------------------------------------
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int l32 = lane & 31, half = lane >> 5;
  const int mb = wave & 1, th = wave >> 1;
  const int prow = mb * 4 + (l32 >> 3), pcol = l32 & 7;
  const float* pa = s_in + ((prow * S) * IT + pcol * S) * FC_PS + half;
  const float* pb = s_w + half * 32 + l32;
  const int npair = (cin + 1) >> 1;
  v16f acc;
#pragma unroll
  for (int r = 0; r < 16; ++r) acc[r] = 0.f;
  for (int tap = th; tap < K * K; tap += 2) {
    const int dy = tap / K, dx = tap - dy * K;
    const float* ta = pa + (dy * IT + dx) * FC_PS;
    const float* tb = pb + tap * (FC_CH * 32);
    for (int p = 0; p < npair; ++p)
      acc = __builtin_amdgcn_mfma_f32_32x32x2f32(ta[2 * p], tb[2 * p * 32], acc, 0, 0, 0);
  }
  __syncthreads();                       // every wave is done with the staged operands
  // ---- epilogue: the two tap halves park their accumulators in LDS; a thread then owns groups of four adjacent
  // output channels of a pixel (16-byte reads of the two partial sums, 16-byte reservoir accesses, 16- / 8-byte
  // delta accesses; all reservoir / addend loads of the thread as one batch, then the stores)
  float* red = smem + th * (64 * 32);
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    const int p = mb * 32 + 8 * (r >> 2) + 4 * half + (r & 3);
    red[p * 32 + l32] = acc[r];
  }
  __syncthreads();
  float4 v[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int idx = tid + 256 * i;
    const float4 s0 = *reinterpret_cast<const float4*>(&smem[4 * idx]);
    const float4 s1 = *reinterpret_cast<const float4*>(&smem[64 * 32 + 4 * idx]);
    v[i] = make_float4(s0.x + s1.x, s0.y + s1.y, s0.z + s1.z, s0.w + s1.w);
  }
  conv_epilogue_store4<T, 2>(a, off, co, ok, v, r0, add, live);
}

// The same layers with bf16 deltas on planes of many tiles.  The kernel above pays for every tile what only the launch
// needs: 25 kB of filter through registers into LDS, operands widened and read a word at a time, and the fp32 instruction
// at a quarter of the bf16 one's rate for values that have eight bits.  Here
//   * every weight is three bf16 terms whose sum is the fp32 weight (by truncation: exact, and no term overflows), so
//     three v_mfma_f32_32x32x16_bf16 multiply what 16 of the deltas need, each product exact in fp32 as before;
//   * a unit is two taps x 8 channels, so that an operand is 16 bytes of LDS: [pixel][8 channels] of the deltas and
//     [unit][term][half][column][8 channels] of the filter, both read without bank conflicts;
//   * the filter is split and staged once per workgroup, two workgroups of eight waves stay on a CU, and a wave walks
//     the tile list by itself: it stages its tile, multiplies all 64 pixels (each filter operand serves two MFMAs) and
//     writes them, with no barrier after the filter's.  Its reservoir loads are in flight during the MFMAs.
// What is left is the traffic of the reservoir and the deltas (8x480x640, 5 -> 32 channels, 20 % of the pixels: 545 MB).
// A delta that is not finite would make NaN of a zero among a weight's small terms: a wave that staged one multiplies the
// finite ones first and then the others by the large terms alone, which decide what comes out.
typedef __bf16 fc_bf16x8 __attribute__((ext_vector_type(8)));
constexpr int FH_WAVES = 8;
constexpr unsigned FH_GRID = 512;                 // two workgroups per CU

__device__ __forceinline__ unsigned fh_finite(unsigned v) {            // two bf16 values, zero where not finite
  const unsigned lo = (v & 0x7f80u) == 0x7f80u ? 0u : v & 0xffffu, hi = (v & 0x7f800000u) == 0x7f800000u ? 0u : v & 0xffff0000u;
  return lo | hi;
}

__global__ __launch_bounds__(64 * FH_WAVES, 4) void k_conv_fewcin_bf16(ConvArgsT<mie_bf16> a) {
  constexpr int K = 5, S = 1;
  constexpr int IT = 7 * S + K, NPIX = IT * IT, KK = K * K, UN = (KK + 1) / 2;
  constexpr int REGION = (NPIX + 1) * 16 > 4096 ? (NPIX + 1) * 16 : 4096;    // of a wave: its tile and a zero pixel; 32 rows of results
  constexpr int NIN = (NPIX + 1 + 63) / 64;
  __shared__ uint4 s_w[UN * 3 * 64];
  __shared__ uint4 s_reg[FH_WAVES * REGION / 16];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int cout = a.cout, cin = a.c1, co0 = blockIdx.y * 32;
  const int cap = a.ts.n * a.ts.tiles_y * a.ts.tiles_x;
  const int n_active = a.ts.counts[MIE_CNT_ACTIVE], n_stale = a.ts.counts[MIE_CNT_STALE];
  const int step = (int)gridDim.x * FH_WAVES;
  int b = (int)blockIdx.x * FH_WAVES + wave;
  int spec = a.ts.tiles[b < cap ? b : 0];

#pragma unroll
  for (int i = 0; i < (UN * 64 + 64 * FH_WAVES - 1) / (64 * FH_WAVES); ++i) {
    const int idx = tid + 64 * FH_WAVES * i;
    if (idx >= UN * 64) break;
    const int tap = idx >> 5, col = idx & 31;
    const float* wp = a.filt + (long long)tap * cout + co0 + col;
    float w[8];
#pragma unroll
    for (int ch = 0; ch < 8; ++ch) w[ch] = (tap < KK && ch < cin) ? wp[(long long)ch * KK * cout] : 0.f;
    unsigned t[3][4];
#pragma unroll
    for (int p = 0; p < 4; ++p) {
      unsigned h[2][3];
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        const float f = w[2 * p + e];
        const unsigned u = __builtin_bit_cast(unsigned, f);
        const bool finite = (u & 0x7f800000u) != 0x7f800000u;
        // (a NaN whose payload lies in the lower half stays one)
        const unsigned u0 = (u & 0xffff0000u) | (!finite && (u & 0x7fffffu) != 0u ? 0x400000u : 0u);
        const float r1 = f - __builtin_bit_cast(float, u0);
        const unsigned u1 = __builtin_bit_cast(unsigned, r1) & 0xffff0000u;
        const float r2 = r1 - __builtin_bit_cast(float, u1);
        h[e][0] = u0 >> 16;
        h[e][1] = finite ? u1 >> 16 : 0u;
        h[e][2] = finite ? __builtin_bit_cast(unsigned, r2) >> 16 : 0u;
      }
#pragma unroll
      for (int q = 0; q < 3; ++q) t[q][p] = h[0][q] | (h[1][q] << 16);
    }
    uint4* dst = s_w + (tap >> 1) * 192 + (tap & 1) * 32 + col;
#pragma unroll
    for (int q = 0; q < 3; ++q) dst[q * 64] = make_uint4(t[q][0], t[q][1], t[q][2], t[q][3]);
  }
  __syncthreads();

  uint4* const s_in = s_reg + wave * (REGION / 16);
  float* const s_out = reinterpret_cast<float*>(s_in);
  const unsigned short* const x = reinterpret_cast<const unsigned short*>(a.x);
  const int hout = a.ts.h, wout = a.ts.w;
  const int l32 = lane & 31, half = lane >> 5;
  // The ordinary epilogue -- reservoir, an activation of two straight pieces -- is branch-free and its reservoir is
  // fetched ahead; any other takes the general code, a group of channels at a time.  (With the general code unrolled in
  // its place the kernel had 8000 instructions, its branches on the activation among them.)
  const bool relu = a.act == MIE_ACT_RELU;
  const bool fast = a.res != nullptr && !a.refresh && (relu || a.act == MIE_ACT_NONE || a.act == MIE_ACT_LEAKY_RELU);
  const float slope = a.act == MIE_ACT_LEAKY_RELU ? a.slope : 1.f;
  const auto act = [&](float f) { return f > 0.f ? f : (relu ? 0.f : __fmul_rn(f, slope)); };
  int py[NIN], px[NIN];                          // pixels of the staged tile this lane loads
#pragma unroll
  for (int i = 0; i < NIN; ++i) { py[i] = (lane + 64 * i) / IT; px[i] = (lane + 64 * i) - py[i] * IT; }
  const int end = n_active + n_stale < cap ? n_active + n_stale : cap;
  for (; b < end; b += step) {
    int n, y0, x0;
    const int tk = mie_pick_tile_loaded(a.ts, b, __builtin_amdgcn_readfirstlane(spec), n_active, n_stale, n, y0, x0);
    spec = a.ts.tiles[b + step < cap ? b + step : 0];
    if (tk == 0) continue;
    // results of a lane: tile rows g = 0..7, column lane >> 3, four channels
    const int ox = x0 + (lane >> 3), col = 4 * (lane & 7);
    const long long obase = ((long long)n * hout + y0) * wout + ox;
    const unsigned short* const xn = x + (long long)n * a.h_in * a.w_in * cin;      // (offsets in a sample fit 32 bits)
    const uint8_t* const xmn = a.xm == nullptr ? nullptr : a.xm + (long long)n * a.h_in * a.w_in;
    if (tk == 2) {
#pragma unroll
      for (int g = 0; g < 8; ++g)
        if (y0 + g < hout && ox < wout)
          mie_st4(a.out, (obase + (long long)g * wout) * cout + co0 + col, make_float4(0.f, 0.f, 0.f, 0.f));
      continue;
    }
    uint8_t pm[8];
#pragma unroll
    for (int g = 0; g < 8; ++g) pm[g] = a.refresh ? (uint8_t)1 : a.ts.pixmask[y0 + g < hout && ox < wout ? obase + (long long)g * wout : 0];
    // ---- stage the tile: a lane takes whole pixels; pixels outside the image or the input mask are loaded from a place
    // that exists and cleared, so that all loads of the lane are in flight together
    const int iy0 = y0 * S - a.pad, ix0 = x0 * S - a.pad;
    unsigned short v[NIN][8];
    bool use[NIN];
#pragma unroll
    for (int i = 0; i < NIN; ++i) {
      const int pix = lane + 64 * i;
      const int iy = iy0 + py[i], ix = ix0 + px[i];
      use[i] = pix < NPIX && iy >= 0 && iy < a.h_in && ix >= 0 && ix < a.w_in;
      const unsigned po = use[i] ? (unsigned)(iy * a.w_in + ix) : 0u;
      if (xmn != nullptr) use[i] = use[i] && xmn[po] != 0;
      const unsigned xo = po * (unsigned)cin;
#pragma unroll
      for (int ch = 0; ch < 8; ++ch) v[i][ch] = ch < cin ? xn[xo + ch] : (unsigned short)0;
    }
    unsigned odd = 0u;                           // a sign bit is set once an exponent was all ones
#pragma unroll
    for (int i = 0; i < NIN; ++i) {
      const int pix = lane + 64 * i;
      unsigned u[4];
#pragma unroll
      for (int p = 0; p < 4; ++p) {
        u[p] = use[i] ? (unsigned)v[i][2 * p] | ((unsigned)v[i][2 * p + 1] << 16) : 0u;
        odd |= (u[p] & 0x7f807f80u) + 0x00800080u;
      }
      if (pix <= NPIX) s_in[pix] = make_uint4(u[0], u[1], u[2], u[3]);       // (pixel NPIX: the zero pixel)
    }
    unsigned live = 0u;                          // of the rows, which are inside the plane and its pixel mask
#pragma unroll
    for (int g = 0; g < 8; ++g) live |= pm[g] != 0 && y0 + g < hout && ox < wout ? 1u << g : 0u;
    float4 r0[8];
#pragma unroll
    for (int g = 0; g < 8; ++g) {
      r0[g] = make_float4(0.f, 0.f, 0.f, 0.f);
      if (fast && ((live >> g) & 1u)) r0[g] = mie_ld4(a.res, (obase + (long long)g * wout) * cout + co0 + col);
    }
    mie_wave_order();

    // ---- contraction: 8 rows of 8 pixels as two blocks of 32
    v16f acc[2];
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[0][r] = acc[1][r] = 0.f;
    int p0 = (l32 >> 3) * S * IT + (l32 & 7) * S, hs = half;
    asm volatile("" : "+v"(p0), "+v"(hs));       // (or the addresses of every unit are kept across tiles, and spilled)
    const bool any_odd = __any((odd & 0x80008000u) != 0u);
    if (any_odd) {                               // the contraction sees the finite values only ...
#pragma unroll 1
      for (int pix = lane; pix < NPIX; pix += 64) {
        const uint4 u = s_in[pix];
        s_in[pix] = make_uint4(fh_finite(u.x), fh_finite(u.y), fh_finite(u.z), fh_finite(u.w));
      }
      mie_wave_order();
    }
    const auto mul = [](v16f& c, const uint4& d, const uint4& w) {
      c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(fc_bf16x8, d), __builtin_bit_cast(fc_bf16x8, w), c, 0, 0, 0);
    };
#pragma unroll
    for (int u = 0; u < UN; ++u) {
      const int t0 = 2 * u, t1 = 2 * u + 1;
      const int o0 = (t0 / K) * IT + t0 % K, o1 = t1 < KK ? (t1 / K) * IT + t1 % K : 0;
      int pa = p0 + (hs ? o1 : o0), pb = pa + 4 * S * IT;
      if (t1 >= KK && hs) pa = pb = NPIX;
      const uint4 d0 = s_in[pa], d1 = s_in[pb];
      const uint4* wp = s_w + u * 192 + lane;
      const uint4 w0 = wp[0], w1 = wp[64], w2 = wp[128];
      mul(acc[0], d0, w2); mul(acc[1], d1, w2);
      mul(acc[0], d0, w1); mul(acc[1], d1, w1);
      mul(acc[0], d0, w0); mul(acc[1], d1, w0);
      __builtin_amdgcn_sched_barrier(0);         // (operands of several units ahead would not fit the registers)
    }
    if (any_odd) {                               // ... and the others follow with the large terms
      mie_wave_order();
#pragma unroll 1
      for (int pix = lane; pix < NPIX; pix += 64) {
        const int iy = iy0 + pix / IT, ix = ix0 + pix % IT;
        const bool in = iy >= 0 && iy < a.h_in && ix >= 0 && ix < a.w_in;
        const unsigned po = in ? (unsigned)(iy * a.w_in + ix) : 0u;
        const bool take = in && (xmn == nullptr || xmn[po] != 0);
        unsigned short* dst = reinterpret_cast<unsigned short*>(s_in + pix);
#pragma unroll 1
        for (int ch = 0; ch < 8; ++ch) {
          const unsigned short f = take && ch < cin ? xn[po * (unsigned)cin + ch] : (unsigned short)0;
          dst[ch] = (f & 0x7f80) == 0x7f80 ? f : (unsigned short)0;
        }
      }
      mie_wave_order();
#pragma unroll 1
      for (int u = 0; u < UN; ++u) {
        const int t = 2 * u + half;
        const int pa = t < KK ? p0 + (t / K) * IT + t % K : NPIX, pb = t < KK ? pa + 4 * S * IT : NPIX;
        const uint4 d0 = s_in[pa], d1 = s_in[pb], w0 = s_w[u * 192 + lane];
        mul(acc[0], d0, w0); mul(acc[1], d1, w0);
      }
    }

    // ---- epilogue: through LDS (over the staged tile, which is done with) to 16-byte groups of channels
#pragma unroll
    for (int mb = 0; mb < 2; ++mb) {
      mie_wave_order();
#pragma unroll
      for (int r = 0; r < 16; ++r) s_out[(8 * (r >> 2) + 4 * half + (r & 3)) * 32 + l32] = acc[mb][r];
      mie_wave_order();
      if (fast) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int g = 4 * mb + i;
          const long long off = (obase + (long long)g * wout) * cout + co0 + col;
          const float4 s4 = *reinterpret_cast<const float4*>(s_out + 4 * (lane + 64 * i));
          const float4 q = r0[g], r1 = make_float4(q.x + s4.x, q.y + s4.y, q.z + s4.z, q.w + s4.w);
          const bool l = (live >> g) & 1u;
          if (l) mie_st4(a.res, off, r1);
          if (y0 + g < hout && ox < wout)
            mie_st4(a.out, off, make_float4(l ? act(r1.x) - act(q.x) : 0.f, l ? act(r1.y) - act(q.y) : 0.f,
                                            l ? act(r1.z) - act(q.z) : 0.f, l ? act(r1.w) - act(q.w) : 0.f));
        }
      } else {
#pragma unroll 1
        for (int i = 0; i < 4; ++i) {
          const int g = 4 * mb + i;
          const long long off[1] = {(obase + (long long)g * wout) * cout + co0 + col};
          const int co[1] = {co0 + col};
          const bool ok[1] = {y0 + g < hout && ox < wout}, l[1] = {((live >> g) & 1u) != 0u};
          const float4 s4[1] = {*reinterpret_cast<const float4*>(s_out + 4 * (lane + 64 * i))};
          float4 r[1], add[1];
          conv_epilogue_load4<mie_bf16, 1>(a, off, l, r, add);
          conv_epilogue_store4<mie_bf16, 1>(a, off, co, ok, s4, r, add, l);
        }
      }
    }
    mie_wave_order();
  }
}

// 5x5, stride 1, from 2048 tiles on.  On few tiles a wave that does a whole tile by itself takes longer than four that
// share it; the times cross between 1500 and 1750 tiles, and near the crossing the number of active ones decides, which the
// host does not know: the line lies where this form is ahead by a clear margin (5 -> 32 channels with a reservoir, graph of
// 20 calls, one workgroup a tile -> this: 1452 tiles, 409 active, 10.2 -> 12.8 us; 1750, 829 active, 14.0 -> 13.4; 2904, 1964 active, 25.4 -> 15.8; 38400, 3190 active, 39.7 -> 22.3, 26543 active, 256
// -> 122, which is 4.5 TB/s).  3x3 stride 2 has so few products that the form above stays ahead at every size in use (4 ->
// 64, 2400 tiles, 1026 active: 16.4 us against 19.6).
constexpr unsigned FH_MIN_TILES = 2048;

bool launch_fewcin_many(const ConvArgsT<float>&, int, int, unsigned, hipStream_t) { return false; }
bool launch_fewcin_many(const ConvArgsT<mie_bf16>& a, int k, int s, unsigned cap, hipStream_t st) {
  if (k != 5 || s != 1 || cap < FH_MIN_TILES || a.addend != nullptr || (long long)a.h_in * a.w_in >= 1 << 27) return false;
  const unsigned wgs = (cap + FH_WAVES - 1) / FH_WAVES;
  hipLaunchKernelGGL(k_conv_fewcin_bf16, dim3(wgs < FH_GRID ? wgs : FH_GRID, a.cout / 32), dim3(64 * FH_WAVES), 0, st, a);
  return true;
}

template <typename T>
bool launch_fewcin(const ConvArgsT<T>& a, int k, int s, unsigned cap, hipStream_t st) {
  if (a.x2 != nullptr || a.c1 < 1 || a.c1 > FC_CH || a.cout % 32 != 0) return false;
  if (launch_fewcin_many(a, k, s, cap, st)) return true;
  const dim3 grid(cap, a.cout / 32), block(256);
  switch (k * 10 + s) {
    case 31: hipLaunchKernelGGL((k_conv_fewcin<T, 3, 1>), grid, block, 0, st, a); return true;
    case 32: hipLaunchKernelGGL((k_conv_fewcin<T, 3, 2>), grid, block, 0, st, a); return true;
    case 51: hipLaunchKernelGGL((k_conv_fewcin<T, 5, 1>), grid, block, 0, st, a); return true;
    case 52: hipLaunchKernelGGL((k_conv_fewcin<T, 5, 2>), grid, block, 0, st, a); return true;
    default: return false;
  }
}

template <typename T>
bool launch_fewcin_up(const ConvArgsT<T>& a, int k, unsigned cap, hipStream_t st) {
  if (a.x2 != nullptr || a.c1 < 1 || a.c1 > FC_CH || a.cout % 32 != 0 || a.pad != k / 2) return false;
  const dim3 grid(cap, a.cout / 32), block(256);
  switch (k) {
    case 3: hipLaunchKernelGGL((k_conv_fewcin<T, 3, 1, true>), grid, block, 0, st, a); return true;
    case 5: hipLaunchKernelGGL((k_conv_fewcin<T, 5, 1, true>), grid, block, 0, st, a); return true;
    default: return false;
  }
}

}  // namespace

bool mie_launch_conv_fewcin_up(const ConvArgsT<float>& a, int k, unsigned cap, hipStream_t st) {
  return launch_fewcin_up(a, k, cap, st);
}
bool mie_launch_conv_fewcin_up(const ConvArgsT<mie_bf16>& a, int k, unsigned cap, hipStream_t st) {
  return launch_fewcin_up(a, k, cap, st);
}
bool mie_launch_conv_fewcin(const ConvArgsT<float>& a, int k, int s, unsigned cap, hipStream_t st) {
  return launch_fewcin(a, k, s, cap, st);
}
bool mie_launch_conv_fewcin(const ConvArgsT<mie_bf16>& a, int k, int s, unsigned cap, hipStream_t st) {
  return launch_fewcin(a, k, s, cap, st);
}
