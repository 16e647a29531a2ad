// The decoder layer -- 5x5 conv, pad 2, over up2x(a + b), the bilinear x2 up-sampling of the sum of two deltas -- computed
// at the resolution of its inputs (gfx950).
//
// Sub-pixel phases.  Along one axis output 2Y + q (q = 0, 1) of the conv over the up-sampled signal is a fixed combination
// of four input samples, L[Y - 2 .. Y + 1] for q = 0 and L[Y - 1 .. Y + 2] for q = 1, with coefficients that are sums of the
// five weights times 1/4 and 3/4.  In two dimensions each of the four output phases (py, px) is therefore an ordinary 4x4
// conv over a + b: 16 taps where the conv over the up-sampled tile multiplies 25, nothing to blend, and a staged tile of
// 11x11 input pixels for 64 outputs where the other form stages and blends 12x12 (k_conv_mfma<..., UP>, which
// this replaces wherever a combined filter can be made: 0.64 of its matrix-core work and none of its blend).
//
// Border.  Up-sampled rows outside the image are the conv's zero padding and the bilinear taps are clamped, so the outputs of
// input rows 0 and H - 1 and of columns 0 and W - 1 have filters of their own: three input rows deep across the border
// instead of four.  Those positions go to workgroups of their own ("strips": 32 positions along one side, half an M block,
// 12 taps; the columns' strips leave the corners to the rows', which subtract there what the column outside the image
// would have given, a 3x1 filter on the corner lane only).  Everything else runs 16 taps and no special case.  (First built
// as corrections inside ordinary blocks: a corner block then ran 25 taps' worth, and on the 33x44 plane, one round of
// workgroups, every launch took as long as its corners.)
//
// Work decomposition: one workgroup (4 waves) = an 8x8 block of input positions (or a strip) x one phase x 32 * WN output
// channels, M = 64, as in k_conv_mfma (same LDS layout, operand pairing, three-term form of fp32 deltas).  The filter runs
// through a register ring three units ahead, across sub-chunks and chunks.
// Work is found from the 8x8 tiles' flag words: a workgroup looks at the tiles its positions touch and leaves if none is
// active (zeroing its pixels of stale ones).  There is no list to walk: behind the bottleneck these planes are active
// throughout (every tile, at every density from 0.5 %), and a list of blocks would be one more tile set to build.
// (Flag words are looked up where they are needed: kept in a small array indexed at run time they went to LDS, whose
// promotion reads the workgroup size from the dispatch packet in host memory -- 7 us at the start of every workgroup.)
#include "mie_conv_mfma_impl.h"
#include "mie_pack_terms.h"

namespace {

// Units of a phase's filter: 16 of the interior, [row][column]; then 12 of each side, [depth across the border][tap along
// it], the sides at the top and the bottom followed by two groups of their corners (three taps across and a zero).
constexpr int UNITS = UP2X_UNITS, U_TOP = 16, U_BOTTOM = 36, U_LEFT = 56, U_RIGHT = 68;
constexpr int STRIP = 32;                 // positions of a border workgroup

struct Up2xOrder {
  const uint32_t* flags;                  // tile flags of the output tile set
  int blocks_y, blocks_x;                 // 8x8 blocks of the positions 1 .. H - 2, 1 .. W - 2
  int strips_x, strips_y;                 // strips of the top (and of the bottom), of the left (and of the right)
  int items;                              // of a sample: the blocks, then the strips
  int combos, groups;                     // (phase, slab) pairs, and how many parts of the launch order they are cut into
  int total;                              // samples * items * combos
  int cpg, per_group;                     // combos, and places of the order, of a group
  unsigned m_group, m_cpg, m_items, m_bx;                  // mie_tile_div by per_group, cpg, items, blocks_x
  int nci;                                // blocks of 16 input channels in the filter
};

// 1-D coefficients of the five weights.  row 0..3: the 4-tap filter of phase q (window row 0 is Y - 2 + q); 4 / 5: what the
// continued signal gives too much at the first / last position; 6..8 / 9..11: the whole filter of the first / last
// position on the samples 0, 1, 2 steps inside.
__device__ void up2x_coef(int q, int row, double (&c)[5]) {
  for (int k = 0; k < 5; ++k) {
    double v = 0.0;
    if (row < 4) {
      // up-sampled sample s = q - 2 + k relative to 2Y; even s = 2R: L[R - 1] / 4 + 3 L[R] / 4, odd: 3 L[R] / 4 + L[R + 1] / 4
      const int s = q - 2 + k, r = (s - (s & 1)) / 2;           // (s & 1 is 0 or 1 for negative s, too)
      const int lo = (s & 1) ? r : r - 1, want = row - 2 + q;
      if (want == lo) v = (s & 1) ? 0.75 : 0.25;
      else if (want == lo + 1) v = (s & 1) ? 0.25 : 0.75;
    } else if (row == 4) {
      v = (k < 2 - q) ? 1.0 : 0.0;
    } else if (row == 5) {
      v = (k > 3 - q) ? 1.0 : 0.0;
    }
    c[k] = v;
  }
  if (row < 6) return;
  const bool first = row < 9;
  const int depth = first ? row - 6 : row - 9;
  double t[5];
  for (int w = 0; w < 4; ++w) {
    const int at = first ? w - 2 + q : 2 - q - w;               // steps inside of window row w (outside: the edge sample)
    if ((at < 0 ? 0 : at) != depth) continue;
    up2x_coef(q, w, t);
    for (int k = 0; k < 5; ++k) c[k] += t[k];
  }
  if (depth == 0) {
    up2x_coef(q, first ? 4 : 5, t);
    for (int k = 0; k < 5; ++k) c[k] -= t[k];
  }
}

// The coefficients of unit u of phase ph's filter, down and across.
__device__ void up2x_unit(int ph, int u, double (&cv)[5], double (&ch)[5]) {
  int vr, hr;
  double sign = 1.0;
  if (u < U_TOP) {
    vr = u >> 2; hr = u & 3;
  } else if (u < U_LEFT) {
    const int side = u < U_BOTTOM ? 0 : 1, k = u - (side ? U_BOTTOM : U_TOP);
    if (k < 12) { vr = 6 + 3 * side + (k >> 2); hr = k & 3; }
    else { vr = 6 + 3 * side + (k & 3); hr = k < 16 ? 4 : 5; sign = (k & 3) < 3 ? -1.0 : 0.0; if ((k & 3) == 3) vr = 0; }
  } else {
    const int side = u < U_RIGHT ? 0 : 1, k = u - (side ? U_RIGHT : U_LEFT);
    vr = k & 3; hr = 6 + 3 * side + (k >> 2);
  }
  up2x_coef(ph >> 1, vr, cv);
  up2x_coef(ph & 1, hr, ch);
  for (int k = 0; k < 5; ++k) cv[k] *= sign;
}
__device__ __forceinline__ float up2x_weight(const float* __restrict__ f, const double (&cv)[5], const double (&ch)[5], int ci, int co, int cout) {
  double v = 0.0;
  for (int ky = 0; ky < 5; ++ky)
    for (int kx = 0; kx < 5; ++kx) v += cv[ky] * ch[kx] * (double)f[((long long)ci * 25 + ky * 5 + kx) * cout + co];
  return (float)v;
}

// P[phase][ci/16][unit][term][(ci%16)/8][co][ci%8] in bf16: one term (bf16 deltas) or the three of an fp32 value.
template <int PL>
__global__ __launch_bounds__(256) void k_pack_up2x(const float* __restrict__ f, mie_bf16* __restrict__ p, int cin, int cout) {
  const long long i = (long long)blockIdx.x * 256 + threadIdx.x;
  if (i >= 4LL * UNITS * cin * cout) return;
  const int co = (int)(i % cout);
  long long t = i / cout;
  const int ci = (int)(t % cin);
  t /= cin;
  const int u = (int)(t % UNITS), ph = (int)(t / UNITS);
  double cv[5], ch[5];
  up2x_unit(ph, u, cv, ch);
  const float w = up2x_weight(f, cv, ch, ci, co, cout);
  const long long o = ((((((long long)ph * (cin / 16) + ci / 16) * UNITS + u) * PL) * 2 + (ci % 16) / 8) * cout + co) * 8 + ci % 8;
  const long long term = 2LL * cout * 8;
  const mie_bf16 hi = (mie_bf16)w;
  p[o] = hi;
  if (PL == 3) {
    const float r1 = w - (float)hi;
    const mie_bf16 mid = (mie_bf16)r1;
    p[o + term] = mid;
    p[o + 2 * term] = (mie_bf16)(r1 - (float)mid);
  }
}
// The fp32 values of the two-term copy in their places, and the ranges of the blocks (mie_pack_terms.h).
__global__ __launch_bounds__(256) void k_f2_up2x_values(const float* __restrict__ f, float* __restrict__ values, unsigned* __restrict__ parts,
                                                        long long groups, int cin, int cout) {
  unsigned most = 0u, least = ~0u;
  for (long long g = (long long)blockIdx.x * 256 + threadIdx.x; g < groups; g += (long long)gridDim.x * 256) {
    const int co = (int)(g % cout), half = (int)((g / cout) & 1);
    const long long t = g / cout / 2;
    const int u = (int)(t % UNITS), blk = (int)(t / UNITS % (cin / 16)), ph = (int)(t / UNITS / (cin / 16));
    double cv[5], ch[5];
    up2x_unit(ph, u, cv, ch);
    float v[8];
#pragma unroll 1
    for (int j = 0; j < 8; ++j) v[j] = up2x_weight(f, cv, ch, blk * 16 + half * 8 + j, co, cout);
    f2_put_values(values, t, half, co, cout, v, most, least);
  }
  f2_put_parts(parts, most, least);
}

// A unit of two M blocks in the three-term form, only the product of the leading terms into `acc` and the five smaller ones
// into `sm` (mma_unit2_x3 has two of them, 2^-9 of the leading one, in `acc`): a third of the roundings at the size of the
// sum.  The four phases' chains are longer than the list-driven form's, which splits the channels over more waves; with
// mma_unit2_x3 the error against fp64 was up to 1.13 times that form's at some layers of the networks (128->64 at 66x88:
// 3.5e-7 of the output against 3.1e-7), this way it is below it at all of them (1.9e-7).  Same time: an MFMA waits for the
// one before the last at most.
__device__ __forceinline__ void mma_up2x_x3(v16f& acc0, v16f& acc1, v16f& sm0, v16f& sm1, const float4 (&a0)[3],
                                            const float4 (&a1)[3], const float4 (&b)[3]) {
  mma_unit(sm0, a0[2], b[0], mie_bf16()); mma_unit(sm1, a1[2], b[0], mie_bf16());
  mma_unit(acc0, a0[0], b[0], mie_bf16()); mma_unit(acc1, a1[0], b[0], mie_bf16());
  mma_unit(sm0, a0[1], b[1], mie_bf16()); mma_unit(sm1, a1[1], b[1], mie_bf16());
  mma_unit(sm0, a0[0], b[2], mie_bf16()); mma_unit(sm1, a1[0], b[2], mie_bf16());
  mma_unit(sm0, a0[1], b[0], mie_bf16()); mma_unit(sm1, a1[1], b[0], mie_bf16());
  mma_unit(sm0, a0[0], b[1], mie_bf16()); mma_unit(sm1, a1[0], b[1], mie_bf16());
}

// The same in two fp16 terms, half as many products (kernel alone, all tiles active, three terms -> two: 256->128 at 33x44 48.0 -> 30.4 us,
// 128->64 at 66x88 45.6 -> 28.8, at 32x32 15.1 -> 12.3).  The leading products of a chunk's units go in turn into two accumulators: with
// one the error, relative 2-norm against fp64, would be that of three terms or above (256->128 at 33x44 2.8e-7), this way it is
// 2.77 -> 2.22e-7, 1.97 -> 1.73e-7 and 1.45 -> 1.43e-7.
__device__ __forceinline__ void mma_up2x_f2(v16f& acc0, v16f& acc1, v16f& sm0, v16f& sm1, const float4 (&a0)[2], const float4 (&a1)[2],
                                            const float4 (&b)[2]) {
  mma_f16(sm0, a0[1], b[0]);  mma_f16(sm1, a1[1], b[0]);
  mma_f16(acc0, a0[0], b[0]); mma_f16(acc1, a1[0], b[0]);
  mma_f16(sm0, a0[0], b[1]);  mma_f16(sm1, a1[0], b[1]);
}

// AR: 0 bf16 deltas, 1 fp32 in three bf16 terms, 2 in two fp16 terms (mie_conv_mfma_impl.h).
template <typename T, int WN, int AR>
__global__ __launch_bounds__(256, sizeof(T) == 4 ? 2 : 3) void k_upconv2x(ConvArgsT<T> a, Up2xOrder od) {
  static_assert((AR != 0) == (sizeof(T) == 4), "fp32 deltas in terms, bf16 as they are");
  constexpr bool X3 = AR != 0, F2 = AR == 2;
  typedef mie_bf16 TL;
  constexpr int PL = F2 ? 2 : X3 ? 3 : 1;
  constexpr int GPS = X3 ? 2 : 1;                            // 16-byte global loads per staging slot
  constexpr int NBUF = X3 ? 2 : 1;
  constexpr int EPS = 8, SUB = 16;
  constexpr int WK = 4 / WN;
  constexpr int IT = 11;
  constexpr int CC = X3 ? 32 : 64;
  constexpr int LS = CC + EPS;
  constexpr int Q4 = CC / EPS;
  constexpr int NSLOT = IT * IT * Q4;
  constexpr int NLD = (NSLOT + 255) / 256;
  constexpr int RP = row_pitch_dw(IT, LS / 2, 1) * 2;
  constexpr int ZOFF = IT * RP;                              // the zero pixel behind the tile
  constexpr int STAGE = ZOFF + LS;
  constexpr int SPX = STRIP + 3;                             // staged positions along a strip, three rows of them
  constexpr int RPS = SPX * LS;
  static_assert(3 * SPX <= IT * IT && 3 * RPS <= ZOFF, "a strip stages less than a block");
  constexpr int NQ = CC / SUB;
  constexpr int KS = NQ < WK ? NQ : WK;                      // the k-split: over sub-chunks, ...
  constexpr int NQW = NQ / KS;                               // ... several of them per wave, ...
  constexpr int RC = WK / KS;                                // ... or one of them and half of the tap rows
  constexpr int NI = 4 / RC;                                 // tap rows of a wave
  constexpr int UPC = 4 * NI * NQW;                          // units per chunk and wave
  constexpr int CO_BLK = 32 * WN;
  constexpr int RED = WK * 64 * CO_BLK;
  constexpr int STAGE_F = NBUF * PL * STAGE / 2;
  constexpr int SMEM = STAGE_F > RED ? STAGE_F : RED;
  static_assert(SMEM * 4 <= 65536, "LDS budget");
  __shared__ __attribute__((aligned(16))) float smem[SMEM];
  __shared__ float s_f2[F2 ? 7 : 1];                         // F2: largest values of the waves' first slots; whether a group of a chunk does not fit,
                                                             // of every other one in the same place
  TL* const sbuf = reinterpret_cast<TL*>(smem);

  // ---- which positions, phase and slab: each XCD (workgroup index mod 8) takes a contiguous eighth of the order (group of
  // (phase, slab) pairs, item, pair within the group)
  const int bid = blockIdx.x + conv_args_entry_zero(a);
  const int share = (od.total + 7) >> 3;
  const int v = (bid & 7) * share + (bid >> 3);
  if ((bid >> 3) >= share || v >= od.total) return;
  const int cg = mie_tile_div(v, od.per_group, od.m_group), rem = v - cg * od.per_group;
  const int it = mie_tile_div(rem, od.cpg, od.m_cpg), combo = cg * od.cpg + (rem - it * od.cpg);
  const int phase = combo & 3, slab = combo >> 2;
  const int n = mie_tile_div(it, od.items, od.m_items);
  const int py = phase >> 1, px = phase & 1;
  const int H = a.h_in, W = a.w_in, hout = a.ts.h, wout = a.ts.w;
  // side: 0 a block at (y0, x0), rows x cols positions; 1 .. 4 a strip at the top, bottom, left, right
  int side = 0, y0, x0, rows, cols;
  {
    int k = it - n * od.items;
    const int nb = od.blocks_y * od.blocks_x;
    if (k < nb) {
      const int by = mie_tile_div(k, od.blocks_x, od.m_bx);
      y0 = 1 + 8 * by; x0 = 1 + 8 * (k - by * od.blocks_x);
      rows = H - 1 - y0 < 8 ? H - 1 - y0 : 8; cols = W - 1 - x0 < 8 ? W - 1 - x0 : 8;
    } else if ((k -= nb) < 2 * od.strips_x) {
      side = 1 + (k >= od.strips_x ? 1 : 0);
      x0 = STRIP * (k - (side - 1) * od.strips_x); y0 = side == 1 ? 0 : H - 1;
      rows = 1; cols = W - x0 < STRIP ? W - x0 : STRIP;
    } else {
      k -= 2 * od.strips_x;
      side = 3 + (k >= od.strips_y ? 1 : 0);
      y0 = 1 + STRIP * (k - (side - 3) * od.strips_y); x0 = side == 3 ? 0 : W - 1;
      rows = H - 1 - y0 < STRIP ? H - 1 - y0 : STRIP; cols = 1;
    }
  }
  const bool lying = side == 1 || side == 2;                 // a strip along a row of the plane
  // position p of the M block, relative to (y0, x0)
  auto pos_y = [&](int p) { return side == 0 ? p >> 3 : (lying ? 0 : p); };
  auto pos_x = [&](int p) { return side == 0 ? p & 7 : (lying ? p : 0); };

  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int l32 = lane & 31, half = lane >> 5;
  const int wn = wave % WN, wk = wave / WN;
  const int co0 = slab * CO_BLK, cout = a.cout;

  // the tiles these positions touch (at most 3x3 or 1x9 of them), one per lane
  const int tl_y = y0 >> 2, tl_x = x0 >> 2, tl_nx = ((2 * (x0 + cols) - 1) >> 3) - tl_x + 1, tl_ny = ((2 * (y0 + rows) - 1) >> 3) - tl_y + 1;
  const int* const flags_n = reinterpret_cast<const int*>(od.flags) + (long long)n * a.ts.tiles_y * a.ts.tiles_x;
  {
    const bool in = lane < tl_nx * tl_ny;
    const int f = flags_n[(tl_y + (in ? lane / tl_nx : 0)) * a.ts.tiles_x + tl_x + (in ? lane % tl_nx : 0)];
    if (__ballot((f & 1) != 0) == 0ull) {
      if (__ballot((f & 2) != 0) != 0ull)          // nothing active, something stale: zero this phase of it
        for (int idx = tid; idx < 64 * (CO_BLK / 4); idx += 256) {
          const int p = idx / (CO_BLK / 4), col = 4 * (idx - p * (CO_BLK / 4));
          const int dy = pos_y(p), dx = pos_x(p);
          if (dy >= rows || dx >= cols) continue;
          const int oy = 2 * (y0 + dy) + py, ox = 2 * (x0 + dx) + px;
          if ((flags_n[(oy >> 3) * a.ts.tiles_x + (ox >> 3)] & 2) != 0)
            mie_st4(a.out, (((long long)n * hout + oy) * wout + ox) * cout + co0 + col, make_float4(0.f, 0.f, 0.f, 0.f));
        }
      return;
    }
  }

  // ---- epilogue plan: a thread owns groups of four adjacent output channels of a pixel; the mask bytes are asked for now
  constexpr int QPP = CO_BLK / 4;
  constexpr int PER = 64 * QPP / 256;
  constexpr int PB = PER > 4 ? 4 : PER;
  int at[PER];
  unsigned in = 0u;
#pragma unroll
  for (int g = 0; g < PER; ++g) {
    const int p = (tid + 256 * g) / QPP;
    const int dy = pos_y(p), dx = pos_x(p);
    const bool k = dy < rows && dx < cols;
    at[g] = k ? (n * hout + 2 * (y0 + dy) + py) * wout + 2 * (x0 + dx) + px : 0;
    in |= (k ? 1u : 0u) << g;
  }
  const uint8_t* const live_m = a.refresh ? nullptr : a.ts.pixmask;
  unsigned live_b[PER];
  mie_mask_ask(live_m, a.filt_mc, at, live_b);

  // ---- staging plan.  A block: its 11x11 window, rows from y0 - 2 + py on.  A strip: three rows of 35, row b the pixels b
  // steps inside the border, from two (one) before the first position on.  Edge pixels continue the plane.
  const bool has2 = a.x2 != nullptr;
  unsigned st_off[NLD];                                      // byte offset of the slot in chunk 0
  int st_lds[NLD], st_po[NLD];
#pragma unroll
  for (int i = 0; i < NLD; ++i) {
    const int slot = tid + 256 * i;
    const int q4 = slot & (Q4 - 1);
    int pix = slot / Q4, iy, ix;
    if (side == 0) {
      if (pix >= IT * IT) pix = 0;
      const int r = pix / IT, c = pix - r * IT;
      iy = y0 - 2 + py + r; ix = x0 - 2 + px + c;
      st_lds[i] = r * RP + c * LS + EPS * q4;
    } else {
      if (pix >= 3 * SPX) pix = 0;
      const int b = pix / SPX, c = pix - b * SPX;
      const int in = (side & 1) ? b : -b, along = c - 2 + (lying ? px : py);
      iy = y0 + (lying ? in : along); ix = x0 + (lying ? along : in);
      st_lds[i] = b * RPS + c * LS + EPS * q4;
    }
    iy = iy < 0 ? 0 : (iy >= H ? H - 1 : iy);
    ix = ix < 0 ? 0 : (ix >= W ? W - 1 : ix);
    const int po = (n * H + iy) * W + ix;
    st_off[i] = ((unsigned)po * (unsigned)a.c1 + (unsigned)(EPS * q4)) * (unsigned)sizeof(T);
    st_po[i] = po;
  }
  const uint8_t* const x2m = has2 ? a.x2m : nullptr;
  unsigned b1[NLD], b2[NLD], ok1 = 0u, ok2 = 0u, live_bits = 0u;      // (taken behind the first chunk's loads)
  mie_mask_ask(a.xm, a.filt_mc, st_po, b1);
  mie_mask_ask(x2m, a.filt_mc, st_po, b2);
  const int n_slots = (side == 0 ? IT * IT : 3 * SPX) * Q4;
  const int nch = a.c1 / CC;

  // Loads are for every pixel, active or not (these planes are dense): masked values are dropped when they are stored.
  float4 ra[NLD][GPS], rb[NLD][GPS];
  const T* x2p = has2 ? a.x2 : a.x;
  auto stage_load = [&](int c) {
    const char* xc = reinterpret_cast<const char*>(a.x + c * CC);
    const char* x2c = reinterpret_cast<const char*>(x2p + c * CC);
#pragma unroll
    for (int i = 0; i < NLD; ++i)
#pragma unroll
      for (int g = 0; g < GPS; ++g) {
        ra[i][g] = *reinterpret_cast<const float4*>(xc + st_off[i] + 16 * g);
        rb[i][g] = *reinterpret_cast<const float4*>(x2c + st_off[i] + 16 * g);
      }
  };
  F2Groups groups;
  // (terms: 1 in terms, F2: 2 in three of them, 0 as it is; first: the first chunk, F2's scale from it)
  auto stage_store = [&](int buf, auto terms, bool first = false) __attribute__((always_inline)) {
    constexpr int FORM = decltype(terms)::value;
    TL* dst = sbuf + buf * (PL * STAGE);
    const float4 z4 = make_float4(0.f, 0.f, 0.f, 0.f);
    float v[F2 ? NLD : 1][8];
    auto sum = [&](int i, float (&f)[8]) __attribute__((always_inline)) {
      const bool k1 = (ok1 >> i) & 1u, k2 = (ok2 >> i) & 1u;
      float fa[8], fb[8];
      if constexpr (X3) {
        const float4 a0 = k1 ? ra[i][0] : z4, a1 = k1 ? ra[i][1] : z4, b0 = k2 ? rb[i][0] : z4, b1 = k2 ? rb[i][1] : z4;
        const float ta[8] = {a0.x, a0.y, a0.z, a0.w, a1.x, a1.y, a1.z, a1.w};
        const float tb[8] = {b0.x, b0.y, b0.z, b0.w, b1.x, b1.y, b1.z, b1.w};
#pragma unroll
        for (int e = 0; e < 8; ++e) fa[e] = ta[e], fb[e] = tb[e];
      } else {
        slot_to_f32(k1 ? ra[i][0] : z4, fa, T());
        slot_to_f32(k2 ? rb[i][0] : z4, fb, T());
      }
#pragma unroll
      for (int e = 0; e < 8; ++e) f[e] = fa[e] + fb[e];
    };
    if constexpr (F2) {
#pragma unroll
      for (int i = 0; i < NLD; ++i) sum(i, v[i]);
      if (FORM == 1 && first) {
        float m = 0.f;
#pragma unroll
        for (int i = 0; i < NLD; ++i) m = __builtin_elementwise_maximum(m, f2_amax8(v[i]));
        m = f2_wave_max(m);
        if (lane == 0) s_f2[wave] = m;
        if (tid < 2) s_f2[4 + tid] = 0.f;
        __syncthreads();
        groups.start(f2_scale(__int_as_float(__builtin_amdgcn_readfirstlane(
            __float_as_int(__builtin_elementwise_maximum(f2_max3(s_f2[0], s_f2[1], s_f2[2]), s_f2[3]))))));
      }
    }
#pragma unroll
    for (int i = 0; i < NLD; ++i) {
      float f[8];
      if constexpr (F2) {
#pragma unroll
        for (int e = 0; e < 8; ++e) f[e] = v[i][e];
      } else {
        sum(i, f);
      }
      if (tid + 256 * i < n_slots) {
        if constexpr (F2) {
          float4 pl[FORM == 2 ? 3 : 2];
          pl[0] = make_float4(f[0], f[1], f[2], f[3]); pl[1] = make_float4(f[4], f[5], f[6], f[7]);
          if constexpr (FORM == 1) groups.terms(f, pl);
          else groups.note(f);
          if constexpr (FORM == 2) split3(f, pl);
#pragma unroll
          for (int q = 0; q < (FORM == 2 ? 3 : 2); ++q) *reinterpret_cast<float4*>(dst + q * STAGE + st_lds[i]) = pl[q];
        } else if constexpr (X3) {
          float4 pl[3];
          split3(f, pl);
#pragma unroll
          for (int q = 0; q < 3; ++q) *reinterpret_cast<float4*>(dst + q * STAGE + st_lds[i]) = pl[q];
        } else {
          *reinterpret_cast<float4*>(dst + st_lds[i]) = f32_to_slot(f, T());
        }
      }
    }
  };

  // ---- the units of this wave ---------------------------------------------------------------------------------------------
  // A block: NI rows of four taps per sub-chunk.  A strip: groups of four units, packed in `strip`: codes 0..2 its rows, 3 / 4
  // the corner groups of its first / last position (the two row classes of a k-split over rows share them out).
  const int q0w = (RC > 1) ? wk % KS : wk * NQW;
  const int cls = (RC > 1) ? wk / KS : 0;
  unsigned strip = 0u;
  int ng = 0;
  {
    auto add = [&](bool on, int code) {
      strip |= on ? (unsigned)code << (4 * ng) : 0u;
      ng += on ? 1 : 0;
    };
    if (cls == 0) { add(true, 0); add(true, 1); }
    if (cls == RC - 1) { add(true, 2); add(lying && x0 == 0, 3); add(lying && x0 + cols == W, 4); }
  }
  const int u_side = side == 1 ? U_TOP : (side == 2 ? U_BOTTOM : (side == 3 ? U_LEFT : U_RIGHT));
  const int jx = 2 - px;                                     // window column of the position itself
  int a_lane[2];
#pragma unroll
  for (int mb = 0; mb < 2; ++mb) {
    const int p = mb * 32 + l32;
    a_lane[mb] = (side == 0 ? (p >> 3) * RP + (p & 7) * LS : l32 * LS) + SUB * q0w + EPS * half;
  }
  const bool at_first = l32 == 0, at_last = l32 == cols - 1;
  const int b_lane = (half * cout + l32) * EPS;
  const int unit_sz = PL * 2 * cout * EPS;                   // elements
  const TL* const filt = reinterpret_cast<const TL*>(a.filt_mc) + (co0 + wn * 32) * EPS;
  // the four units from `unit` on, of sub-chunk qi of this wave in chunk c
  auto group_b = [&](int c, int qi, int unit) -> const TL* {
    return filt + ((long long)(phase * od.nci + c * NQ + q0w + qi) * UNITS + unit) * unit_sz;
  };
  auto strip_unit = [&](int g) { return u_side + 4 * (int)((strip >> (4 * g)) & 15u); };
  // the filter is read in order through one pointer per lane, set anew where a group does not follow the one before it
  // (offsets from a base would all be kept in registers across the chunks)
  const TL* bp;
  auto seek_b = [&](const TL* gb) { bp = gb + b_lane; };
  auto load_b = [&](float4 (&bv)[PL]) {
#pragma unroll
    for (int q = 0; q < PL; ++q) {
      bv[q] = *reinterpret_cast<const float4*>(bp);
      bp += 2 * cout * EPS;
    }
  };
  auto first_b = [&](int c) { return group_b(c, 0, side == 0 ? 4 * NI * cls : strip_unit(0)); };

  v16f acc[2], acc_odd[F2 ? 2 : 1], sm[X3 ? 2 : 1];
#pragma unroll
  for (int mb = 0; mb < 2; ++mb)
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      acc[mb][r] = 0.f;
      if (F2) acc_odd[mb][r] = 0.f;
      if (X3) sm[mb][r] = 0.f;
    }
  // F2: the filter's scale and whether it fits, on their way from here on
  const long long weights = 4LL * UNITS * a.c1 * cout;
  float filt_unscale = 1.f;
  float filt_form = 1.f;
  if constexpr (F2) {
    const float* const end = f2_filter_end(a.filt_mc, weights);
    filt_unscale = end[0];
    filt_form = end[1] - end[2];
  }
  int c_end = nch;                         // F2: where the contraction in two terms ends: in front of the first chunk that does not fit
  auto note_misfit = [&](int c) __attribute__((always_inline)) {      // in front of the barrier behind the stores of chunk c ...
    if constexpr (F2) {
      s_f2[groups.misfit() ? 4 + (c & 1) : 6] = 1.f;      // (without a branch)
    }
  };
  // ... asked behind it whether some thread noted one, and looked at where the chunk begins (true: it does not fit)
  float stop = 0.f;
  auto ask_stop = [&](int c) __attribute__((always_inline)) {
    if constexpr (F2) stop = s_f2[4 + (c & 1)];
  };
  auto stops_at = [&](int c) __attribute__((always_inline)) {
    if constexpr (F2) {
      if (__builtin_expect(__builtin_amdgcn_readfirstlane(__float_as_int(stop)) != 0, 0)) {
        c_end = c;
        return true;
      }
    }
    return false;
  };

  float4 bring[4][PL];
  seek_b(first_b(0));
  stage_load(0);
#pragma unroll
  for (int i = 0; i < 3; ++i) load_b(bring[i]);
  mie_mask_asked();
  ok1 = mie_mask_take(a.xm, b1, ~0u);
  ok2 = mie_mask_take(x2m, b2, has2 ? ~0u : 0u);
  live_bits = mie_mask_take(live_m, live_b, in);
  // the zero pixels
  for (int i = tid; i < NBUF * PL * (LS / EPS); i += 256) {
    const int pl = i / (LS / EPS);
    *reinterpret_cast<float4*>(sbuf + pl * STAGE + ZOFF + EPS * (i - pl * (LS / EPS))) = make_float4(0.f, 0.f, 0.f, 0.f);
  }
  const auto in_terms = std::integral_constant<int, 1>();
  stage_store(0, in_terms, true);
  note_misfit(0);
  __syncthreads();
  if (F2 && filt_form != 1.f) c_end = 0;
  ask_stop(0);

  // All loads of a chunk are unconditional (see k_conv_mfma); behind the last one "the next" is the chunk itself.
  auto contract = [&](auto block) {
    for (int c = 0; c < c_end; ++c) {
      const bool more = c + 1 < nch;
      const int cn = more ? c + 1 : c;
      const TL* const ub_next = first_b(cn);
      stage_load(cn);
      const TL* sin = sbuf + (c % NBUF) * (PL * STAGE);
      if constexpr (decltype(block)::value) {
        const TL* sa = sin + cls * NI * RP;
        float4 av[2][2][PL];
        auto load_a = [&](int u, float4 (&dst)[2][PL]) {
          const int qi = u / (4 * NI), k = u % (4 * NI);
#pragma unroll
          for (int mb = 0; mb < 2; ++mb)
#pragma unroll
            for (int q = 0; q < PL; ++q)
              dst[mb][q] = *reinterpret_cast<const float4*>(&sa[q * STAGE + a_lane[mb] + (k >> 2) * RP + (k & 3) * LS + SUB * qi]);
        };
        load_a(0, av[0]);
        if (stops_at(c)) break;
#pragma unroll
        for (int i = 0; i < UPC; ++i) {
          const int ip = i + 3;
          if (ip == UPC) seek_b(ub_next);
          else if (ip % (4 * NI) == 0) seek_b(group_b(c, ip / (4 * NI), 4 * NI * cls));
          load_b(bring[ip & 3]);
          if (i + 1 < UPC) load_a(i + 1, av[(i + 1) & 1]);
          __builtin_amdgcn_sched_barrier(0);
          const auto& A = av[i & 1];
          const auto& B = bring[i & 3];
          if constexpr (F2) {
            if (i & 1) mma_up2x_f2(acc_odd[0], acc_odd[1], sm[0], sm[1], A[0], A[1], B);
            else mma_up2x_f2(acc[0], acc[1], sm[0], sm[1], A[0], A[1], B);
          } else if constexpr (X3) mma_up2x_x3(acc[0], acc[1], sm[0], sm[1], A[0], A[1], B);
          else mma_unit2(acc[0], acc[1], A[0][0], A[1][0], B[0], mie_bf16());
          __builtin_amdgcn_sched_barrier(0);
        }
      } else {
        // (lane's LDS offset, step from unit to unit) of group g of sub-chunk qi: rows for every lane, corners for theirs
        auto lane_of = [&](int g, int qi, int& base, int& step) {
          const int code = (int)((strip >> (4 * g)) & 15u);
          const bool corner = code >= 3, on = !corner || (code == 3 ? at_first : at_last);
          base = on ? a_lane[0] + (corner ? jx * LS : code * RPS) + SUB * qi : ZOFF;
          step = on ? (corner ? RPS : LS) : 0;
        };
        float4 av[2][PL];
        auto load_a = [&](int at, float4 (&dst)[PL]) {
#pragma unroll
          for (int q = 0; q < PL; ++q) dst[q] = *reinterpret_cast<const float4*>(&sin[q * STAGE + at]);
        };
        int base, step, qi = 0, g = 0;
        lane_of(0, 0, base, step);
        load_a(base, av[0]);
        if (stops_at(c)) break;
        for (int left = NQW * ng; left > 0; --left) {
          const bool end = g + 1 == ng;
          const int gn = end ? 0 : g + 1, qn = left == 1 ? 0 : (end ? qi + 1 : qi);
          const TL* const gb_next = left == 1 ? ub_next : group_b(c, qn, strip_unit(gn));
          const bool corner = ((strip >> (4 * g)) & 15u) >= 3u;
          int base_n, step_n;
          lane_of(gn, qn, base_n, step_n);
#pragma unroll
          for (int t = 0; t < 4; ++t) {
            if (t == 1) seek_b(gb_next);
            load_b(bring[(t + 3) & 3]);
            // (a corner group has three units; its fourth A operand is read and not used)
            load_a(t == 3 ? base_n : base + (t == 2 && corner ? 0 : (t + 1) * step), av[(t + 1) & 1]);
            __builtin_amdgcn_sched_barrier(0);
            const auto& A = av[t & 1];
            const auto& B = bring[t];
            if (t < 3 || !corner) {
              if constexpr (F2) {
                mma_f16(sm[0], A[1], B[0]);
                mma_f16(t & 1 ? acc_odd[0] : acc[0], A[0], B[0]);
                mma_f16(sm[0], A[0], B[1]);
              } else if constexpr (X3) {
                mma_unit(sm[0], A[2], B[0], mie_bf16()); mma_unit(sm[0], A[1], B[1], mie_bf16());
                mma_unit(acc[0], A[0], B[0], mie_bf16()); mma_unit(sm[0], A[0], B[2], mie_bf16());
                mma_unit(sm[0], A[1], B[0], mie_bf16()); mma_unit(sm[0], A[0], B[1], mie_bf16());
              } else {
                mma_unit(acc[0], A[0], B[0], mie_bf16());
              }
            }
            __builtin_amdgcn_sched_barrier(0);
          }
          base = base_n; step = step_n; g = gn; qi = qn;
        }
      }
      if (NBUF == 1) __syncthreads();
      if (more) stage_store((c + 1) % NBUF, in_terms);
      note_misfit(c + 1);
      __syncthreads();
      ask_stop(c + 1);
    }
  };
  if (side == 0) contract(std::true_type());
  else contract(std::false_type());
  if constexpr (F2) {
    const float c0 = f2_unscale(groups.scale) * filt_unscale, c1 = c0 * (1.f / F2_STEP);      // exactly: powers of two, 2^-143 at the least but for sums of zeros
#pragma unroll
    for (int mb = 0; mb < 2; ++mb)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[mb][r] = fmaf(sm[mb][r], c1, (acc[mb][r] + acc_odd[mb][r]) * c0);
    // from the first chunk on that does not fit: three bf16 terms of the input and of the fp32 copy of the filter behind the two, as in k_conv_mfma.
    // us where all fit | later channels 2^8 larger | no chunk fits | three terms: 256->128 at 33x44 28.9 | 47 | 65 | 42, 128->64 at 66x88 27.6 | 37 | 44 |
    // 41, and of k_upconv2x_all 64->32 at 132x176 30.8 | 39.5 | 46 | 44.5.
    if (__builtin_expect(c_end < nch, 0)) {
      auto plainly = [&](int c_from, auto form) __attribute__((always_inline)) {
        constexpr bool THREE = decltype(form)::value == 2;
        constexpr int PA = THREE ? 3 : 2;
        auto load = [&](const TL* gb, float4 (&b)[PL]) __attribute__((always_inline)) {
#pragma unroll
          for (int q = 0; q < PL; ++q) b[q] = *reinterpret_cast<const float4*>(gb + 2 * weights + b_lane + q * (2 * cout * EPS));
        };
        auto read_x = [&](int at, float4 (&x)[PA]) __attribute__((always_inline)) {
#pragma unroll
          for (int q = 0; q < PA; ++q) x[q] = *reinterpret_cast<const float4*>(&sbuf[q * STAGE + at]);
        };
        auto unit = [&](const float4 (&b)[PL], const float4 (&x0)[PA], const float4 (&x1)[PA], auto block) __attribute__((always_inline)) {
          if constexpr (THREE) {
            float4 b3[3];
            split3_raw(b, b3);
            if constexpr (decltype(block)::value) {
              mma_up2x_x3(acc[0], acc[1], sm[0], sm[1], x0, x1, b3);
            } else {
              mma_unit(sm[0], x0[2], b3[0], mie_bf16()); mma_unit(sm[0], x0[1], b3[1], mie_bf16());
              mma_unit(acc[0], x0[0], b3[0], mie_bf16()); mma_unit(sm[0], x0[0], b3[2], mie_bf16());
              mma_unit(sm[0], x0[1], b3[0], mie_bf16()); mma_unit(sm[0], x0[0], b3[1], mie_bf16());
            }
          } else {
#pragma unroll
            for (int q = 0; q < PL; ++q) {
              mma_unit(acc[0], x0[q], b[q], float());
              if constexpr (decltype(block)::value) mma_unit(acc[1], x1[q], b[q], float());
            }
          }
        };
        for (int c = c_from; c < nch; ++c) {
          stage_load(c);
          __syncthreads();
          stage_store(0, form);
          __syncthreads();
          for (int qi = 0; qi < NQW; ++qi) {
            if (side == 0) {
              const TL* const gb = group_b(c, qi, 4 * NI * cls);
              float4 br[4][PL];
#pragma unroll
              for (int j = 0; j < 3; ++j) load(gb + j * unit_sz, br[j]);
              float4 xv[2][2][PA];
#pragma unroll
              for (int mb = 0; mb < 2; ++mb) read_x(a_lane[mb] + cls * NI * RP + SUB * qi, xv[0][mb]);
#pragma unroll 1
              for (int ky = 0; ky < NI; ++ky) {
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                  const int ahead = 4 * ky + j + 3;
                  load(gb + (ahead < 4 * NI ? ahead : 4 * NI - 1) * unit_sz, br[(j + 3) & 3]);
                  const int k = 4 * ky + j + 1 < 4 * NI ? 4 * ky + j + 1 : 0, at = (cls * NI + (k >> 2)) * RP + (k & 3) * LS + SUB * qi;
#pragma unroll
                  for (int mb = 0; mb < 2; ++mb) read_x(a_lane[mb] + at, xv[(j + 1) & 1][mb]);
                  __builtin_amdgcn_sched_barrier(0);
                  unit(br[j], xv[j & 1][0], xv[j & 1][1], std::true_type());
                }
              }
            } else {
#pragma unroll 1
              for (int g = 0; g < ng; ++g) {
                const int code = (int)((strip >> (4 * g)) & 15u);
                const bool corner = code >= 3, on = !corner || (code == 3 ? at_first : at_last);
                const int base = on ? a_lane[0] + (corner ? jx * LS : code * RPS) + SUB * qi : ZOFF, step = on ? (corner ? RPS : LS) : 0;
#pragma unroll 1
                for (int t = 0; t < (corner ? 3 : 4); ++t) {
                  float4 b[PL];
                  load(group_b(c, qi, strip_unit(g) + t), b);
                  float4 x[PA];
                  read_x(base + t * step, x);
                  unit(b, x, x, std::false_type());
                }
              }
            }
          }
        }
      };
      auto clear = [&](v16f (&v)[2]) __attribute__((always_inline)) {
#pragma unroll
        for (int mb = 0; mb < 2; ++mb)
#pragma unroll
          for (int r = 0; r < 16; ++r) v[mb][r] = 0.f;
      };
      clear(sm);
      if (filt_form >= 0.f) plainly(c_end, std::integral_constant<int, 2>());
#pragma unroll
      for (int mb = 0; mb < 2; ++mb)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[mb][r] += sm[mb][r];
      __syncthreads();
      if (tid == 0) s_f2[4] = filt_form < 0.f ? 1.f : 0.f;
      __syncthreads();
      if (groups.huge()) s_f2[4] = 1.f;
      __syncthreads();
      if (__builtin_amdgcn_readfirstlane(__float_as_int(s_f2[4])) != 0) {      // values that three bf16 terms do not hold: all of it on the fp32 instruction
        clear(acc);
        plainly(0, std::integral_constant<int, 0>());
        __syncthreads();
      }
    }
  }

  // ---- epilogue ----------------------------------------------------------------------------------------------------------
  long long off[PB];
  int co[PB];
  bool ok[PB], live[PB];
  float4 r0[PB], add[PB];
  auto fetch = [&](int h0) {
#pragma unroll
    for (int i = 0; i < PB; ++i) {
      const int idx = tid + 256 * (h0 + i);
      const int p = idx / QPP, col = 4 * (idx - p * QPP);
      const int dy = pos_y(p), dx = pos_x(p);
      ok[i] = dy < rows && dx < cols;
      live[i] = ((live_bits >> (h0 + i)) & 1u) != 0;
      off[i] = (((long long)n * hout + 2 * (y0 + dy) + py) * wout + 2 * (x0 + dx) + px) * cout + co0 + col;
      co[i] = co0 + col;
    }
    conv_epilogue_load4<T, PB>(a, off, live, r0, add);
  };
  fetch(0);      // (ahead of the exchange)
  float* red = smem + wk * (64 * CO_BLK);
#pragma unroll
  for (int mb = 0; mb < 2; ++mb)
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int p = mb * 32 + 8 * (r >> 2) + 4 * half + (r & 3);
      float s = acc[mb][r];
      if (X3 && !F2) s += sm[mb][r];
      red[p * CO_BLK + wn * 32 + l32] = s;
    }
  __syncthreads();
#pragma unroll
  for (int h0 = 0; h0 < PER; h0 += PB) {
    if (h0 > 0) fetch(h0);
    float4 s[PB];
#pragma unroll
    for (int i = 0; i < PB; ++i) {
      const int idx = tid + 256 * (h0 + i);
      float4 sum = *reinterpret_cast<const float4*>(&smem[4 * idx]);
#pragma unroll
      for (int k2 = 1; k2 < WK; ++k2) {
        const float4 part = *reinterpret_cast<const float4*>(&smem[k2 * (64 * CO_BLK) + 4 * idx]);
        sum.x += part.x; sum.y += part.y; sum.z += part.z; sum.w += part.w;
      }
      s[i] = sum;
    }
    conv_epilogue_store4<T, PB>(a, off, co, ok, s, r0, add, live);
  }
}

// The same with all four phases of a block (or strip) in one workgroup, a phase to a wave x 32 output channels, for fp32 deltas in two fp16
// terms and for bf16 ones of 64 channels (one chunk).  The window (12x12 pixels, 3 rows of 36) is loaded, added up and split once instead of
// four times, and the waves' sums do not have to meet in LDS: what layers of few channels spend their time on, whose workgroups in k_upconv2x
// are two or three chunks long between a prologue and an exchange (64->32 at 132x176, all tiles active: 1580 workgroups there, 50 us; here
// 396, 31 us, 37 with reservoir and activation, of which the matrix cores are busy for a third).
//
// fp32 sums.  With all of K in one wave the chain of roundings at the size of the sum would be four times as long, and the fp16 leading terms
// fill the accumulator's 24 bits where bf16 ones do not (in one chain 64 channels are 1.41e-7 from fp64, relative 2-norm, k_upconv2x in
// three terms 1.10e-7).  So every BL = 4 units start from zero, and are added to the total, under the MFMAs of the next four (two sets of
// accumulators), with what the addition rounds off carried on in the accumulator of the small products: 1.04e-7 at any number of
// channels (BL = 8 1.15e-7, 16 1.35e-7; without the carry 1.28, 1.27 and 1.41e-7).  Four VALU instructions a value, 128 a block, beside
// 24 MFMAs of 32 cycles.
//
// The next chunk is staged a slot at a time, its loads ten units ahead of its LDS writes (16 registers instead of 48).
template <typename T>
__global__ __launch_bounds__(256, sizeof(T) == 4 ? 2 : 3) void k_upconv2x_all(ConvArgsT<T> a, Up2xOrder od) {
  constexpr bool F2 = sizeof(T) == 4;
  typedef mie_bf16 TL;
  constexpr int PL = F2 ? 2 : 1, GPS = F2 ? 2 : 1;           // operand planes, 16-byte loads of a slot
  constexpr int NBUF = F2 ? 2 : 1;                           // (bf16: one chunk)
  constexpr int EPS = 8, SUB = 16, IT = 12, CC = F2 ? 32 : 64, LS = CC + EPS, Q4 = CC / EPS;
  constexpr int NLD = (IT * IT * Q4 + 255) / 256;
  constexpr int RP = row_pitch_dw(IT, LS / 2, 1) * 2;
  constexpr int ZOFF = IT * RP, STAGE = ZOFF + LS;           // the zero pixel behind the tile
  constexpr int SPX = STRIP + 4, RPS = SPX * LS;
  static_assert(3 * SPX <= IT * IT && 3 * RPS <= ZOFF, "a strip stages less than a block");
  constexpr int NQ = CC / SUB, UPC = 16 * NQ, BL = 4;
  constexpr int RING = F2 ? 4 : 8, PD = RING - 1, AHEAD = F2 ? 2 : 4;      // units of the filter and of LDS in registers
  static_assert(UPC % (2 * BL) == 0, "a chunk ends with a block of the odd accumulators");
  constexpr int CO_BLK = 32, RED = 4 * 64 * CO_BLK;
  constexpr int STAGE_F = NBUF * PL * STAGE / 2, SMEM = STAGE_F > RED ? STAGE_F : RED;
  static_assert(SMEM * 4 <= 65536, "LDS budget");
  __shared__ __attribute__((aligned(16))) float smem[SMEM];
  __shared__ float s_f2[F2 ? 7 : 1];                                  // as in k_upconv2x
  TL* const sbuf = reinterpret_cast<TL*>(smem);

  // the strips first, dealt out to the XCDs one by one: they are the longest of the workgroups; then the blocks as in k_upconv2x
  const int bid = blockIdx.x + conv_args_entry_zero(a);
  const int xcd = bid & 7, slot = bid >> 3, slabs = od.combos;
  const int strips = 2 * (od.strips_x + od.strips_y), all_strips = a.ts.n * strips * slabs, s8 = (all_strips + 7) >> 3;
  const int H = a.h_in, W = a.w_in, hout = a.ts.h, wout = a.ts.w;
  int side = 0, n, slab, y0, x0, rows, cols;
  if (slot >= s8) {
    const int share = (od.total + 7) >> 3, at = slot - s8, v = xcd * share + at;
    if (at >= share || v >= od.total) return;
    const int cg = mie_tile_div(v, od.per_group, od.m_group), rem = v - cg * od.per_group;
    const int it = mie_tile_div(rem, od.cpg, od.m_cpg);
    slab = cg * od.cpg + (rem - it * od.cpg);
    n = mie_tile_div(it, od.items, od.m_items);
    const int k = it - n * od.items, by = mie_tile_div(k, od.blocks_x, od.m_bx);
    y0 = 1 + 8 * by; x0 = 1 + 8 * (k - by * od.blocks_x);
    rows = H - 1 - y0 < 8 ? H - 1 - y0 : 8; cols = W - 1 - x0 < 8 ? W - 1 - x0 : 8;
  } else {
    const int v = 8 * slot + xcd;
    if (v >= all_strips) return;
    const int at = v / slabs;
    slab = v - at * slabs;
    n = at / strips;
    int k = at - n * strips;
    if (k < 2 * od.strips_x) {
      side = 1 + (k >= od.strips_x ? 1 : 0);
      x0 = STRIP * (k - (side - 1) * od.strips_x); y0 = side == 1 ? 0 : H - 1;
      rows = 1; cols = W - x0 < STRIP ? W - x0 : STRIP;
    } else {
      k -= 2 * od.strips_x;
      side = 3 + (k >= od.strips_y ? 1 : 0);
      y0 = 1 + STRIP * (k - (side - 3) * od.strips_y); x0 = side == 3 ? 0 : W - 1;
      rows = H - 1 - y0 < STRIP ? H - 1 - y0 : STRIP; cols = 1;
    }
  }
  const bool lying = side == 1 || side == 2;
  auto pos_y = [&](int p) { return side == 0 ? p >> 3 : (lying ? 0 : p); };
  auto pos_x = [&](int p) { return side == 0 ? p & 7 : (lying ? p : 0); };

  const int tid = threadIdx.x;
  const int phase = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int py = phase >> 1, px = phase & 1;
  const int l32 = lane & 31, half = lane >> 5;
  const int co0 = slab * CO_BLK, cout = a.cout;

  const int tl_y = y0 >> 2, tl_x = x0 >> 2, tl_nx = ((2 * (x0 + cols) - 1) >> 3) - tl_x + 1, tl_ny = ((2 * (y0 + rows) - 1) >> 3) - tl_y + 1;
  const int* const flags_n = reinterpret_cast<const int*>(od.flags) + (long long)n * a.ts.tiles_y * a.ts.tiles_x;
  // item g of a thread: four channels of phase g / 2 of position 32 * (g % 2) + tid / 8
  constexpr int PER = 8, PB = 4;
  int item = tid;
  auto pixel = [&](int g, int& oy, int& ox) __attribute__((always_inline)) -> bool {
    const int p = 32 * (g & 1) + (item >> 3), dy = pos_y(p), dx = pos_x(p);
    oy = 2 * (y0 + dy) + (g >> 2); ox = 2 * (x0 + dx) + ((g >> 1) & 1);
    return dy < rows && dx < cols;
  };
  const int col = 4 * (tid & 7);
  {
    const bool in = lane < tl_nx * tl_ny;
    const int f = flags_n[(tl_y + (in ? lane / tl_nx : 0)) * a.ts.tiles_x + tl_x + (in ? lane % tl_nx : 0)];
    if (__ballot((f & 1) != 0) == 0ull) {
      if (__ballot((f & 2) != 0) != 0ull)          // nothing active, something stale: zero it
        for (int g = 0; g < PER; ++g) {
          int oy, ox;
          if (!pixel(g, oy, ox)) continue;
          if ((flags_n[(oy >> 3) * a.ts.tiles_x + (ox >> 3)] & 2) != 0)
            mie_st4(a.out, (((long long)n * hout + oy) * wout + ox) * cout + co0 + col, make_float4(0.f, 0.f, 0.f, 0.f));
        }
      return;
    }
  }
  int at[PER];
  unsigned in = 0u;
#pragma unroll
  for (int g = 0; g < PER; ++g) {
    int oy, ox;
    const bool k = pixel(g, oy, ox);
    at[g] = k ? (n * hout + oy) * wout + ox : 0;
    in |= (k ? 1u : 0u) << g;
  }
  const uint8_t* const live_m = a.refresh ? nullptr : a.ts.pixmask;
  unsigned live_b[PER];
  mie_mask_ask(live_m, a.filt_mc, at, live_b);

  const bool has2 = a.x2 != nullptr;
  unsigned st_off[NLD];
  int st_lds[NLD], st_po[NLD];
  const int n_slots = (side == 0 ? IT * IT : 3 * SPX) * Q4;
#pragma unroll
  for (int i = 0; i < NLD; ++i) {
    const int slot = tid + 256 * i;
    const int q4 = slot & (Q4 - 1);
    int pix = slot / Q4, iy, ix;
    if (side == 0) {
      if (pix >= IT * IT) pix = 0;
      const int r = pix / IT, c = pix - r * IT;
      iy = y0 - 2 + r; ix = x0 - 2 + c;
      st_lds[i] = r * RP + c * LS + EPS * q4;
    } else {
      if (pix >= 3 * SPX) pix = 0;
      const int b = pix / SPX, c = pix - b * SPX;
      const int deep = (side & 1) ? b : -b, along = c - 2;
      iy = y0 + (lying ? deep : along); ix = x0 + (lying ? along : deep);
      st_lds[i] = b * RPS + c * LS + EPS * q4;
    }
    if (slot >= n_slots) st_lds[i] = CC;                     // the padding of the first pixel
    iy = iy < 0 ? 0 : (iy >= H ? H - 1 : iy);
    ix = ix < 0 ? 0 : (ix >= W ? W - 1 : ix);
    const int po = (n * H + iy) * W + ix;
    st_off[i] = ((unsigned)po * (unsigned)a.c1 + (unsigned)(EPS * q4)) * (unsigned)sizeof(T);
    st_po[i] = po;
  }
  const uint8_t* const x2m = has2 ? a.x2m : nullptr;
  unsigned b1[NLD], b2[NLD], ok1 = 0u, ok2 = 0u, live_bits = 0u;
  mie_mask_ask(a.xm, a.filt_mc, st_po, b1);
  mie_mask_ask(x2m, a.filt_mc, st_po, b2);
  const int nch = a.c1 / CC;

  float4 ra[GPS], rb[GPS];
  const T* x2p = has2 ? a.x2 : a.x;
  auto load = [&](int i, int c) __attribute__((always_inline)) {
    const char* xc = reinterpret_cast<const char*>(a.x + c * CC);
    const char* x2c = reinterpret_cast<const char*>(x2p + c * CC);
#pragma unroll
    for (int g = 0; g < GPS; ++g) {
      ra[g] = *reinterpret_cast<const float4*>(xc + st_off[i] + 16 * g);
      rb[g] = *reinterpret_cast<const float4*>(x2c + st_off[i] + 16 * g);
    }
  };
  F2Groups groups;
  auto sum = [&](int i, const float4 (&u)[GPS], const float4 (&w)[GPS], float (&f)[8]) __attribute__((always_inline)) {
    const bool k1 = (ok1 >> i) & 1u, k2 = (ok2 >> i) & 1u;
    if constexpr (F2) {
      const float ta[8] = {u[0].x, u[0].y, u[0].z, u[0].w, u[1].x, u[1].y, u[1].z, u[1].w};
      const float tb[8] = {w[0].x, w[0].y, w[0].z, w[0].w, w[1].x, w[1].y, w[1].z, w[1].w};
#pragma unroll
      for (int e = 0; e < 8; ++e) f[e] = (k1 ? ta[e] : 0.f) + (k2 ? tb[e] : 0.f);
    } else {
      const float4 z4 = make_float4(0.f, 0.f, 0.f, 0.f);
      float fa[8], fb[8];
      slot_to_f32(k1 ? u[0] : z4, fa, T());
      slot_to_f32(k2 ? w[0] : z4, fb, T());
#pragma unroll
      for (int e = 0; e < 8; ++e) f[e] = fa[e] + fb[e];
    }
  };
  auto put = [&](int i, const float (&f)[8], TL* dst, auto terms) __attribute__((always_inline)) {
    if constexpr (F2) {
      constexpr int FORM = decltype(terms)::value;
      float4 pl[FORM == 2 ? 3 : 2];
      pl[0] = make_float4(f[0], f[1], f[2], f[3]); pl[1] = make_float4(f[4], f[5], f[6], f[7]);
      if constexpr (FORM == 1) groups.terms(f, pl);
      else groups.note(f);
      if constexpr (FORM == 2) split3(f, pl);
#pragma unroll
      for (int q = 0; q < (FORM == 2 ? 3 : 2); ++q) *reinterpret_cast<float4*>(dst + q * STAGE + st_lds[i]) = pl[q];
    } else {
      *reinterpret_cast<float4*>(dst + st_lds[i]) = f32_to_slot(f, T());
    }
  };
  auto store = [&](int i, TL* dst, auto terms) __attribute__((always_inline)) {
    float f[8];
    sum(i, ra, rb, f);
    put(i, f, dst, terms);
  };
  auto stage = [&](int c, TL* dst, auto terms) __attribute__((always_inline)) {      // (where nothing else is to be done meanwhile)
#pragma unroll
    for (int i = 0; i < NLD; ++i) {
      load(i, c);
      store(i, dst, terms);
    }
  };

  unsigned strip = 0u;
  int ng = 0;
  {
    auto add = [&](bool on, int code) {
      strip |= on ? (unsigned)code << (4 * ng) : 0u;
      ng += on ? 1 : 0;
    };
    add(true, 0); add(true, 1); add(true, 2);
    add(lying && x0 == 0, 3); add(lying && x0 + cols == W, 4);
  }
  const int u_side = side == 1 ? U_TOP : (side == 2 ? U_BOTTOM : (side == 3 ? U_LEFT : U_RIGHT));
  const int jx = 2 - px;
  int a_lane[2];
#pragma unroll
  for (int mb = 0; mb < 2; ++mb) {
    const int p = mb * 32 + l32;
    a_lane[mb] = (side == 0 ? ((p >> 3) + py) * RP + ((p & 7) + px) * LS : (l32 + (lying ? px : py)) * LS) + EPS * half;
  }
  const bool at_first = l32 == 0, at_last = l32 == cols - 1;
  const int b_lane = (half * cout + l32) * EPS;
  const int unit_sz = PL * 2 * cout * EPS;
  const TL* const filt = reinterpret_cast<const TL*>(a.filt_mc) + co0 * EPS;
  auto group_b = [&](int c, int qi, int unit) -> const TL* {
    return filt + ((long long)(phase * od.nci + c * NQ + qi) * UNITS + unit) * unit_sz;
  };
  auto strip_unit = [&](int g) { return u_side + 4 * (int)((strip >> (4 * g)) & 15u); };
  const TL* bp;
  auto seek_b = [&](const TL* gb) { bp = gb + b_lane; };
  auto load_b = [&](float4 (&bv)[PL]) __attribute__((always_inline)) {
#pragma unroll
    for (int q = 0; q < PL; ++q) {
      bv[q] = *reinterpret_cast<const float4*>(bp);
      bp += 2 * cout * EPS;
    }
  };
  auto first_b = [&](int c) { return group_b(c, 0, side == 0 ? 0 : strip_unit(0)); };

  v16f zero, acc[2], tot[F2 ? 2 : 1], odd[F2 ? 2 : 1], sm[F2 ? 2 : 1];
#pragma unroll
  for (int r = 0; r < 16; ++r) zero[r] = 0.f;
#pragma unroll
  for (int mb = 0; mb < 2; ++mb) {
    acc[mb] = zero;
    if constexpr (F2) tot[mb] = zero, odd[mb] = zero, sm[mb] = zero;
  }
  const long long weights = 4LL * UNITS * a.c1 * cout;
  float filt_unscale = 1.f;
  float filt_form = 1.f;
  if constexpr (F2) {
    const float* const end = f2_filter_end(a.filt_mc, weights);
    filt_unscale = end[0];
    filt_form = end[1] - end[2];
  }
  int c_end = nch;
  auto note_misfit = [&](int c) __attribute__((always_inline)) {
    if constexpr (F2) {
      s_f2[groups.misfit() ? 4 + (c & 1) : 6] = 1.f;      // (without a branch)
    }
  };
  float stop = 0.f;
  auto ask_stop = [&](int c) __attribute__((always_inline)) {
    if constexpr (F2) stop = s_f2[4 + (c & 1)];
  };
  auto stops_at = [&](int c) __attribute__((always_inline)) {
    if constexpr (F2) {
      if (__builtin_expect(__builtin_amdgcn_readfirstlane(__float_as_int(stop)) != 0, 0)) {
        c_end = c;
        return true;
      }
    }
    return false;
  };
  auto flush = [&](const v16f (&from)[2], int mb, int r) __attribute__((always_inline)) {      // (F2)
    const float t = tot[mb][r], x = from[mb][r], u = t + x;
    sm[mb][r] = fmaf(x - (u - t), F2_STEP, sm[mb][r]);      // (exactly what is lost where |x| <= |t|)
    tot[mb][r] = u;
  };
  float4 bring[RING][PL];
  seek_b(first_b(0));
  float4 fa[NLD][GPS], fb[NLD][GPS];
#pragma unroll
  for (int i = 0; i < NLD; ++i)
#pragma unroll
    for (int g = 0; g < GPS; ++g) {
      fa[i][g] = *reinterpret_cast<const float4*>(reinterpret_cast<const char*>(a.x) + st_off[i] + 16 * g);
      fb[i][g] = *reinterpret_cast<const float4*>(reinterpret_cast<const char*>(x2p) + st_off[i] + 16 * g);
    }
#pragma unroll
  for (int i = 0; i < PD; ++i) load_b(bring[i]);
  mie_mask_asked();
  ok1 = mie_mask_take(a.xm, b1, ~0u);
  ok2 = mie_mask_take(x2m, b2, has2 ? ~0u : 0u);
  live_bits = mie_mask_take(live_m, live_b, in);
  for (int i = tid; i < NBUF * PL * (LS / EPS); i += 256) {
    const int pl = i / (LS / EPS);
    *reinterpret_cast<float4*>(sbuf + pl * STAGE + ZOFF + EPS * (i - pl * (LS / EPS))) = make_float4(0.f, 0.f, 0.f, 0.f);
  }
  const auto in_terms = std::integral_constant<int, 1>();
  {
    float f[NLD][8];
#pragma unroll
    for (int i = 0; i < NLD; ++i) sum(i, fa[i], fb[i], f[i]);
    if constexpr (F2) {
      float m = 0.f;
#pragma unroll
      for (int i = 0; i < NLD; ++i) m = __builtin_elementwise_maximum(m, f2_amax8(f[i]));
      m = f2_wave_max(m);
      if (lane == 0) s_f2[phase] = m;
      if (tid < 2) s_f2[4 + tid] = 0.f;
      __syncthreads();
      groups.start(f2_scale(__int_as_float(__builtin_amdgcn_readfirstlane(
          __float_as_int(__builtin_elementwise_maximum(f2_max3(s_f2[0], s_f2[1], s_f2[2]), s_f2[3]))))));
    }
#pragma unroll
    for (int i = 0; i < NLD; ++i) put(i, f[i], sbuf, in_terms);
  }
  note_misfit(0);
  __syncthreads();
  if (F2 && filt_form != 1.f) c_end = 0;
  ask_stop(0);

  if (side == 0) {
    const TL* sin = sbuf;
    TL* snext = sbuf + (NBUF - 1) * PL * STAGE;
    float4 av[AHEAD][2][PL];
    auto load_a = [&](const TL* s, int u, float4 (&dst)[2][PL]) __attribute__((always_inline)) {
      const int qi = u / 16, k = u % 16;
#pragma unroll
      for (int mb = 0; mb < 2; ++mb)
#pragma unroll
        for (int q = 0; q < PL; ++q)
          dst[mb][q] = *reinterpret_cast<const float4*>(&s[q * STAGE + a_lane[mb] + (k >> 2) * RP + (k & 3) * LS + SUB * qi]);
    };
#pragma unroll
    for (int i = 0; i < AHEAD - 1; ++i) load_a(sin, i, av[i]);
    for (int c = 0; c < c_end; ++c) {
      const int cn = c + 1 < nch ? c + 1 : c;
      if (stops_at(c)) break;
#pragma unroll
      for (int i = 0; i < UPC; ++i) {
        const int ip = i + PD;
        if (ip == UPC) seek_b(first_b(cn));
        else if (ip % 16 == 0) seek_b(group_b(c, ip / 16, 0));
        load_b(bring[ip % RING]);
        if (i + AHEAD - 1 < UPC) load_a(sin, i + AHEAD - 1, av[(i + AHEAD - 1) % AHEAD]);
        __builtin_amdgcn_sched_barrier(0);
        const auto& A = av[i % AHEAD];
        const auto& B = bring[i % RING];
        if constexpr (F2) {
          v16f (&now)[2] = (i / BL) % 2 ? odd : acc;
          v16f (&was)[2] = (i / BL) % 2 ? acc : odd;
          if (i % BL == 0) now[0] = zero, now[1] = zero;
          mma_f16(now[0], A[0][0], B[0]); mma_f16(now[1], A[1][0], B[0]);
          mma_f16(sm[0], A[0][1], B[0]);  mma_f16(sm[1], A[1][1], B[0]);
          mma_f16(sm[0], A[0][0], B[1]);  mma_f16(sm[1], A[1][0], B[1]);
#pragma unroll
          for (int e = (32 / BL) * (i % BL); e < (32 / BL) * (i % BL + 1); ++e) flush(was, e / 16, e % 16);
          static_assert(!F2 || NLD == 3, "the slots' places in the units");
          if (i % 10 == 9) store(i / 10, snext, in_terms);
          if (i % 10 == 0 && i < 30) load(i / 10, cn);
        } else {
          mma_unit2(acc[0], acc[1], A[0][0], A[1][0], B[0], mie_bf16());
        }
        __builtin_amdgcn_sched_barrier(0);
        if (F2 && i == UPC - 2) {
          note_misfit(c + 1);
          __syncthreads();
          ask_stop(c + 1);
          load_a(snext, 0, av[0]);
          __builtin_amdgcn_sched_barrier(0);
        }
      }
      TL* const t = const_cast<TL*>(sin);
      sin = snext;
      snext = t;
    }
    if constexpr (F2) {
#pragma unroll
      for (int e = 0; e < 32; ++e) flush(odd, e / 16, e % 16);
    } else {
      __syncthreads();
    }
  } else {
    if constexpr (PD > 3) seek_b(first_b(0) + 3 * unit_sz);
    auto lane_of = [&](int g, int qi, int& base, int& step) {
      const int code = (int)((strip >> (4 * g)) & 15u);
      const bool corner = code >= 3, on = !corner || (code == 3 ? at_first : at_last);
      base = on ? a_lane[0] + (corner ? jx * LS : code * RPS) + SUB * qi : ZOFF;
      step = on ? (corner ? RPS : LS) : 0;
    };
    for (int c = 0; c < c_end; ++c) {
      const bool more = c + 1 < nch;
      const int cn = more ? c + 1 : c;
      const TL* sin = sbuf + c % NBUF * (PL * STAGE);
      if (stops_at(c)) break;
      if constexpr (F2) {
        if (more) stage(cn, sbuf + (c + 1) % NBUF * (PL * STAGE), in_terms);
      }
      float4 av[2][PL];
      auto load_a = [&](int at, float4 (&dst)[PL]) __attribute__((always_inline)) {
#pragma unroll
        for (int q = 0; q < PL; ++q) dst[q] = *reinterpret_cast<const float4*>(&sin[q * STAGE + at]);
      };
      int base, step, qi = 0, g = 0;
      lane_of(0, 0, base, step);
      load_a(base, av[0]);
      for (int left = NQ * ng; left > 0; --left) {
        const bool last = g + 1 == ng;
        const int gn = last ? 0 : g + 1, qn = left == 1 ? 0 : (last ? qi + 1 : qi);
        const TL* const gb_next = left == 1 ? first_b(cn) : group_b(c, qn, strip_unit(gn));
        const bool corner = ((strip >> (4 * g)) & 15u) >= 3u;
        int base_n, step_n;
        lane_of(gn, qn, base_n, step_n);
        if (F2) acc[0] = zero;
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          if (t == 1) seek_b(gb_next);
          load_b(bring[(t + 3) & 3]);
          load_a(t == 3 ? base_n : base + (t == 2 && corner ? 0 : (t + 1) * step), av[(t + 1) & 1]);
          __builtin_amdgcn_sched_barrier(0);
          const auto& A = av[t & 1];
          const auto& B = bring[t];
          if (t < 3 || !corner) {
            if constexpr (F2) {
              mma_f16(sm[0], A[1], B[0]);
              mma_f16(acc[0], A[0], B[0]);
              mma_f16(sm[0], A[0], B[1]);
            } else {
              mma_unit(acc[0], A[0], B[0], mie_bf16());
            }
          }
          __builtin_amdgcn_sched_barrier(0);
        }
        if constexpr (F2) {
#pragma unroll
          for (int r = 0; r < 16; ++r) flush(acc, 0, r);
        }
        base = base_n; step = step_n; g = gn; qi = qn;
      }
      note_misfit(c + 1);
      __syncthreads();
      ask_stop(c + 1);
    }
  }
  if constexpr (F2) {
    const float c0 = f2_unscale(groups.scale) * filt_unscale, c1 = c0 * (1.f / F2_STEP);      // exactly: powers of two, 2^-143 at the least but for sums of zeros
#pragma unroll
    for (int mb = 0; mb < 2; ++mb)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[mb][r] = fmaf(sm[mb][r], c1, tot[mb][r] * c0);
  }
  if constexpr (F2) {
    // from the first chunk on that does not fit: as in k_upconv2x
    if (__builtin_expect(c_end < nch, 0)) {
      auto plainly = [&](int c_from, auto form) __attribute__((always_inline)) {
        constexpr bool THREE = decltype(form)::value == 2;
        constexpr int PA = THREE ? 3 : 2;
        auto read = [&](const TL* gb, float4 (&b)[PL]) __attribute__((always_inline)) {
#pragma unroll
          for (int q = 0; q < PL; ++q) b[q] = *reinterpret_cast<const float4*>(gb + 2 * weights + b_lane + q * (2 * cout * EPS));
        };
        auto read_x = [&](int at, float4 (&x)[PA]) __attribute__((always_inline)) {
#pragma unroll
          for (int q = 0; q < PA; ++q) x[q] = *reinterpret_cast<const float4*>(&sbuf[q * STAGE + at]);
        };
        auto unit = [&](const float4 (&b)[PL], const float4 (&x0)[PA], const float4 (&x1)[PA], auto block) __attribute__((always_inline)) {
          if constexpr (THREE) {
            float4 b3[3];
            split3_raw(b, b3);
            if constexpr (decltype(block)::value) {
              mma_up2x_x3(acc[0], acc[1], sm[0], sm[1], x0, x1, b3);
            } else {
              mma_unit(sm[0], x0[2], b3[0], mie_bf16()); mma_unit(sm[0], x0[1], b3[1], mie_bf16());
              mma_unit(acc[0], x0[0], b3[0], mie_bf16()); mma_unit(sm[0], x0[0], b3[2], mie_bf16());
              mma_unit(sm[0], x0[1], b3[0], mie_bf16()); mma_unit(sm[0], x0[0], b3[1], mie_bf16());
            }
          } else {
#pragma unroll
            for (int q = 0; q < PL; ++q) {
              mma_unit(acc[0], x0[q], b[q], float());
              if constexpr (decltype(block)::value) mma_unit(acc[1], x1[q], b[q], float());
            }
          }
        };
        for (int c = c_from; c < nch; ++c) {
          __syncthreads();
          stage(c, sbuf, form);
          if (tid < PA * (LS / EPS)) {
            const int pl = tid / (LS / EPS);
            *reinterpret_cast<float4*>(sbuf + pl * STAGE + ZOFF + EPS * (tid - pl * (LS / EPS))) = make_float4(0.f, 0.f, 0.f, 0.f);
          }
          __syncthreads();
          for (int qi = 0; qi < NQ; ++qi) {
            if (side == 0) {
              const TL* const gb = group_b(c, qi, 0);
              float4 br[4][PL];
#pragma unroll
              for (int j = 0; j < 3; ++j) read(gb + j * unit_sz, br[j]);
              float4 xv[2][2][PA];
#pragma unroll
              for (int mb = 0; mb < 2; ++mb) read_x(a_lane[mb] + SUB * qi, xv[0][mb]);
#pragma unroll 1
              for (int ky = 0; ky < 4; ++ky) {
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                  const int ahead = 4 * ky + j + 3;
                  read(gb + (ahead < 16 ? ahead : 15) * unit_sz, br[(j + 3) & 3]);
                  const int k = (4 * ky + j + 1) & 15, at = (k >> 2) * RP + (k & 3) * LS + SUB * qi;
#pragma unroll
                  for (int mb = 0; mb < 2; ++mb) read_x(a_lane[mb] + at, xv[(j + 1) & 1][mb]);
                  __builtin_amdgcn_sched_barrier(0);
                  unit(br[j], xv[j & 1][0], xv[j & 1][1], std::true_type());
                }
              }
            } else {
#pragma unroll 1
              for (int g = 0; g < ng; ++g) {
                const int code = (int)((strip >> (4 * g)) & 15u);
                const bool corner = code >= 3, on = !corner || (code == 3 ? at_first : at_last);
                const int base = on ? a_lane[0] + (corner ? jx * LS : code * RPS) + SUB * qi : ZOFF, step = on ? (corner ? RPS : LS) : 0;
#pragma unroll 1
                for (int t = 0; t < (corner ? 3 : 4); ++t) {
                  float4 b[PL];
                  read(group_b(c, qi, strip_unit(g) + t), b);
                  float4 x[PA];
                  read_x(base + t * step, x);
                  unit(b, x, x, std::false_type());
                }
              }
            }
          }
        }
      };
      sm[0] = sm[1] = zero;
      if (filt_form >= 0.f) plainly(c_end, std::integral_constant<int, 2>());
#pragma unroll
      for (int mb = 0; mb < 2; ++mb)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[mb][r] += sm[mb][r];
      __syncthreads();
      if (tid == 0) s_f2[4] = filt_form < 0.f ? 1.f : 0.f;
      __syncthreads();
      if (groups.huge()) s_f2[4] = 1.f;
      __syncthreads();
      if (__builtin_amdgcn_readfirstlane(__float_as_int(s_f2[4])) != 0) {      // values that three bf16 terms do not hold: all of it on the fp32 instruction
        acc[0] = acc[1] = zero;
        plainly(0, std::integral_constant<int, 0>());
        __syncthreads();
      }
    }
  }
  float* const red = smem + phase * (64 * CO_BLK);
  // ---- epilogue: as in k_upconv2x, but that every wave parks whole sums ------------------------------------------------------
  long long off[PB];
  int co[PB];
  bool ok[PB], live[PB];
  float4 r0[PB], add[PB];
  auto fetch = [&](int h0) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < PB; ++i) {
      int oy, ox;
      ok[i] = pixel(h0 + i, oy, ox);
      live[i] = ((live_bits >> (h0 + i)) & 1u) != 0;
      co[i] = co0 + 4 * (item & 7);
      off[i] = (((long long)n * hout + oy) * wout + ox) * cout + co[i];
    }
    conv_epilogue_load4<T, PB>(a, off, live, r0, add);
  };
  asm volatile("" : "+v"(item));      // (its places anew: kept from the start they would be spilled across the contraction)
  fetch(0);
#pragma unroll
  for (int mb = 0; mb < 2; ++mb)
#pragma unroll
    for (int r = 0; r < 16; ++r) red[(mb * 32 + 8 * (r >> 2) + 4 * half + (r & 3)) * CO_BLK + l32] = acc[mb][r];
  __syncthreads();
#pragma unroll
  for (int h0 = 0; h0 < PER; h0 += PB) {
    if (h0 > 0) fetch(h0);
    float4 s[PB];
#pragma unroll
    for (int i = 0; i < PB; ++i) s[i] = *reinterpret_cast<const float4*>(&smem[4 * (tid + 256 * (h0 + i))]);
    conv_epilogue_store4<T, PB>(a, off, co, ok, s, r0, add, live);
  }
}

// (WN 0: k_upconv2x_all)
template <typename T, int WN, int AR>
void launch_one(const ConvArgsT<T>& a, Up2xOrder od, hipStream_t st) {
  od.combos = WN == 0 ? a.cout / 32 : 4 * (a.cout / (32 * WN));
  if (WN == 0) od.items = od.blocks_y * od.blocks_x;      // (the strips have places of their own)
  od.total = a.ts.n * od.items * od.combos;
  // Launch order: the (phase, slab) pairs in `groups` parts.  Every part of the filter then reaches 8 / groups of the eight
  // L2s and the input all of them `groups` times; the split that moves the least is taken.
  const double filt = 4.0 * 16 * a.c1 * a.cout * (AR == 2 ? 4 : AR == 1 ? 6 : 2);
  const double in = (double)a.ts.n * a.h_in * a.w_in * a.c1 * sizeof(T) * (a.x2 ? 2 : 1);
  double best = 8 * filt + in;
  od.groups = 1;
  for (int g = 2; g <= 8 && od.combos % g == 0; g *= 2)
    if (8 / g * filt + g * in < best) { best = 8 / g * filt + g * in; od.groups = g; }
  od.cpg = od.combos / od.groups;
  od.per_group = a.ts.n * od.items * od.cpg;
  od.m_group = mie_tile_magic(od.total, od.per_group);
  od.m_cpg = mie_tile_magic(od.per_group, od.cpg);
  od.m_items = mie_tile_magic((long long)a.ts.n * od.items, od.items);
  od.m_bx = od.blocks_x > 0 ? mie_tile_magic(od.items, od.blocks_x) : 0u;
  if constexpr (WN == 0) {
    const int strips = a.ts.n * 2 * (od.strips_x + od.strips_y) * od.combos;
    hipLaunchKernelGGL(k_upconv2x_all<T>, dim3(8 * ((od.total + 7) / 8 + (strips + 7) / 8)), dim3(256), 0, st, a, od);
  } else {
    hipLaunchKernelGGL((k_upconv2x<T, WN, AR>), dim3(8 * ((od.total + 7) / 8)), dim3(256), 0, st, a, od);
  }
}

// Slab width of k_upconv2x, by how many rounds of workgroups it takes.  A 64-column workgroup takes 1.75 times as long as a 32-column one.
//   * fp32, three terms: one workgroup fills a CU's matrix cores (two take twice as long), so a round is 256: 64 columns where they need half
//     the rounds or close to it, which leaves 32 columns up to one round (256->128 at 20x20: 26 us against 39) and in the third (at
//     42x46, 608 of them: 68 against 78; at 33x44, 480: 48 against 45; at 60x80 134 against 122).
//   * two terms: 64 columns from one round on (256->128 at 25x35 29.9 against 27.7, at 42x46 45.4 and 46.5, 128->64 at 80x100 48.3 and 45.1;
//     at 20x20 21.8 against 28.1).
//   * bf16: workgroups are short and three of a CU hide each other's latencies, so 64 columns start where 32 no longer fit one round of
//     768 (128->64 at 66x74, 656 of them: 15.7 against 17.2; at 66x88, 784: 20.4 against 17.7), 128 columns, which read the input least,
//     where they make more than a round themselves (256->128 at 8x60x80: 246 against 217; at 4x60x80, 1440: 126 against 116; at 3x60x80,
//     1080: 92 either way; at 8x30x40, 832: 76 against 83).
//
// k_upconv2x_all or k_upconv2x (wgs: of 32 columns, of the latter):
//   * fp32: where the latter, in three terms, needs more workgroups than two to a CU, and the layer has 64 or 96 channels.  64->32 at 80x112
//     (608 of them) 22.2 -> 19.1 us, at 132x176 (1584) 50 -> 31, at 240x320 137 -> 87; 64->64 at 64x64 (576) 22 -> 18.8, 96->32 at 96x96
//     31 -> 24.4; at 72x80 (400) 15.7 against 18.1.  (k_upconv2x in two terms would be 1.13 and 1.05 times as far from fp64 with 64 and 96
//     channels.)  From 128 channels on, in two terms either way, a workgroup here is longer than the launch is wide: 128->64 at 66x88
//     29.3 against 32, at 120x160 78 against 87, 256->128 at 60x80 86 against 96.  In one chunk of 32 channels three terms are as near:
//     9.94e-8 and 1.00e-7.  Planes of two rows or columns are all strips.
//   * bf16: 64 channels, from more workgroups here than CUs on.  (For calls of this form; networks keep the list-driven one for these
//     layers, which holds a + b in 32 bits up to the blend.)
bool up2x_all(int c, long long wgs, const Up2xOrder& od, bool bf) {
  return (bf ? c == 64 && wgs > 1024 : c >= 64 && c < 128 && wgs > 512) && od.blocks_y * od.blocks_x > 0;
}

template <typename T>
void launch_up2x(const ConvArgsT<T>& a, Up2xOrder od, hipStream_t st) {
  const int cout = a.cout;
  const long long wgs = (long long)a.ts.n * od.items * 4 * (cout / 32);
  if constexpr (sizeof(T) == 4) {
    const bool wide = cout % 64 == 0 && wgs > 256 && (wgs <= 512 || wgs > 768 || a.x3 == 2);
    if (a.x3 == 2 && up2x_all(a.c1, wgs, od, false)) launch_one<T, 0, 2>(a, od, st);
    else if (a.x3 == 2) wide ? launch_one<T, 2, 2>(a, od, st) : launch_one<T, 1, 2>(a, od, st);
    else wide ? launch_one<T, 2, 1>(a, od, st) : launch_one<T, 1, 1>(a, od, st);
  } else {
    if (up2x_all(a.c1, wgs, od, true)) launch_one<T, 0, 0>(a, od, st);
    else if (cout % 128 == 0 && wgs / 4 >= 1024) launch_one<T, 4, 0>(a, od, st);
    else if (cout % 64 == 0 && wgs > 768) launch_one<T, 2, 0>(a, od, st);
    else launch_one<T, 1, 0>(a, od, st);
  }
}

void up2x_items(Up2xOrder& od, int h, int w) {
  od.blocks_y = (h - 2 + 7) / 8; od.blocks_x = (w - 2 + 7) / 8;
  od.strips_x = mie_div_up(w, STRIP); od.strips_y = mie_div_up(h - 2, STRIP);
  od.items = od.blocks_y * od.blocks_x + 2 * od.strips_x + 2 * od.strips_y;
}

template <typename T>
int up2x_impl(const char* who, const void* x, const uint8_t* xm, const void* x2, const uint8_t* x2m, int c, int h, int w,
              const void* filter_up, int cout, const float* bias, const mie_tileset* out, void* out_delta, const void* addend,
              float* reservoir, int act_kind, float slope, bool refresh, int terms, void* stream) {
  const int rc = mie_check_tileset(out, who);
  if (rc != MIE_OK) return rc;
  MIE_REQUIRE(x != nullptr && filter_up != nullptr && out_delta != nullptr, MIE_ERR_INVALID_ARG,
              "%s: NULL pointer (a, filter_up and the output are required)", who);
  MIE_REQUIRE(x2 != nullptr || x2m == nullptr, MIE_ERR_INVALID_ARG, "%s: mask of absent b", who);
  MIE_REQUIRE(c > 0 && cout > 0 && h > 0 && w > 0, MIE_ERR_INVALID_ARG, "%s: sizes out of range (c=%d cout=%d h=%d w=%d)", who, c,
              cout, h, w);
  MIE_REQUIRE(c % (sizeof(T) == 4 ? 32 : 64) == 0 && cout % 32 == 0, MIE_ERR_UNSUPPORTED,
              "%s: needs c %% %d == 0 and cout %% 32 == 0 (c=%d cout=%d)", who, sizeof(T) == 4 ? 32 : 64, c, cout);
  MIE_REQUIRE(h >= 2 && w >= 2, MIE_ERR_UNSUPPORTED, "%s: planes of at least 2x2 pixels (%dx%d)", who, h, w);
  MIE_REQUIRE(out->h == 2 * h && out->w == 2 * w, MIE_ERR_INVALID_ARG, "%s: the tile set is (%d,%d), twice the input is (%d,%d)", who,
              out->h, out->w, 2 * h, 2 * w);
  MIE_REQUIRE((long long)out->n * h * w * c * (long long)sizeof(T) < 0xffffff00LL && (long long)out->n * out->h * out->w < 0x7fffffffLL &&
                  (long long)c * cout < (1LL << 24),
              MIE_ERR_CAPACITY, "%s: tensor too large", who);
  MIE_REQUIRE(mie_aligned(x, 16) && mie_aligned(x2, 16) && mie_aligned(filter_up, 16) && mie_aligned(out_delta, 16) &&
                  mie_aligned(addend, 16) && mie_aligned(reservoir, 16) && mie_aligned(bias, 4),
              MIE_ERR_INVALID_ARG, "%s: buffers must be 16-byte aligned (bias: 4)", who);
  MIE_REQUIRE(act_kind >= MIE_ACT_NONE && act_kind <= MIE_ACT_TANH, MIE_ERR_UNSUPPORTED, "%s: unknown activation %d", who, act_kind);
  MIE_REQUIRE(refresh || reservoir != nullptr || act_kind == MIE_ACT_NONE, MIE_ERR_INVALID_ARG, "%s: activation %d needs a reservoir",
              who, act_kind);
  MIE_REQUIRE(x != out_delta && x2 != out_delta && addend != out_delta, MIE_ERR_INVALID_ARG, "%s: inputs must not alias the output", who);
  ConvArgsT<T> a = {};
  a.x = (const T*)x; a.xm = xm; a.c1 = c; a.x2 = (const T*)x2; a.x2m = x2m; a.c2 = x2 ? c : 0;
  a.h_in = h; a.w_in = w; a.cin_total = c; a.filt_mc = (const T*)filter_up; a.pad = 2; a.cout = cout;
  a.out = (T*)out_delta; a.res = reservoir; a.act = act_kind; a.slope = slope; a.addend = (const T*)addend;
  a.refresh = refresh ? 1 : 0; a.bias = bias;
  a.x3 = terms;
  a.ts = mie_dev_tileset(out);
  Up2xOrder od = {};
  od.flags = (const uint32_t*)out->flags;
  up2x_items(od, h, w);
  od.nci = c / 16;
  MIE_REQUIRE((long long)out->n * od.items * 4 * (cout / 32) < 0x7ffffff0LL, MIE_ERR_CAPACITY, "%s: tensor too large", who);
  if constexpr (sizeof(T) == 2) {
    // many items of 128 -> 64 channels: the inner positions in a persistent kernel, the strips here
    if (mie_launch_upconv2x_rows(a, od.flags, (hipStream_t)stream)) {
      od.blocks_y = od.blocks_x = 0;
      od.items = 2 * od.strips_x + 2 * od.strips_y;
    }
  }
  launch_up2x<T>(a, od, (hipStream_t)stream);
  return mie_check_launch(who);
}

}  // namespace

extern "C" int mie_pack_filter_up2x(const float* filter, int cin, int cout, void* packed, int dtype, void* stream) {
  const char* who = "mie_pack_filter_up2x";
  mie_clear_error();
  MIE_REQUIRE(filter != nullptr && packed != nullptr && (const void*)filter != packed, MIE_ERR_INVALID_ARG,
              "%s: filter and packed must be given and differ", who);
  MIE_REQUIRE(dtype == MIE_DTYPE_BF16 || dtype == MIE_DTYPE_F32_BF16X3 || dtype == MIE_DTYPE_F32_F16X2, MIE_ERR_UNSUPPORTED, "%s: no combined filter of dtype %d", who, dtype);
  MIE_REQUIRE(cin > 0 && cout > 0 && cin % 16 == 0 && cout % 32 == 0 && (long long)cin * cout < (1LL << 24), MIE_ERR_UNSUPPORTED,
              "%s: needs cin %% 16 == 0 and cout %% 32 == 0 (cin=%d cout=%d)", who, cin, cout);
  MIE_REQUIRE(mie_aligned(filter, 4) && mie_aligned(packed, 16), MIE_ERR_INVALID_ARG, "%s: packed must be 16-byte aligned", who);
  const dim3 grid((unsigned)((4LL * UNITS * cin * cout + 255) / 256));
  if (dtype == MIE_DTYPE_F32_F16X2) {
    const long long groups = 4LL * UNITS * (cin / 8) * cout;
    const int blocks = mie_f2_blocks(groups);
    hipLaunchKernelGGL(k_f2_up2x_values, dim3(blocks), dim3(256), 0, (hipStream_t)stream, filter, mie_f2_values(packed, groups),
                       mie_f2_parts(packed, groups), groups, cin, cout);
    mie_f2_split(packed, groups, blocks, cout, (hipStream_t)stream);
  } else if (dtype == MIE_DTYPE_BF16)
    hipLaunchKernelGGL(k_pack_up2x<1>, grid, dim3(256), 0, (hipStream_t)stream, filter, (mie_bf16*)packed, cin, cout);
  else
    hipLaunchKernelGGL(k_pack_up2x<3>, grid, dim3(256), 0, (hipStream_t)stream, filter, (mie_bf16*)packed, cin, cout);
  return mie_check_launch(who);
}

extern "C" int mie_upconv2x_masked(const void* a, const uint8_t* amask, const void* b, const uint8_t* bmask, int c, int h_in,
                                   int w_in, const void* filter_up, int cout, const mie_tileset* out, void* out_delta,
                                   const void* addend, float* reservoir, int act_kind, float slope, int dtype, void* stream) {
  const char* who = "mie_upconv2x_masked";
  mie_clear_error();
  MIE_REQUIRE(dtype == MIE_DTYPE_BF16 || dtype == MIE_DTYPE_F32_BF16X3 || dtype == MIE_DTYPE_F32_F16X2, MIE_ERR_UNSUPPORTED, "%s: dtype %d not implemented", who, dtype);
  if (dtype == MIE_DTYPE_BF16)
    return up2x_impl<mie_bf16>(who, a, amask, b, bmask, c, h_in, w_in, filter_up, cout, nullptr, out, out_delta, addend, reservoir,
                               act_kind, slope, false, 0, stream);
  return up2x_impl<float>(who, a, amask, b, bmask, c, h_in, w_in, filter_up, cout, nullptr, out, out_delta, addend, reservoir,
                          act_kind, slope, false, dtype == MIE_DTYPE_F32_F16X2 ? 2 : 1, stream);
}

extern "C" int mie_upconv2x_refresh(const void* a, const void* b, int c, int h_in, int w_in, const void* filter_up, int cout,
                                    const float* bias, const mie_tileset* out, void* out_dense, float* reservoir, int act_kind,
                                    float slope, int dtype, void* stream) {
  const char* who = "mie_upconv2x_refresh";
  mie_clear_error();
  MIE_REQUIRE(dtype == MIE_DTYPE_BF16 || dtype == MIE_DTYPE_F32_BF16X3 || dtype == MIE_DTYPE_F32_F16X2, MIE_ERR_UNSUPPORTED, "%s: dtype %d not implemented", who, dtype);
  if (dtype == MIE_DTYPE_BF16)
    return up2x_impl<mie_bf16>(who, a, nullptr, b, nullptr, c, h_in, w_in, filter_up, cout, bias, out, out_dense, nullptr, reservoir,
                               act_kind, slope, true, 0, stream);
  return up2x_impl<float>(who, a, nullptr, b, nullptr, c, h_in, w_in, filter_up, cout, bias, out, out_dense, nullptr, reservoir,
                          act_kind, slope, true, dtype == MIE_DTYPE_F32_F16X2 ? 2 : 1, stream);
}

extern "C" int mie_all_phases_upconv2x(int n, int h_in, int w_in, int c, int cout, int dtype) {
  const bool bf = dtype == MIE_DTYPE_BF16;
  if (n <= 0 || h_in < 2 || w_in < 2 || c <= 0 || cout <= 0 || c % 32 != 0 || cout % 32 != 0 || !(bf || dtype == MIE_DTYPE_F32_F16X2)) return 0;
  Up2xOrder od = {};
  up2x_items(od, h_in, w_in);
  return up2x_all(c, (long long)n * od.items * 4 * (cout / 32), od, bf) ? 1 : 0;
}

extern "C" int mie_f16x2_takes_upconv2x(int n, int h_in, int w_in, int c, int cout) {
  if (n <= 0 || h_in < 2 || w_in < 2 || c <= 0 || cout <= 0 || c % 32 != 0 || cout % 32 != 0) return 0;
  return c >= 128 || mie_all_phases_upconv2x(n, h_in, w_in, c, cout, MIE_DTYPE_F32_F16X2);
}
