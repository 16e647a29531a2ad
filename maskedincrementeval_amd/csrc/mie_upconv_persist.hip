// The last decoder of the batched bf16 network -- 5x5 conv over up2x(a + b), 64 -> 32 channels, bf16 deltas -- as a
// persistent kernel (gfx950).
//
// Per 8x8 output tile this layer holds 0.7 us of matrix-core work (1600 x 32 per pixel) against 22 KB of reservoir and
// delta traffic and a chain of dependent memory round trips -- tile id, mask bytes, source pixels, filter, reservoir --
// that a one-tile workgroup walks once per tile: at four resident workgroups per CU each lives 14 us for those 0.7.
// Here 512 workgroups stay resident (two per CU) and walk the tile list:
//   * the filter never moves again: a wave owns 16 of the 64 input channels for all 25 taps, which is 25 x 16 bytes
//     per lane -- 100 registers -- loaded once per workgroup instead of once per tile (102 KB per tile from L2);
//   * the next tile's source pixels, mask bytes and list entry are asked for while the current tile is blended and
//     multiplied, this tile's reservoir values before its contraction: no load is waited for where it is issued;
//   * staging buffer, source block and the k-split reduction buffer have LDS of their own (72 KB), so a tile takes
//     three barriers;
//   * and, what counts most, a tile costs fewer instructions: this layer is bound by instruction issue (the one-tile
//     kernel spends about 1900 issue slots per wave and tile, the bilinear blend of the 12 x 12 x 64 staged values
//     first among them).  The blend here is separable -- a thread owns one column, eight channels and six rows of the
//     staged tile, forms the column-blended values of its five source rows once and takes every output row from two
//     of them -- tile coordinates come from multiplications instead of divisions, and the epilogue's cases (reservoir,
//     activation) are template arguments.
// Arithmetic, operand layouts and summation order are those of k_conv_mfma<bf16, 5, 1, 1, 1, ..., UP> (32-column
// slab, four-way k-split added in wave order, fp32 blend of the fp32 sums a + b), so the two kernels agree bit for bit.
// XCD-aware order: workgroup b lives on XCD b % 8; each XCD takes a contiguous eighth of the tile list and its 64
// workgroups walk it side by side, so neighbouring tiles, which share their halo, meet in one L2 at about the same time.
#include "mie_conv.h"

#include <stdlib.h>

#include <type_traits>

namespace {

typedef float v16f __attribute__((ext_vector_type(16)));
typedef float v4f __attribute__((ext_vector_type(4)));

constexpr int C = 64;                 // input channels (one staged chunk of bf16)
constexpr int COUT = 32;              // output channels (one slab)
constexpr int K = 5;
constexpr int EPS = 8;                // bf16 elements per 16-byte slot
constexpr int Q4 = C / EPS;           // slots per pixel
constexpr int IT = 7 + K;             // staged tile edge (12)
constexpr int NPIX = IT * IT;
constexpr int NSLOT = NPIX * Q4;      // 1152
constexpr int NLD = (NSLOT + 255) / 256;
constexpr int LS = C + EPS;           // staged elements per pixel (72)
constexpr int RP = 960;               // staged elements per tile row: 12 * 72 = 864, raised to 480 dwords = 32 (mod 64)
constexpr int STAGE = IT * RP;        // bf16 elements
constexpr int LO_F = 64 * C;          // floats of the 8x8 source block
constexpr int RED_F = 4 * 64 * COUT;  // floats of the k-split reduction buffer
constexpr int GRID = 512;             // resident workgroups: two per CU
static_assert(RP % 8 == 0 && (RP / 2) % 64 == 32, "row pitch: 32 dwords modulo 64");
static_assert(STAGE * 2 + LO_F * 4 + RED_F * 4 <= 80 * 1024, "two workgroups per CU");

__device__ __forceinline__ void bf16x8_to_f32(const float4& raw, float (&f)[8]) {
  const v4f r4 = {raw.x, raw.y, raw.z, raw.w};
  const mie_bf16x8 b = __builtin_bit_cast(mie_bf16x8, r4);
#pragma unroll
  for (int e = 0; e < 8; ++e) f[e] = (float)b[e];
}
__device__ __forceinline__ float4 f32_to_bf16x8(const float (&f)[8]) {
  mie_bf16x8 b;
#pragma unroll
  for (int e = 0; e < 8; ++e) b[e] = (mie_bf16)f[e];
  const v4f r4 = __builtin_bit_cast(v4f, b);
  return make_float4(r4[0], r4[1], r4[2], r4[3]);
}
__device__ __forceinline__ void mma(v16f& acc, const float4& av, const float4& bv) {
  const v4f a4 = {av.x, av.y, av.z, av.w}, b4 = {bv.x, bv.y, bv.z, bv.w};
  acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(mie_bf16x8, a4), __builtin_bit_cast(mie_bf16x8, b4), acc, 0, 0, 0);
}

// (batch index, top-left output pixel) of tile id `tile`; divisions by the tile grid as multiplications by
// ceil(2^32 / d) (exact while tile * d < 2^32: tile ids stay below 2^30 / d here, see the launcher)
struct TileGrid { int tiles_x, tiles_y; unsigned mx, my; };
struct TilePos { int n, y0, x0; };
__device__ __forceinline__ int div_magic(int a, int d, unsigned m) { return d == 1 ? a : (int)__umulhi((unsigned)a, m); }
__device__ __forceinline__ TilePos tile_pos(const TileGrid& g, int tile) {
  TilePos p;
  const int t2 = div_magic(tile, g.tiles_x, g.mx);
  p.x0 = (tile - t2 * g.tiles_x) * MIE_TILE;
  p.n = div_magic(t2, g.tiles_y, g.my);
  p.y0 = (t2 - p.n * g.tiles_y) * MIE_TILE;
  return p;
}

// v of another lane, chosen by a DPP control word (lanes without a source read 0)
template <int CTRL>
__device__ __forceinline__ float dpp_f32(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xf, 0xf, true));
}

// epilogue of one group of four adjacent channels, its cases fixed at compile time
template <bool RES, int ACT>
__device__ __forceinline__ void epilogue4(const ConvArgsT<mie_bf16>& a, long long off, const float4& v, const float4& r0, bool live) {
  if (!live) {      // outside the output pixel mask: the reservoir stays as it is
    mie_st4(a.out, off, make_float4(0.f, 0.f, 0.f, 0.f));
    return;
  }
  if (!RES) {
    mie_st4(a.out, off, v);
    return;
  }
  const float4 r1 = make_float4(r0.x + v.x, r0.y + v.y, r0.z + v.z, r0.w + v.w);
  mie_st4(a.res, off, r1);
  mie_st4(a.out, off, make_float4(mie_act(ACT, a.slope, r1.x) - mie_act(ACT, a.slope, r0.x),
                                  mie_act(ACT, a.slope, r1.y) - mie_act(ACT, a.slope, r0.y),
                                  mie_act(ACT, a.slope, r1.z) - mie_act(ACT, a.slope, r0.z),
                                  mie_act(ACT, a.slope, r1.w) - mie_act(ACT, a.slope, r0.w)));
}

// PRED: the network's tail rides along.  The layer's activation increment y (32 channels, rounded to bf16 as the
// delta it would have been stored as) is not written; instead the 1x1 prediction conv over y and over a second
// 32-channel delta at the same resolution (the head's output: pred(x + head) = w . y + w . head, the conv being
// linear) is summed over the eight lanes that share a pixel, added to the prediction's pre-activation reservoir, and
// the one-channel activation increment is the output.
struct PredTail {
  const mie_bf16* skip;        // [n, h, w, 32] delta, clean outside skip_mask
  const uint8_t* skip_mask;    // may be NULL: every pixel
  const float* w;              // [2][32]: weights of y, weights of skip
  float* res;                  // [n, h, w] pre-activation reservoir of the prediction
  mie_bf16* out;               // [n, h, w] prediction delta
  int act;
  float slope;
  const uint32_t* flags;       // tile flags of the output tile set (BORDER, k_upconv2x_pred)
};

// BORDER: of the active tiles only those along the border of the plane (k_upconv2x_pred makes the others), found by their
// flags instead of through the list; the stale tiles are all zeroed here.
template <bool RES, int ACT, bool PRED = false, bool BORDER = false>
__global__ __launch_bounds__(256, 2) void k_upconv64_persist(ConvArgsT<mie_bf16> a, PredTail pt) {
  static_assert(!PRED || RES, "the fused tail needs the layer's reservoir");
  static_assert(!BORDER || PRED, "the border's tiles belong to the fused tail");
  __shared__ __attribute__((aligned(16))) mie_bf16 s_stage[STAGE];
  __shared__ __attribute__((aligned(16))) float s_lo[LO_F];
  __shared__ __attribute__((aligned(16))) float s_red[RED_F];
  const int entry_zero = conv_args_entry_zero(a);
  const int bid = blockIdx.x + entry_zero;
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int l32 = lane & 31, half = lane >> 5;
  const int cap = a.ts.n * a.ts.tiles_y * a.ts.tiles_x;
  const int n_act = a.ts.counts[MIE_CNT_ACTIVE], n_st = a.ts.counts[MIE_CNT_STALE];
  if (n_act < 0 || n_st < 0 || n_act > cap || n_st > cap) return;       // corrupt counts
  const int hout = a.ts.h, wout = a.ts.w;
  const int h_lo = a.h_in >> 1, w_lo = a.w_in >> 1;
  TileGrid grid;
  grid.tiles_x = a.ts.tiles_x; grid.tiles_y = a.ts.tiles_y;
  grid.mx = 0xffffffffu / (unsigned)grid.tiles_x + 1u;
  grid.my = 0xffffffffu / (unsigned)grid.tiles_y + 1u;

  // ---- stale tiles: zero this layer's delta there (the whole grid shares them) ----------------------------------
  for (int s = bid; s < n_st; s += GRID) {
    const int tile = a.ts.stale[s];
    if (tile < 0 || tile >= cap) continue;
    const TilePos tp = tile_pos(grid, tile);
    if (PRED) {
      const int oy = tp.y0 + (tid >> 3), ox = tp.x0 + (tid & 7);
      if (tid < 64 && oy < hout && ox < wout) pt.out[((long long)tp.n * hout + oy) * wout + ox] = (mie_bf16)0.f;
      continue;
    }
    for (int idx = tid; idx < 64 * (COUT / 4); idx += 256) {
      const int p = idx / (COUT / 4), col = 4 * (idx - p * (COUT / 4));
      const int oy = tp.y0 + (p >> 3), ox = tp.x0 + (p & 7);
      if (oy < hout && ox < wout)
        mie_st4(a.out, (((long long)tp.n * hout + oy) * wout + ox) * COUT + col, make_float4(0.f, 0.f, 0.f, 0.f));
    }
  }

  // ---- this workgroup's walk over the active list ------------------------------------------------------------------
  const int xcd = bid & 7, per = GRID >> 3;
  const int edge = 2 * grid.tiles_x + 2 * (grid.tiles_y - 2);        // BORDER: border tiles of a sample
  const int n_walk = BORDER ? a.ts.n * edge : n_act;
  const int c_act = (n_walk + 7) >> 3;
  const int t_hi = (xcd + 1) * c_act < n_walk ? (xcd + 1) * c_act : n_walk;
  int t = xcd * c_act + (bid >> 3);
  if (t >= t_hi) return;
  auto list_entry = [&](int pos) -> int {     // tile id at position pos of this walk, -1 past its end, -2: nothing to do there
    if constexpr (BORDER) {
      if (pos >= t_hi) return -1;
      const int n = pos / edge, k = pos - n * edge, s = k - 2 * grid.tiles_x;
      const int ty = k < grid.tiles_x ? 0 : (s < 0 ? grid.tiles_y - 1 : 1 + (s >> 1));
      const int tx = s < 0 ? (k < grid.tiles_x ? k : k - grid.tiles_x) : ((s & 1) ? grid.tiles_x - 1 : 0);
      const int v = (n * grid.tiles_y + ty) * grid.tiles_x + tx;
      return (pt.flags[v] & 1u) != 0u ? v : -2;
    }
    const int v = a.ts.tiles[pos < t_hi ? pos : t_hi - 1];
    return (pos < t_hi && v >= 0 && v < cap) ? v : -1;
  };

  // ---- the filter: this wave's 16 input channels of every tap, for good ----------------------------------------
  // matrix-core filter copy P[ci/16][tap][(ci%16)/8][co][ci%8]: a lane's 16 bytes of unit (sub-chunk `wave`, tap)
  float4 bfrag[K * K];
  {
    const mie_bf16* fb = a.filt_mc + ((long long)wave * (K * K) * 2 * COUT) * EPS + (half * COUT + l32) * EPS;
#pragma unroll
    for (int tap = 0; tap < K * K; ++tap) bfrag[tap] = *reinterpret_cast<const float4*>(fb + (long long)tap * 2 * COUT * EPS);
  }

  // ---- the tail's weights of this thread's four channels (its column group is the same in both epilogue groups) ----
  float4 pw_y = make_float4(0.f, 0.f, 0.f, 0.f), pw_s = pw_y;
  if (PRED) {
    pw_y = *reinterpret_cast<const float4*>(pt.w + 4 * (tid & 7));
    pw_s = *reinterpret_cast<const float4*>(pt.w + COUT + 4 * (tid & 7));
  }

  // ---- per-thread constants of the staging plan -------------------------------------------------------------------
  // source block: 64 pixels x 8 slots per tensor; this thread copies slot q4 of pixels lp0 and lp0 + 32
  const int q4 = tid & 7, lp0 = tid >> 3;
  // operand reads: pixel p = 32 * mb + l32 of the tile, channels 16 * wave + 8 * half ...
  int a_lane[2];
#pragma unroll
  for (int mb = 0; mb < 2; ++mb) {
    const int p = mb * 32 + l32;
    a_lane[mb] = (p >> 3) * RP + (p & 7) * LS + 16 * wave + EPS * half;
  }
  const bool has2 = a.x2 != nullptr;
  const uint8_t* const x2m = has2 ? a.x2m : nullptr;
  const mie_bf16* dummy = a.filt_mc;      // lanes outside the plane read one cache-resident address

  // source pixels and mask bits of a tile, into registers (loads unconditional in control flow)
  // (values and mask bytes go out together and are looked at when the tile's turn comes: with the reservoirs, the other delta
  // and its mask likewise, the tail at 8x480x640 takes 262 us instead of 270, both launches)
  struct Src {
    float4 a[2], b[2];
    unsigned ma[2], mb[2], in;
  } src;
  auto load_src = [&](int tile) {
    const TilePos tp = tile_pos(grid, tile < 0 ? 0 : tile);
    const int lo_y0 = ((tp.y0 - 2) >> 1) - 1, lo_x0 = ((tp.x0 - 2) >> 1) - 1;
    int po[2];
    src.in = 0u;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int lp = lp0 + 32 * i;
      const int ly = lo_y0 + (lp >> 3), lx = lo_x0 + (lp & 7);
      const bool inb = tile >= 0 && ly >= 0 && ly < h_lo && lx >= 0 && lx < w_lo;
      po[i] = inb ? (tp.n * h_lo + ly) * w_lo + lx : 0;
      const long long eo = (long long)po[i] * C + EPS * q4;
      src.a[i] = *reinterpret_cast<const float4*>(inb ? a.x + eo : dummy);
      src.b[i] = *reinterpret_cast<const float4*>((inb && has2) ? a.x2 + eo : dummy);
      src.in |= (inb ? 1u : 0u) << i;
    }
    mie_mask_ask(a.xm, dummy, po, src.ma);
    mie_mask_ask(x2m, dummy, po, src.mb);
  };

  int tile = list_entry(t);
  int tile_next = list_entry(t + per);
  load_src(tile);

  while (BORDER ? tile != -1 : tile >= 0) {
    if (BORDER && tile < 0) {
      t += per;
      tile = tile_next;
      tile_next = list_entry(t + per);
      load_src(tile);
      continue;
    }
    const TilePos tp = tile_pos(grid, tile);
    const int n = tp.n, y0 = tp.y0, x0 = tp.x0;
    const int iy0 = y0 - 2, ix0 = x0 - 2;
    const int lo_y0 = (iy0 >> 1) - 1, lo_x0 = (ix0 >> 1) - 1;

    // A. a + b of the source block to LDS, fp32 (masked pixels: the raw registers are zeroed, bit pattern 0 = 0.0)
    const unsigned ok_a = mie_mask_take(a.xm, src.ma, src.in), ok_b = mie_mask_take(x2m, src.mb, has2 ? src.in : 0u);
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const bool ka = (ok_a >> i) & 1u, kb = (ok_b >> i) & 1u;
      const float4 ra = src.a[i], rb = src.b[i];
      const float4 za = make_float4(ka ? ra.x : 0.f, ka ? ra.y : 0.f, ka ? ra.z : 0.f, ka ? ra.w : 0.f);
      const float4 zb = make_float4(kb ? rb.x : 0.f, kb ? rb.y : 0.f, kb ? rb.z : 0.f, kb ? rb.w : 0.f);
      float fa[8], fb[8];
      bf16x8_to_f32(za, fa);
      bf16x8_to_f32(zb, fb);
      float* d = s_lo + (lp0 + 32 * i) * C + q4 * EPS;
      *reinterpret_cast<float4*>(d) = make_float4(fa[0] + fb[0], fa[1] + fb[1], fa[2] + fb[2], fa[3] + fb[3]);
      *reinterpret_cast<float4*>(d + 4) = make_float4(fa[4] + fb[4], fa[5] + fb[5], fa[6] + fb[6], fa[7] + fb[7]);
    }

    // B. this tile's reservoir values: asked for now, used after the contraction
    long long e_off[2];
    bool e_ok[2];
    float4 e_r0[2];
    long long t_pix[2];          // PRED: pixel index, the second delta's four channels and mask, the prediction's reservoir value
    mie_bf16x4 t_skip[2];
    float t_p0[2];
    int t_at[2];
    unsigned t_in = 0u, t_m[2];  // mask bytes: of the second delta (PRED), of the output pixel mask otherwise
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int idx = tid + 256 * i;
      const int p = idx >> 3, col = 4 * (idx & 7);
      const int oy = y0 + (p >> 3), ox = x0 + (p & 7);
      e_ok[i] = oy < hout && ox < wout;
      const int pix = e_ok[i] ? (n * hout + oy) * wout + ox : 0;
      e_off[i] = (long long)pix * COUT + col;
      e_r0[i] = make_float4(0.f, 0.f, 0.f, 0.f);
      if (RES) e_r0[i] = *reinterpret_cast<const float4*>(a.res + e_off[i]);
      t_at[i] = pix;
      t_in |= (e_ok[i] ? 1u : 0u) << i;
      if (PRED) {
        t_pix[i] = pix;
        t_skip[i] = *reinterpret_cast<const mie_bf16x4*>(pt.skip + e_off[i]);
        t_p0[i] = pt.res[pix];
      }
    }
    const uint8_t* const t_mask = PRED ? pt.skip_mask : a.ts.pixmask;
    mie_mask_ask(t_mask, dummy, t_at, t_m);

    // C. the next tile's source pixels and the list entry after it
    t += per;
    const int tile_nn = list_entry(t + per);
    load_src(tile_next);
    __syncthreads();                                   // (1) the source block is in LDS

    // D. the staged tile, blended from the source block.  Thread u < 192 owns column pcol, channels 8 * sq .. and rows
    // 6 * rh .. 6 * rh + 5 of the 12 x 12 tile: the column blend of its five source rows (local rows 3 * rh .. 3 * rh + 4 of
    // the 8 x 8 block) once, then every output row from two of them.  Row 2m of the up-sampled image takes source rows
    // (m - 1, m) with weights (1/4, 3/4), row 2m + 1 rows (m, m + 1) with (3/4, 1/4); at the image border the missing
    // neighbour is the row itself, i.e. weights (0, 1) / (1, 0) on the pair as it lies in the block (rows outside the image
    // are stored as zeros); rows and columns outside the up-sampled image are the conv's zero padding: weights (0, 0).
    if (tid < 192) {
      const int sq = tid & 7, cu = tid >> 3;
      const int rh = cu >= IT ? 1 : 0, pcol = cu - IT * rh;
      const int hx = ix0 + pcol;
      int c0 = 0, c1 = 0;
      float lq0 = 0.f, lq1 = 0.f;
      if (hx >= 0 && hx < a.w_in) conv_up2x_coef(hx, w_lo, c0, c1, lq0, lq1);
      else c0 = c1 = lo_x0 < 0 ? 0 : lo_x0;
      const float* s0 = s_lo + ((3 * rh) * 8 + (c0 - lo_x0)) * C + sq * EPS;
      const float* s1 = s_lo + ((3 * rh) * 8 + (c1 - lo_x0)) * C + sq * EPS;
      float hb[5][EPS];
#pragma unroll
      for (int r = 0; r < 5; ++r)
#pragma unroll
        for (int e = 0; e < EPS; e += 4) {
          const float4 t0 = *reinterpret_cast<const float4*>(s0 + r * 8 * C + e), t1 = *reinterpret_cast<const float4*>(s1 + r * 8 * C + e);
          hb[r][e] = conv_up2x_h(lq0, lq1, t0.x, t1.x);
          hb[r][e + 1] = conv_up2x_h(lq0, lq1, t0.y, t1.y);
          hb[r][e + 2] = conv_up2x_h(lq0, lq1, t0.z, t1.z);
          hb[r][e + 3] = conv_up2x_h(lq0, lq1, t0.w, t1.w);
        }
#pragma unroll
      for (int i = 0; i < 6; ++i) {
        const int pr = 6 * rh + i;
        const int hy = iy0 + pr, m = hy >> 1;
        const bool odd = (i & 1) != 0;                       // iy0 is even: row parity is the parity of i
        const int ra_ = (i >> 1) + (odd ? 1 : 0);            // first row of the pair, relative to 3 * rh
        float lr0 = odd ? 0.75f : 0.25f, lr1 = odd ? 0.25f : 0.75f;
        if (odd ? (m + 1 >= h_lo) : (m == 0)) lr0 = odd ? 1.f : 0.f, lr1 = odd ? 0.f : 1.f;
        if (hy < 0 || hy >= a.h_in) lr0 = lr1 = 0.f;
        float o[EPS];
#pragma unroll
        for (int e = 0; e < EPS; ++e) o[e] = conv_up2x_v(lr0, lr1, hb[ra_][e], hb[ra_ + 1][e]);
        *reinterpret_cast<float4*>(s_stage + pr * RP + pcol * LS + EPS * sq) = f32_to_bf16x8(o);
      }
    }
    __syncthreads();                                   // (2) the staged tile is in LDS

    // E. the contraction: 25 units (taps) of this wave's sub-chunk, two pixel blocks each
    v16f acc[2];
#pragma unroll
    for (int mb = 0; mb < 2; ++mb)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[mb][r] = 0.f;
    {
      float4 av[2][2];
      av[0][0] = *reinterpret_cast<const float4*>(&s_stage[a_lane[0]]);
      av[0][1] = *reinterpret_cast<const float4*>(&s_stage[a_lane[1]]);
#pragma unroll
      for (int tap = 0; tap < K * K; ++tap) {
        if (tap + 1 < K * K) {
          const int ky = (tap + 1) / K, kx = (tap + 1) - ky * K;
          av[(tap + 1) & 1][0] = *reinterpret_cast<const float4*>(&s_stage[a_lane[0] + ky * RP + kx * LS]);
          av[(tap + 1) & 1][1] = *reinterpret_cast<const float4*>(&s_stage[a_lane[1] + ky * RP + kx * LS]);
        }
        __builtin_amdgcn_sched_barrier(0);
        mma(acc[0], av[tap & 1][0], bfrag[tap]);
        mma(acc[1], av[tap & 1][1], bfrag[tap]);
        __builtin_amdgcn_sched_barrier(0);
      }
    }

    // F. the four k-split partial sums meet in LDS (a buffer of its own: nobody has to be waited for first)
    {
      float* red = s_red + wave * (64 * COUT);
#pragma unroll
      for (int mb = 0; mb < 2; ++mb)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int p = mb * 32 + 8 * (r >> 2) + 4 * half + (r & 3);
          red[p * COUT + l32] = acc[mb][r];
        }
    }
    __syncthreads();                                   // (3) the partial sums are in LDS
    {
      float4 v[2];
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const int idx = tid + 256 * i;
        float4 sum = *reinterpret_cast<const float4*>(&s_red[4 * idx]);
#pragma unroll
        for (int k2 = 1; k2 < 4; ++k2) {
          const float4 part = *reinterpret_cast<const float4*>(&s_red[k2 * (64 * COUT) + 4 * idx]);
          sum.x += part.x; sum.y += part.y; sum.z += part.z; sum.w += part.w;
        }
        v[i] = sum;
      }
      const unsigned t_on = mie_mask_take(t_mask, t_m, t_in);
      if constexpr (PRED) {
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          const bool on = (t_on >> i) & 1u;
          const float4 sk = make_float4(on ? (float)t_skip[i][0] : 0.f, on ? (float)t_skip[i][1] : 0.f, on ? (float)t_skip[i][2] : 0.f, on ? (float)t_skip[i][3] : 0.f);
          const float4 r0 = e_r0[i];
          const float4 r1 = make_float4(r0.x + v[i].x, r0.y + v[i].y, r0.z + v[i].z, r0.w + v[i].w);
          if (e_ok[i]) mie_st4(a.res, e_off[i], r1);
          // the increment as the bf16 delta it would be stored as
          const float y0_ = (float)(mie_bf16)(mie_act(ACT, a.slope, r1.x) - mie_act(ACT, a.slope, r0.x));
          const float y1_ = (float)(mie_bf16)(mie_act(ACT, a.slope, r1.y) - mie_act(ACT, a.slope, r0.y));
          const float y2_ = (float)(mie_bf16)(mie_act(ACT, a.slope, r1.z) - mie_act(ACT, a.slope, r0.z));
          const float y3_ = (float)(mie_bf16)(mie_act(ACT, a.slope, r1.w) - mie_act(ACT, a.slope, r0.w));
          float z = pw_y.x * y0_ + pw_y.y * y1_ + pw_y.z * y2_ + pw_y.w * y3_;
          z += pw_s.x * sk.x + pw_s.y * sk.y + pw_s.z * sk.z + pw_s.w * sk.w;
          if (!e_ok[i]) z = 0.f;
          // the eight lanes of a pixel, by data-parallel moves inside the wave's rows of 16 (no LDS round trip):
          // neighbours within quads, then the quad four lanes up -- complete in the lanes 0 and 8 of a row, the ones
          // that own the pixel's prediction
          z += dpp_f32<0xB1>(z);               // quad_perm [1,0,3,2]
          z += dpp_f32<0x4E>(z);               // quad_perm [2,3,0,1]
          z += dpp_f32<0x104>(z);              // row_shl:4 (lane l reads lane l + 4)
          if (e_ok[i] && (tid & 7) == 0) {
            float r[2] = {t_p0[i] + z, t_p0[i]};
            pt.res[t_pix[i]] = r[0];
            mie_act_n(pt.act, pt.slope, r);
            pt.out[t_pix[i]] = (mie_bf16)(r[0] - r[1]);
          }
        }
      } else {
#pragma unroll
        for (int i = 0; i < 2; ++i)
          if (e_ok[i]) epilogue4<RES, ACT>(a, e_off[i], v[i], e_r0[i], ((t_on >> i) & 1u) != 0u);
      }
    }
    // (the next tile's barriers (1) and (2) stand between these reads of s_red and its next writes, barrier (3) between
    // this tile's reads of s_lo / s_stage and their next writes)
    tile = tile_next;
    tile_next = tile_nn;
  }
}

// ---- the same tail at the resolution of its inputs ---------------------------------------------------------------------
// The conv over the up-sampled image is four 4x4 convs over a + b, one per output phase (py, px), away from the image's
// border (mie_upconv2x.hip): 16 taps instead of 25, nothing to blend, and an input pixel is staged once for the four
// outputs it stands for.  What bounds the one-tile form above is instruction issue (1900 slots a wave and tile, the blend
// first among them); what is left here is the traffic of the reservoirs, and the wait for it.
//   * An item is 8 x 16 input positions = 16 x 32 outputs = 2 x 4 tiles.  A workgroup (8 waves, one per CU) makes the output
//     rows of one parity py; a wave takes one column parity px, half of the 32 output channels and half of the 64 input
//     channels.  Its filter -- 16 taps x 32 x 16 -- stays in 64 registers for good, which leaves room for everything the
//     next item needs.  (Four waves with 128 registers of filter each, two workgroups a CU: 370 us at 8x480x640, three
//     quarters of them waiting, for what was asked for too late.)
//   * 16x16x32 MFMAs with the filter as the first operand: a lane then holds four adjacent channels of one position, so
//     reservoirs, the other delta and the prediction's products go from the accumulators to memory and back without LDS.
//     A fragment of input row r serves the output rows r - 3 .. r: 44 fragments are read for 128 MFMAs.  The two waves
//     that share their outputs exchange half of their sums: each finishes four of the eight rows.
//   * Nothing is waited for where it is asked for, and loads are spread over an item: a slot of the window after next and a
//     row of the next item's reservoir are asked for between the MFMAs of this item's sums.  (A CU keeps about 32 KB of misses
//     on their way; asked for in one go, what an item needs -- 115 KB -- held its waves at the issue of their loads for 7400
//     of 16000 clocks.)
//   * One barrier an item, so that some waves make sums while others are at the reservoirs.
//   * Tiles along the border are left to k_upconv64_persist<..., BORDER>, in a launch of its own before this one (45 us of
//     the 268 below).
// Sums of a wave run over K = 16 x 32 in one accumulator.  Measured against the one-tile form, all tiles active: 8x480x640
// 570 -> 268 us (2.8 TB/s of reservoirs and deltas), 1x480x640 66 -> 49, 2x264x352 44 -> 39, 1x360x500 44 -> 38.  Error of the layer's sums
// against fp64 in networks of 1 .. 20 % input density 0.88 - 0.91 of that form's, of the prediction's 0.91 - 0.95 (white
// noise, which no layer sees: 1.04).
constexpr int PR = 8, PC = 16;                     // positions of an item
constexpr int SR = PR + 3, SC = PC + 4;            // its staged window
constexpr int PSTG = (SR * SC + 1) * LS;           // bf16 elements; the last pixel takes what lies behind the window
constexpr int PTHR = 512, PGRID = 256, PITEMS = 2048;      // threads, workgroups, items of a walk at most
constexpr int PSLOT = SR * SC * Q4;                // 1760
constexpr int PLD = (PSLOT + PTHR - 1) / PTHR;     // 4
static_assert(PSTG * 2 * 2 + 2 * 8 * (PR / 2) * 64 * 16 + 2 * 4 * PR * PC * 4 + 512 + PITEMS * 4 + 32 + 8 * COUT <= 160 * 1024, "LDS of a CU");

struct PhaseItems {
  const mie_bf16* filter;       // the combined filter of mie_pack_filter_up2x
  int iy, ix, total;            // items of a sample along y and x, items of all samples (at most 2^18: cap <= 2^20 tiles)
  unsigned my, mx;              // ceil(2^32 / iy), ceil(2^32 / ix)
};

__device__ __forceinline__ v4f mma16(const v4f& w, const v4f& x, const v4f& acc) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(mie_bf16x8, w), __builtin_bit_cast(mie_bf16x8, x), acc, 0, 0, 0);
}

template <int ACT>
__global__ __launch_bounds__(PTHR, 2) void k_upconv2x_pred(ConvArgsT<mie_bf16> a, PredTail pt, PhaseItems g) {
  __shared__ __attribute__((aligned(16))) mie_bf16 s_stage[2][PSTG];
  __shared__ v4f s_sum[2][8][PR / 2][64];          // [parity of the item][wave that finishes them][row][lane]
  __shared__ float s_z[2][2][2][PR][PC];           // [parity of the item][half of the output channels][px][row][position]
  __shared__ unsigned char s_m[2][256];            // [parity][pixel of the window]: bit 0 a's mask, bit 1 b's
  __shared__ unsigned s_list[PITEMS];
  __shared__ int s_count[PTHR / 64];
  __shared__ __attribute__((aligned(16))) float s_w[2 * COUT];
  const int bid = blockIdx.x + conv_args_entry_zero(a);
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int pos = lane & 15, cg = lane >> 4, px = wave & 1, nh = (wave >> 1) & 1, ks = wave >> 2;
  const int xcd = bid & 7, py = (bid >> 3) & 1, step = PGRID >> 4;
  const int H = a.h_in >> 1, W = a.w_in >> 1, hout = a.ts.h, wout = a.ts.w, tiles_x = a.ts.tiles_x, tiles_y = a.ts.tiles_y;
  const int chunk = (g.total + 7) >> 3;
  const int hi = (xcd + 1) * chunk < g.total ? (xcd + 1) * chunk : g.total;
  const int first = xcd * chunk + (bid >> 4);
  if (first >= hi) return;

  // ---- the items of this walk with an active tile: place in the walk, and which of the 2 x 4 tiles (bit 4 * row + column)
  // in the upper half
  int n_items = 0;
  {
    const int n_walk = (hi - first + step - 1) / step;       // at most 2048: see the launcher
    for (int k0 = 0; k0 < n_walk; k0 += PTHR / 8) {
      const int k = k0 + (tid >> 3), it = first + step * k;
      const int t2 = div_magic(it, g.ix, g.mx), n = div_magic(t2, g.iy, g.my);
      const int ty = 1 + 2 * (t2 - n * g.iy) + ((tid >> 2) & 1), tx = 1 + 4 * (it - t2 * g.ix) + (tid & 3);
      const bool in = k < n_walk && ty < tiles_y - 1 && tx < tiles_x - 1;
      const unsigned f = in ? pt.flags[(n * tiles_y + ty) * tiles_x + tx] : 0u;
      const unsigned act = (unsigned)(__ballot((f & 1u) != 0u) >> (lane & 56)) & 0xffu;
      const bool has = (lane & 7) == 0 && act != 0u;
      const unsigned long long b = __ballot(has);
      if (lane == 0) s_count[wave] = __popcll(b);
      __syncthreads();
      int at = n_items, all = 0;
#pragma unroll
      for (int w = 0; w < PTHR / 64; ++w) {
        at += w < wave ? s_count[w] : 0;
        all += s_count[w];
      }
      if (has) s_list[at + __popcll(b & ((1ull << lane) - 1ull))] = (unsigned)k | act << 16;
      n_items += all;
      __syncthreads();
    }
    if (n_items == 0) return;
  }
  struct Item { int n, ty, tx; unsigned act; };
  auto item_at = [&](int i) -> Item {            // past the end: the last one with nothing active
    const unsigned e = __builtin_amdgcn_readfirstlane(s_list[i < n_items ? i : n_items - 1]);
    const int it = first + step * (int)(e & 0xffffu);
    const int t2 = div_magic(it, g.ix, g.mx), n = div_magic(t2, g.iy, g.my);
    return {n, 1 + 2 * (t2 - n * g.iy), 1 + 4 * (it - t2 * g.ix), i < n_items ? e >> 16 : 0u};
  };

  // ---- this wave's filter: taps x 32 input channels x 16 output channels
  v4f wt[16];
  {
    const int phase = 2 * py + px;
    const mie_bf16* f = g.filter + ((long long)(phase * (C / 16) + 2 * ks + (cg >> 1)) * UP2X_UNITS * 2 + (cg & 1)) * COUT * EPS + (16 * nh + pos) * EPS;
#pragma unroll
    for (int t = 0; t < 16; ++t) wt[t] = *reinterpret_cast<const v4f*>(f + (long long)t * 2 * COUT * EPS);
  }
  if (tid < 2 * COUT) s_w[tid] = pt.w[tid];

  // ---- staging: slot tid + 512 i = 16 bytes (eight channels) of pixel (tid >> 3) + 64 i of the window
  int sid = tid;         // (opaque in every item, below: the places of all slots, kept from item to item, would be spilled)
  const bool has2 = a.x2 != nullptr;
  const mie_bf16* x2p = has2 ? a.x2 : a.x;
  // A mask that is not there: bytes of the tensor itself are read in its place (a branch around a load is a place where it
  // is waited for) and `all` makes a one of them.
  const uint8_t* m1p = a.xm != nullptr ? a.xm : reinterpret_cast<const uint8_t*>(a.x);
  const uint8_t* m2p = has2 && a.x2m != nullptr ? a.x2m : reinterpret_cast<const uint8_t*>(x2p);
  const unsigned m_all = (a.xm == nullptr ? 1u : 0u) | (has2 && a.x2m == nullptr ? 2u : 0u), m_use = has2 ? 3u : 1u;
  typedef const __attribute__((address_space(1))) uint8_t* GlobalBytes;      // (said, or the selected pointer is read with flat loads)
  const GlobalBytes skm = (GlobalBytes)(pt.skip_mask != nullptr ? pt.skip_mask : reinterpret_cast<const uint8_t*>(pt.skip));
  const unsigned sk_all = pt.skip_mask == nullptr ? 1u : 0u;
  // pixel p of an item's window (beyond the last inner tile, and beyond the window: read, not used)
  auto window_pixel = [&](const Item& q, int p) -> unsigned {
    const int r = p / SC, c = p - r * SC;
    int y = 4 * q.ty - 2 + py + r, x = 4 * q.tx - 2 + c;
    y = y < H ? y : H - 1;
    x = x < W ? x : W - 1;
    return (unsigned)((q.n * H + y) * W + x);
  };
  auto load_slot = [&](const Item& q, int i, float4& va, float4& vb) {
    const unsigned eo = (window_pixel(q, (sid >> 3) + 64 * i) * C + EPS * (sid & 7)) * 2u;      // bytes: below 2^31
    va = *reinterpret_cast<const float4*>(reinterpret_cast<const char*>(a.x) + eo);
    vb = *reinterpret_cast<const float4*>(reinterpret_cast<const char*>(x2p) + eo);
  };
  // (masks go through LDS: two bytes a thread on their way instead of two for each slot)
  struct MaskBytes { unsigned a, b; };
  auto load_masks = [&](const Item& q) -> MaskBytes {
    const unsigned po = window_pixel(q, sid < SR * SC ? sid : 0);
    return {m1p[po], m2p[po]};
  };
  auto store_masks = [&](int buf, const MaskBytes& m) {
    if (tid < 256) s_m[buf][tid] = (unsigned char)(((m.a != 0u ? 1u : 0u) | (m.b != 0u ? 2u : 0u) | m_all) & m_use);
  };
  auto store_slot = [&](int buf, int mbuf, int i, const float4& va, const float4& vb) {
    const int p = (tid >> 3) + 64 * i, at = p < SR * SC ? p : SR * SC;
    const unsigned ok = s_m[mbuf][p];
    const float4 z4 = make_float4(0.f, 0.f, 0.f, 0.f);
    float fa[8], fb[8], f[8];
    bf16x8_to_f32((ok & 1u) ? va : z4, fa);
    bf16x8_to_f32((ok & 2u) ? vb : z4, fb);
#pragma unroll
    for (int e = 0; e < 8; ++e) f[e] = fa[e] + fb[e];
    *reinterpret_cast<float4*>(&s_stage[buf][at * LS + EPS * (tid & 7)]) = f32_to_bf16x8(f);
  };

  // ---- the rows this wave finishes: 4 ks .. 4 ks + 3 of the item, position pos, channels 16 nh + 4 cg ..
  const unsigned row = 2u * (unsigned)wout;
  unsigned l_pix = (unsigned)(2 * pos + px), l_ch = (unsigned)(16 * nh + 4 * cg);
  auto item_pix = [&](const Item& q) -> long long { return ((long long)q.n * hout + 8 * q.ty + py) * wout + 8 * q.tx; };
  auto row_live = [&](unsigned act) -> bool { return ((act >> (4 * ks + (pos >> 2))) & 1u) != 0u; };
  struct Rows { float4 r0[PR / 2]; mie_bf16x4 sk[PR / 2]; unsigned on[PR / 2]; float p0; };
  // the prediction: thread tid < 256 owns pixel (row tid >> 5, column tid & 31) of the item's outputs
  const int p_r = (tid >> 5) & 7, p_x = tid & 31;
  const unsigned p_off = p_r * row + p_x;
  auto pred_live = [&](unsigned act) -> bool { return tid < 256 && ((act >> (4 * (p_r >> 2) + (p_x >> 3))) & 1u) != 0u; };
  // (no branch around the loads, or what they fetch would be waited for in it: lanes of inactive tiles read the item's first
  // pixel)
  auto load_row = [&](Rows& rows, long long pix0, bool live, int r) {
    const unsigned p = live ? (4 * ks + r) * row + l_pix : 0u, off = p * COUT + l_ch;       // bytes below 2^32: w < 2^20
    rows.r0[r] = *reinterpret_cast<const float4*>(reinterpret_cast<const char*>(a.res + pix0 * COUT) + 4u * off);
    rows.sk[r] = *reinterpret_cast<const mie_bf16x4*>(reinterpret_cast<const char*>(pt.skip + pix0 * COUT) + 2u * off);
    rows.on[r] = (skm + pix0)[p];
  };
  auto load_pred = [&](Rows& rows, long long pix0, unsigned act) { rows.p0 = (pt.res + pix0)[pred_live(act) ? p_off : 0u]; };

  // ---- before the first item: its window and its rows, the second item's window and masks, the third's masks
  Item cur = item_at(0), nxt = item_at(1), after = item_at(2);
  float4 va[PLD], vb[PLD];
  Rows rows_a, rows_b;
#pragma unroll
  for (int i = 0; i < PLD; ++i) load_slot(cur, i, va[i], vb[i]);
  store_masks(0, load_masks(cur));
  store_masks(1, load_masks(nxt));
  __syncthreads();
#pragma unroll
  for (int i = 0; i < PLD; ++i) store_slot(0, 0, i, va[i], vb[i]);
#pragma unroll
  for (int i = 0; i < PLD; ++i) load_slot(nxt, i, va[i], vb[i]);
  MaskBytes masks = load_masks(after);
#pragma unroll
  for (int r = 0; r < PR / 2; ++r) load_row(rows_a, item_pix(cur), row_live(cur.act), r);
  load_pred(rows_a, item_pix(cur), cur.act);
  __syncthreads();

  int par = 0;
  // the predictions of an item, once its products are in LDS: behind the next item's barrier
  long long z_pix = 0;
  unsigned z_act = 0u;
  float z_p0 = 0.f;
  auto predict = [&]() {
    if (pred_live(z_act)) {
      float r[2] = {z_p0 + (s_z[par ^ 1][0][p_x & 1][p_r][p_x >> 1] + s_z[par ^ 1][1][p_x & 1][p_r][p_x >> 1]), z_p0};
      (pt.res + z_pix)[p_off] = r[0];
      mie_act_n(pt.act, pt.slope, r);
      (pt.out + z_pix)[p_off] = (mie_bf16)(r[0] - r[1]);
    }
  };
  auto one_item = [&](int i, const Rows& rows, Rows& rows_next) {
    asm volatile("" : "+v"(sid), "+v"(l_pix), "+v"(l_ch));
    const long long pix_next = item_pix(nxt);
    const bool live_next = row_live(nxt.act);
    // ---- sums
    v4f acc[PR];
    {
#pragma unroll
      for (int r = 0; r < PR; ++r) acc[r] = v4f{0.f, 0.f, 0.f, 0.f};
      const mie_bf16* s = &s_stage[par][(pos + px) * LS + 32 * ks + EPS * cg];
      constexpr int NF = 4 * SR, AHEAD = 3;          // fragments: window column j, row r; asked for three ahead
      v4f x[AHEAD + 1];
      auto fetch = [&](int f) { x[f % (AHEAD + 1)] = *reinterpret_cast<const v4f*>(s + ((f % SR) * SC + f / SR) * LS); };
#pragma unroll
      for (int f = 0; f < AHEAD; ++f) fetch(f);
#pragma unroll
      for (int f = 0; f < NF; ++f) {
        if (f + AHEAD < NF) fetch(f + AHEAD);
        // the next item's window, a slot per window column: its conversions fill the time between MFMAs
        // and a slot of the window behind that is asked for in its place
        if (f % SR == 2) store_slot(par ^ 1, par ^ 1, f / SR, va[f / SR], vb[f / SR]);
        if (f % SR == 6) load_slot(after, f / SR, va[f / SR], vb[f / SR]);
        if (f % SR == 10) load_row(rows_next, pix_next, live_next, f / SR);
        __builtin_amdgcn_sched_barrier(0);
        const int j = f / SR, r = f % SR;
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if (r - i >= 0 && r - i < PR) acc[r - i] = mma16(wt[4 * i + j], x[f % (AHEAD + 1)], acc[r - i]);
        __builtin_amdgcn_sched_barrier(0);
      }
      load_pred(rows_next, pix_next, nxt.act);
      // the rows the other wave finishes
#pragma unroll
      for (int r = 0; r < PR / 2; ++r) s_sum[par][wave ^ 4][r][lane] = ks == 0 ? acc[PR / 2 + r] : acc[r];
    }
    store_masks(par, masks);
    // Sums exchanged; the next window is there, this one has been read; the products of the item before this are there.  (The
    // one barrier of an item: a wave may finish this item while another makes the next one's sums.)
    __syncthreads();
    const Item later = item_at(i + 3);
    masks = load_masks(later);
    predict();
    // ---- reservoirs and increments
    const long long pix0 = item_pix(cur);
    const bool live = row_live(cur.act);
    const float4 pw_y = *reinterpret_cast<const float4*>(&s_w[16 * nh + 4 * cg]);
    const float4 pw_s = *reinterpret_cast<const float4*>(&s_w[COUT + 16 * nh + 4 * cg]);
    z_pix = pix0;
    z_act = cur.act;
    asm volatile("v_mov_b32 %0, %1" : "=v"(z_p0) : "v"(rows.p0));      // here: a copy left to the loop's end waits for the load below
#pragma unroll
    for (int r = 0; r < PR / 2; ++r) {
      {
        const v4f mine = ks == 0 ? acc[r] : acc[PR / 2 + r], other = s_sum[par][wave][r][lane];
        const float4 q0 = rows.r0[r], q1 = make_float4(q0.x + (mine[0] + other[0]), q0.y + (mine[1] + other[1]),
                                                       q0.z + (mine[2] + other[2]), q0.w + (mine[3] + other[3]));
        // the increment as the bf16 delta it would be stored as
        const float y0 = (float)(mie_bf16)(mie_act(ACT, a.slope, q1.x) - mie_act(ACT, a.slope, q0.x));
        const float y1 = (float)(mie_bf16)(mie_act(ACT, a.slope, q1.y) - mie_act(ACT, a.slope, q0.y));
        const float y2 = (float)(mie_bf16)(mie_act(ACT, a.slope, q1.z) - mie_act(ACT, a.slope, q0.z));
        const float y3 = (float)(mie_bf16)(mie_act(ACT, a.slope, q1.w) - mie_act(ACT, a.slope, q0.w));
        float z = pw_y.x * y0 + pw_y.y * y1 + pw_y.z * y2 + pw_y.w * y3;
        const mie_bf16x4 v = rows.sk[r];
        const float zs = pw_s.x * (float)v[0] + pw_s.y * (float)v[1] + pw_s.z * (float)v[2] + pw_s.w * (float)v[3];
        z += (rows.on[r] | sk_all) != 0u ? zs : 0.f;
        if (live) *reinterpret_cast<float4*>(reinterpret_cast<char*>(a.res + pix0 * COUT) + 4u * (((4 * ks + r) * row + l_pix) * COUT + l_ch)) = q1;
        z += __shfl_xor(z, 16);
        z += __shfl_xor(z, 32);
        if (cg == 0) s_z[par][nh][px][4 * ks + r][pos] = z;
      }
    }
    cur = nxt;
    nxt = after;
    after = later;
    par ^= 1;
  };
  // Two items a round: the two sets of rows change places without copies, which would wait for their loads (the second may
  // lie past the end)
  for (int i = 0; i < n_items; i += 2) {
    one_item(i, rows_a, rows_b);
    one_item(i + 1, rows_b, rows_a);
  }
  __syncthreads();
  predict();
}


// ---- the decoder before it, 128 -> 64 channels ---------------------------------------------------------------------------
// The inner positions of mie_upconv2x_masked's layer on planes of many items, in the same manner: an item of 8 x 16 input
// positions, one output phase a workgroup, a wave = 16 of the 64 output channels and half of the 128 input channels, its
// filter (16 taps x 64 x 16) in 128 registers for good, sums exchanged between the two waves that share their outputs.
// Against k_upconv2x's blocks of 8 x 8, which read the filter (256 KB a phase) anew for each: one workgroup of eight waves a
// CU instead of three of four, no filter traffic, and every load between MFMAs, ahead of its use: the window's slots, four at
// a time, a slot of the window after next as one of the next window's is stored; the reservoir's rows at the beginning of
// the sums that go with them.  A second barrier behind the exchange stands for a second buffer (32 KB that the LDS does not
// have).  The positions along the border stay with k_upconv2x's strips.
// Measured, all tiles active, the strips' launch included: 8x120x160 265 -> 192 us (the matrix instructions alone 144 at the
// rate of a large product), 4x120x160 124 -> 99; in a masked 8x480x640 pass 281 -> 156 + 22.  An item takes 15500 cycles:
// 8000 to 10500 for its 512 matrix instructions a SIMD of 16 cycles, 2000 to 4000 for the exchange and the reservoir's rows,
// the rest at the two barriers.  The terms and their rounding are k_upconv2x's: against 64 bits the same 0.0020 from each.
// Like there, a pixel of an active tile outside the output pixel mask gets a zero delta and keeps its reservoir (its sum is
// zero, but an infinity or a NaN in the reservoir has no increment of zero).  The byte of each costs a pass 0 to 0.4 %.
constexpr int DC = 128, DCO = 64;
constexpr int DSC = PC + 3, DLS = DC + EPS, DQ4 = DC / EPS;
constexpr int DPIX = SR * DSC;                     // 209 pixels of the window
constexpr int DSTG = (DPIX + 1) * DLS;             // the last pixel takes what lies behind the window
constexpr int DLD = (DPIX * DQ4 + PTHR - 1) / PTHR, DRING = 4;      // slots of a thread, and of them on their way at a time
constexpr int DITEMS = 1024;
static_assert(DSTG * 2 * 2 + 8 * (PR / 2) * 64 * 16 + 512 + DITEMS * 4 + 32 <= 160 * 1024, "LDS of a CU");

template <bool RES, int ACT>
__global__ __launch_bounds__(PTHR, 2) void k_upconv2x_rows(ConvArgsT<mie_bf16> a, const uint32_t* flags, PhaseItems g) {
  __shared__ __attribute__((aligned(16))) mie_bf16 s_stage[2][DSTG];
  __shared__ v4f s_sum[8][PR / 2][64];             // [wave that finishes them][row][lane]
  __shared__ unsigned char s_m[2][256];            // [parity][pixel of the window]: bit 0 a's mask, bit 1 b's
  __shared__ unsigned s_list[DITEMS];
  __shared__ int s_count[PTHR / 64];
  const int bid = blockIdx.x + conv_args_entry_zero(a);
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int pos = lane & 15, cg = lane >> 4, q = wave & 3, ks = wave >> 2;
  const int xcd = bid & 7, phase = (bid >> 3) & 3, py = phase >> 1, px = phase & 1, step = PGRID >> 5;
  const int H = a.h_in, W = a.w_in, hout = a.ts.h, wout = a.ts.w, tiles_x = a.ts.tiles_x, tiles_y = a.ts.tiles_y;
  const int chunk = (g.total + 7) >> 3;
  const int hi = (xcd + 1) * chunk < g.total ? (xcd + 1) * chunk : g.total;
  const int first = xcd * chunk + (bid >> 5);
  if (first >= hi) return;

  // ---- the items of this walk with an active or a stale tile: place in the walk (16 bits), active tiles, stale tiles (8 each;
  // bit 4 * row + column of the 2 x 4)
  int n_items = 0;
  {
    const int n_walk = (hi - first + step - 1) / step;       // at most DITEMS: see the launcher
    for (int k0 = 0; k0 < n_walk; k0 += PTHR / 8) {
      const int k = k0 + (tid >> 3), it = first + step * k;
      const int t2 = div_magic(it, g.ix, g.mx), n = div_magic(t2, g.iy, g.my);
      const int ty = 2 * (t2 - n * g.iy) + ((tid >> 2) & 1), tx = 4 * (it - t2 * g.ix) + (tid & 3);
      const bool in = k < n_walk && ty < tiles_y && tx < tiles_x;
      const unsigned f = in ? flags[(n * tiles_y + ty) * tiles_x + tx] : 0u;
      const unsigned act = (unsigned)(__ballot((f & 1u) != 0u) >> (lane & 56)) & 0xffu;
      const unsigned old = (unsigned)(__ballot((f & 3u) == 2u) >> (lane & 56)) & 0xffu;
      const bool has = (lane & 7) == 0 && (act | old) != 0u;
      const unsigned long long b = __ballot(has);
      if (lane == 0) s_count[wave] = __popcll(b);
      __syncthreads();
      int at = n_items, all = 0;
#pragma unroll
      for (int w = 0; w < PTHR / 64; ++w) {
        at += w < wave ? s_count[w] : 0;
        all += s_count[w];
      }
      if (has) s_list[at + __popcll(b & ((1ull << lane) - 1ull))] = (unsigned)k | act << 16 | old << 24;
      n_items += all;
      __syncthreads();
    }
    if (n_items == 0) return;
  }
  struct Item { int n, y0, x0; unsigned act, old; };      // sample, first position
  auto item_at = [&](int i) -> Item {            // past the end: the last one (looked at, not used)
    const unsigned e = __builtin_amdgcn_readfirstlane(s_list[i < n_items ? i : n_items - 1]);
    const int it = first + step * (int)(e & 0xffffu);
    const int t2 = div_magic(it, g.ix, g.mx), n = div_magic(t2, g.iy, g.my);
    return {n, PR * (t2 - n * g.iy), PC * (it - t2 * g.ix), (e >> 16) & 0xffu, e >> 24};
  };

  // ---- this wave's filter: taps x two blocks of 32 input channels x 16 output channels
  v4f wt[16][2];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const mie_bf16* f = g.filter + ((long long)(phase * (DC / 16) + 4 * ks + 2 * h + (cg >> 1)) * UP2X_UNITS * 2 + (cg & 1)) * DCO * EPS + (16 * q + pos) * EPS;
#pragma unroll
    for (int t = 0; t < 16; ++t) wt[t][h] = *reinterpret_cast<const v4f*>(f + (long long)t * 2 * DCO * EPS);
  }

  // ---- staging: slot tid + 512 i = 16 bytes (eight channels) of pixel (tid >> 4) + 32 i of the window
  int sid = tid;         // (opaque in every item, below: the places of all slots, kept from item to item, would be spilled)
  const bool has2 = a.x2 != nullptr;
  const mie_bf16* x2p = has2 ? a.x2 : a.x;
  // (masks that are not there: see k_upconv2x_pred)
  const uint8_t* m1p = a.xm != nullptr ? a.xm : reinterpret_cast<const uint8_t*>(a.x);
  const uint8_t* m2p = has2 && a.x2m != nullptr ? a.x2m : reinterpret_cast<const uint8_t*>(x2p);
  const unsigned m_all = (a.xm == nullptr ? 1u : 0u) | (has2 && a.x2m == nullptr ? 2u : 0u), m_use = has2 ? 3u : 1u;
  // pixel p of an item's window; edge pixels continue the plane
  auto window_pixel = [&](const Item& o, int p) -> unsigned {
    const int r = p / DSC, c = p - r * DSC;
    int y = o.y0 - 2 + py + r, x = o.x0 - 2 + px + c;
    y = y < 0 ? 0 : (y < H ? y : H - 1);
    x = x < 0 ? 0 : (x < W ? x : W - 1);
    return (unsigned)((o.n * H + y) * W + x);
  };
  auto load_slot = [&](const Item& o, int i, float4& va, float4& vb) {
    const unsigned eo = (window_pixel(o, (sid >> 4) + 32 * i) * DC + EPS * (sid & 15)) * 2u;      // bytes: below 2^32
    va = *reinterpret_cast<const float4*>(reinterpret_cast<const char*>(a.x) + eo);
    vb = *reinterpret_cast<const float4*>(reinterpret_cast<const char*>(x2p) + eo);
  };
  struct MaskBytes { unsigned a, b; };
  auto load_masks = [&](const Item& o) -> MaskBytes {
    const unsigned po = window_pixel(o, sid < DPIX ? sid : 0);
    return {m1p[po], m2p[po]};
  };
  auto store_masks = [&](int buf, const MaskBytes& m) {
    if (tid < 256) s_m[buf][tid] = (unsigned char)(((m.a != 0u ? 1u : 0u) | (m.b != 0u ? 2u : 0u) | m_all) & m_use);
  };
  auto store_slot = [&](int buf, int i, const float4& va, const float4& vb) {
    const int p = (sid >> 4) + 32 * i, at = p < DPIX ? p : DPIX;
    const unsigned ok = s_m[buf][p];
    const float4 z4 = make_float4(0.f, 0.f, 0.f, 0.f);
    float fa[8], fb[8], f[8];
    bf16x8_to_f32((ok & 1u) ? va : z4, fa);
    bf16x8_to_f32((ok & 2u) ? vb : z4, fb);
#pragma unroll
    for (int e = 0; e < 8; ++e) f[e] = fa[e] + fb[e];
    *reinterpret_cast<float4*>(&s_stage[buf][at * DLS + EPS * (sid & 15)]) = f32_to_bf16x8(f);
  };

  // ---- the rows this wave finishes: 4 ks .. 4 ks + 3 of the item, position pos, channels 16 q + 4 cg ..
  const unsigned row = 2u * (unsigned)wout;
  unsigned l_pix = (unsigned)(2 * pos + px), l_ch = (unsigned)(16 * q + 4 * cg);
  auto item_pix = [&](const Item& o) -> long long { return ((long long)o.n * hout + 2 * o.y0 + py) * wout + 2 * o.x0; };
  // (the first and the last row and column of positions belong to the strips)
  auto inner = [&](const Item& o, int r) -> bool {
    const int y = o.y0 + 4 * ks + r, x = o.x0 + pos;
    return (y > 0) & (y < H - 1) & (x > 0) & (x < W - 1);
  };
  auto tile_bit = [&](unsigned bits) -> bool { return ((bits >> (4 * ks + (pos >> 2))) & 1u) != 0u; };
  float4 r0[PR / 2];
  auto load_row = [&](const Item& o, int r) {      // (no branch around the load; lanes without a pixel read the item's first)
    const unsigned off = (tile_bit(o.act) & inner(o, r)) ? ((4 * ks + r) * row + l_pix) * DCO + l_ch : l_ch;
    r0[r] = *reinterpret_cast<const float4*>(reinterpret_cast<const char*>(a.res + item_pix(o) * DCO) + 4u * off);
  };

  // The output pixel mask of the four rows, a byte a lane: of row cg, position pos.  (Outside it the delta is zero and the
  // reservoir stays as it is; a ballot hands the bits round.)
  auto load_live = [&](const Item& o) -> unsigned {
    const unsigned p = (tile_bit(o.act) & inner(o, cg)) ? (4 * ks + cg) * row + 2 * pos + px : 0u;
    return (a.ts.pixmask + item_pix(o))[p];
  };

  // ---- before the first item: its window, the first slots of the second item's, the masks of the first three
  Item cur = item_at(0), nxt = item_at(1), after = item_at(2);
  float4 va[DRING], vb[DRING];
  store_masks(0, load_masks(cur));
  store_masks(1, load_masks(nxt));
  __syncthreads();
#pragma unroll
  for (int i0 = 0; i0 < DLD; i0 += DRING) {
#pragma unroll
    for (int i = i0; i < i0 + DRING && i < DLD; ++i) load_slot(cur, i, va[i - i0], vb[i - i0]);
#pragma unroll
    for (int i = i0; i < i0 + DRING && i < DLD; ++i) store_slot(0, i, va[i - i0], vb[i - i0]);
  }
#pragma unroll
  for (int i = 0; i < DRING; ++i) load_slot(nxt, i, va[i], vb[i]);
  MaskBytes masks = load_masks(after);
  __syncthreads();

  int par = 0;
  for (int i = 0; i < n_items; ++i, par ^= 1) {
    asm volatile("" : "+v"(sid), "+v"(l_pix), "+v"(l_ch));
    // ---- sums
    v4f acc[PR];
    unsigned live_b = 0u;
    unsigned long long live = 0ull;      // bit 16 * row + position
#pragma unroll
    for (int r = 0; r < PR; ++r) acc[r] = v4f{0.f, 0.f, 0.f, 0.f};
    {
      const mie_bf16* s = &s_stage[par][pos * DLS + 64 * ks + EPS * cg];
      constexpr int NF = 8 * SR, AHEAD = 2;          // fragments: block of channels, window column j, row r; two ahead
      v4f x[AHEAD + 1];
      auto fetch = [&](int f) { x[f % (AHEAD + 1)] = *reinterpret_cast<const v4f*>(s + (f % SR) * DSC * DLS + (f / SR % 4) * DLS + f / (4 * SR) * 32); };
#pragma unroll
      for (int f = 0; f < AHEAD; ++f) fetch(f);
#pragma unroll
      for (int f = 0; f < NF; ++f) {
        if (f + AHEAD < NF) fetch(f + AHEAD);
        const int u = f / SR;                        // the next window's slot u; then slot u + 4, of it or of the one after it
        if (f % SR == 2 && u < DLD) store_slot(par ^ 1, u, va[u % DRING], vb[u % DRING]);
        if (f % SR == 6 && (u + DRING) % 8 < DLD) load_slot(u + DRING < 8 ? nxt : after, (u + DRING) % 8, va[u % DRING], vb[u % DRING]);
        if (f == 0) live_b = load_live(cur);
        if (f == 3 * SR) live = __ballot(live_b != 0u);      // (two scalars from here on: what the sums leave of the registers is the rows')
        if (RES && f % SR == 9 && u < PR / 2) load_row(cur, u);
        __builtin_amdgcn_sched_barrier(0);
        const int h = f / (4 * SR), j = u % 4, r = f % SR;
#pragma unroll
        for (int t = 0; t < 4; ++t)
          if (r - t >= 0 && r - t < PR) acc[r - t] = mma16(wt[4 * t + j][h], x[f % (AHEAD + 1)], acc[r - t]);
        __builtin_amdgcn_sched_barrier(0);
      }
      // the rows the other wave finishes
#pragma unroll
      for (int r = 0; r < PR / 2; ++r) s_sum[wave ^ 4][r][lane] = ks == 0 ? acc[PR / 2 + r] : acc[r];
    }
    store_masks(par, masks);
    __syncthreads();      // sums exchanged; the next window is there, this one has been read
    v4f sum[PR / 2];
#pragma unroll
    for (int r = 0; r < PR / 2; ++r) {
      const v4f mine = ks == 0 ? acc[r] : acc[PR / 2 + r];
      sum[r] = mine + s_sum[wave][r][lane];
    }
    __syncthreads();      // the exchanged sums have been read
    const Item later = item_at(i + 3);
    masks = load_masks(later);
    const long long pix0 = item_pix(cur);
    const bool on = tile_bit(cur.act), zero = tile_bit(cur.old);
#pragma unroll
    for (int r = 0; r < PR / 2; ++r) {
      const unsigned off = ((4 * ks + r) * row + l_pix) * DCO + l_ch;
      mie_bf16* out = reinterpret_cast<mie_bf16*>(reinterpret_cast<char*>(a.out + pix0 * DCO) + 2u * off);
      float4 d = make_float4(sum[r][0], sum[r][1], sum[r][2], sum[r][3]);
      const bool in = inner(cur, r), keep = on & (((live >> (16 * r + pos)) & 1ull) != 0ull);
      if (RES) {
        const float4 q0 = r0[r], q1 = make_float4(q0.x + d.x, q0.y + d.y, q0.z + d.z, q0.w + d.w);
        if (keep & in) *reinterpret_cast<float4*>(reinterpret_cast<char*>(a.res + pix0 * DCO) + 4u * off) = q1;
        d = make_float4(mie_act(ACT, a.slope, q1.x) - mie_act(ACT, a.slope, q0.x), mie_act(ACT, a.slope, q1.y) - mie_act(ACT, a.slope, q0.y),
                        mie_act(ACT, a.slope, q1.z) - mie_act(ACT, a.slope, q0.z), mie_act(ACT, a.slope, q1.w) - mie_act(ACT, a.slope, q0.w));
      }
      if (!keep) d = make_float4(0.f, 0.f, 0.f, 0.f);
      if ((on | zero) & in) mie_st4(out, 0, d);
    }
    cur = nxt;
    nxt = after;
    after = later;
  }
}

}  // namespace

// Takes the shape of the batched bf16 network's last decoder on planes large enough to keep the resident grid busy
// (launches nothing and returns false otherwise; MIE_UPCONV_PERSIST=0 switches the kernel off, for measurements).
static bool persist_takes(const ConvArgsT<mie_bf16>& a, unsigned cap) {
  static const bool enabled = [] {
    const char* e = getenv("MIE_UPCONV_PERSIST");
    return e == nullptr || atoi(e) != 0;
  }();
  if (!enabled || a.c1 != C || a.cout != COUT || a.pad != 2 || a.refresh || a.filt_mc == nullptr || a.x3 || a.addend != nullptr) return false;
  if (a.x2 != nullptr && a.c2 != C) return false;
  return cap >= 4u * GRID && cap <= (1u << 20);      // small planes: one tile per workgroup is as good
}

bool mie_launch_upconv_persist(const ConvArgsT<mie_bf16>& a, unsigned cap, hipStream_t st) {
  if (!persist_takes(a, cap)) return false;
  const dim3 g(GRID), b(256);
  const PredTail none = {};
  if (a.res == nullptr) {
    hipLaunchKernelGGL((k_upconv64_persist<false, MIE_ACT_NONE>), g, b, 0, st, a, none);
    return true;
  }
  switch (a.act) {
    case MIE_ACT_NONE: hipLaunchKernelGGL((k_upconv64_persist<true, MIE_ACT_NONE>), g, b, 0, st, a, none); return true;
    case MIE_ACT_RELU: hipLaunchKernelGGL((k_upconv64_persist<true, MIE_ACT_RELU>), g, b, 0, st, a, none); return true;
    case MIE_ACT_LEAKY_RELU: hipLaunchKernelGGL((k_upconv64_persist<true, MIE_ACT_LEAKY_RELU>), g, b, 0, st, a, none); return true;
    default: return false;                                      // sigmoid / tanh epilogues: the one-tile kernel
  }
}

// The same with the network's tail fused in (a.out is not written): see PredTail.
bool mie_launch_upconv_pred_persist(const ConvArgsT<mie_bf16>& a, const mie_bf16* skip, const uint8_t* skip_mask,
                                    const float* pred_w, float* pred_res, mie_bf16* pred_out, int pred_act,
                                    float pred_slope, unsigned cap, hipStream_t st) {
  if (!persist_takes(a, cap) || a.res == nullptr) return false;
  PredTail pt;
  pt.skip = skip; pt.skip_mask = skip_mask; pt.w = pred_w; pt.res = pred_res; pt.out = pred_out; pt.act = pred_act;
  pt.slope = pred_slope;
  pt.flags = nullptr;
  const dim3 g(GRID), b(256);
  switch (a.act) {
    case MIE_ACT_NONE: hipLaunchKernelGGL((k_upconv64_persist<true, MIE_ACT_NONE, true>), g, b, 0, st, a, pt); return true;
    case MIE_ACT_RELU: hipLaunchKernelGGL((k_upconv64_persist<true, MIE_ACT_RELU, true>), g, b, 0, st, a, pt); return true;
    case MIE_ACT_LEAKY_RELU: hipLaunchKernelGGL((k_upconv64_persist<true, MIE_ACT_LEAKY_RELU, true>), g, b, 0, st, a, pt); return true;
    default: return false;
  }
}

// The same with the inner tiles at the resolution of the inputs (filter_up: mie_pack_filter_up2x's, bf16).
template <int ACT>
static void launch_up2x_pred(const ConvArgsT<mie_bf16>& a, const PredTail& pt, const PhaseItems& g, hipStream_t st) {
  hipLaunchKernelGGL((k_upconv64_persist<true, ACT, true, true>), dim3(GRID), dim3(256), 0, st, a, pt);
  hipLaunchKernelGGL((k_upconv2x_pred<ACT>), dim3(PGRID), dim3(PTHR), 0, st, a, pt, g);
}
bool mie_launch_upconv2x_pred_persist(const ConvArgsT<mie_bf16>& a, const mie_bf16* filter_up, const uint32_t* flags,
                                      const mie_bf16* skip, const uint8_t* skip_mask, const float* pred_w, float* pred_res,
                                      mie_bf16* pred_out, int pred_act, float pred_slope, unsigned cap, hipStream_t st) {
  if (!persist_takes(a, cap) || a.res == nullptr || a.ts.tiles_y < 3 || a.ts.tiles_x < 3 || a.ts.w >= (1 << 20)) return false;
  PredTail pt;
  pt.skip = skip; pt.skip_mask = skip_mask; pt.w = pred_w; pt.res = pred_res; pt.out = pred_out; pt.act = pred_act;
  pt.slope = pred_slope; pt.flags = flags;
  PhaseItems g;
  g.filter = filter_up;
  g.iy = (a.ts.tiles_y - 2 + 1) / 2;
  g.ix = (a.ts.tiles_x - 2 + 3) / 4;
  g.total = a.ts.n * g.iy * g.ix;
  if (((g.total + 7) / 8 + PGRID / 16 - 1) / (PGRID / 16) > PITEMS) return false;      // (no plane of 2^20 tiles has as many)
  g.my = 0xffffffffu / (unsigned)g.iy + 1u;
  g.mx = 0xffffffffu / (unsigned)g.ix + 1u;
  switch (a.act) {
    case MIE_ACT_NONE: launch_up2x_pred<MIE_ACT_NONE>(a, pt, g, st); return true;
    case MIE_ACT_RELU: launch_up2x_pred<MIE_ACT_RELU>(a, pt, g, st); return true;
    case MIE_ACT_LEAKY_RELU: launch_up2x_pred<MIE_ACT_LEAKY_RELU>(a, pt, g, st); return true;
    default: return false;
  }
}

// The inner positions of mie_upconv2x_masked's layer, 128 -> 64 channels in bf16 without an addend (a.h_in, a.w_in: the input
// plane).  From three items a workgroup on (192 in all): there both forms take as long (1x120x160, 150 items, 38.1 us with
// k_upconv2x against 36.8; 3x54x76, 210: 32.0 against 31.2; 4x66x88, 216: 48.2 against 48.3), below it the fill of 128
// registers with the filter weighs more, and above it this one wins (2x120x160, 300: 67.8 against 58.2).  False, launching
// nothing, for other calls.
bool mie_launch_upconv2x_rows(const ConvArgsT<mie_bf16>& a, const uint32_t* flags, hipStream_t st) {
  if (a.c1 != DC || a.cout != DCO || a.refresh || a.addend != nullptr || a.ts.w >= (1 << 20) || a.h_in < 3 || a.w_in < 3) return false;
  PhaseItems g;
  g.filter = a.filt_mc;
  g.iy = (a.ts.tiles_y + 1) / 2;
  g.ix = (a.ts.tiles_x + 3) / 4;
  const long long total = (long long)a.ts.n * g.iy * g.ix;
  if (total > (long long)DITEMS * (PGRID / 32) * 8 - 64 || 4 * total < 3 * PGRID) return false;
  g.total = (int)total;
  g.my = 0xffffffffu / (unsigned)g.iy + 1u;
  g.mx = 0xffffffffu / (unsigned)g.ix + 1u;
  const dim3 grid(PGRID), block(PTHR);
  if (a.res == nullptr) {
    if (a.act != MIE_ACT_NONE) return false;
    hipLaunchKernelGGL((k_upconv2x_rows<false, MIE_ACT_NONE>), grid, block, 0, st, a, flags, g);
    return true;
  }
  switch (a.act) {
    case MIE_ACT_NONE: hipLaunchKernelGGL((k_upconv2x_rows<true, MIE_ACT_NONE>), grid, block, 0, st, a, flags, g); return true;
    case MIE_ACT_RELU: hipLaunchKernelGGL((k_upconv2x_rows<true, MIE_ACT_RELU>), grid, block, 0, st, a, flags, g); return true;
    case MIE_ACT_LEAKY_RELU: hipLaunchKernelGGL((k_upconv2x_rows<true, MIE_ACT_LEAKY_RELU>), grid, block, 0, st, a, flags, g); return true;
    default: return false;
  }
}
