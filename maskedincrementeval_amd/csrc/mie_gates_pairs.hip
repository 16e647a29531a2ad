// The gates conv of a ConvLSTM in bf16 on planes of many tiles: k_conv_mfma<..., GATES> with two tiles a workgroup.
//
// There every 1 KB of filter that a wave reads from L2 serves two MFMAs, one for each half of its tile, and a CU takes in 20
// to 30 bytes a cycle of vector memory with the matrix cores at a quarter to a third; here it serves four.  A wave holds 64
// sums for its 32 columns (two workgroups a CU: the sums of two tiles, six units of filter on their way, the next chunk's
// slots and, in the last chunk, the first tile's reservoirs).  The filter is read in the order it lies in -- 16 channels,
// tap after tap -- so that a unit is a step of one scalar; the next chunk's slots are asked for one a unit.
// Measured, every tile active, one tile a workgroup -> two: 64+64->256 at 8x240x320 677 -> 633 us, 128+128->512 at 8x120x160
// 527 -> 475, 256+256->1024 at 8x60x80 477 -> 413 (878 TFLOP/s; a large product of this type reaches 1115), 128+128->512 at
// 2x66x88 51.2 -> 45.6, at 2x50x70 32.0 -> 30.1.  Whole passes: 8x480x640 2487 -> 2451 us (20 % active), 1669 -> 1646 (1 %),
// 2x200x280 293 -> 290.  The plain convs of 256 channels lose by it (8x60x80 65 -> 74 us: 640 workgroups are one round and a
// quarter), so they keep one tile.
// The second tile costs a workgroup half as long again as one alone takes, which pays where it saves a round of workgroups:
// while the active tiles alone are at most one workgroup a CU, each has its own (a sparse step on a large plane; the sums are
// in the same order either way).  64+64->256 at 240x320, two -> one: 13 tiles 13.1 -> 8.6 us, 81 tiles 16.1 -> 10.1;
// 128+128->512 at 120x160, 57 tiles 21.7 -> 14.5; 256+256->1024 at 60x80, 26 tiles 32.1 -> 21.3.  Just above the line (274,
// 280 workgroups of one tile) both forms take as long (16.1 and 15.7 us; 34.5 and 35.1).
#include "mie_conv_mfma_impl.h"

namespace {

typedef mie_bf16 T;
constexpr int K = 3, EPS = 8, SUB = 16, IT = 10, CC = 64, Q4 = CC / EPS;
constexpr int LS = CC + EPS, RP = row_pitch_dw(IT, LS / 2, 1) * 2, STAGE = IT * RP;      // elements: pixel, row, tile
constexpr int NQ = CC / SUB, UPC = K * K * NQ;                                           // units of a chunk: 36
constexpr int RING = 6, PD = RING - 1;
constexpr int COLS = 128;
static_assert(UPC % RING == 0, "a ring slot means the same registers in every chunk");
static_assert(256 % Q4 == 0, "a thread's channels are the same in all of its slots");
constexpr int ONE_MOST = 256;                                                            // workgroups of one tile, at most
constexpr int SMEM = (2 * STAGE * 2 > 64 * COLS * 4 ? 2 * STAGE * 2 : 64 * COLS * 4) / 4;

// The workgroup's NT tiles (the second of two may be none: `second`).
template <int NT>
__device__ __forceinline__ void gates_tiles(const ConvArgsT<T>& a, T* const sbuf, float* const smem, const int (&n)[2], const int (&y0)[2], const int (&x0)[2],
                                            const bool second, const int co0) {
  constexpr int NSLOT = NT * IT * IT * Q4, NLD = (NSLOT + 255) / 256;                    // 800 or 1600, 4 or 7
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, l32 = lane & 31, half = lane >> 5;
  const int hout = a.ts.h, wout = a.ts.w, cout = a.cout;

  // which of this thread's outputs lie on a pixel of the mask: bit 8 * t + i, item i of tile t
  constexpr int PER = 2;
  int live_at[NT * PER];
  unsigned live_in = 0u;
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const int p = (tid + 256 * i) >> 3;
      const int oy = y0[t] + (p >> 3), ox = x0[t] + (p & 7);
      const bool k = oy < hout && ox < wout && (t == 0 || second);
      live_at[t * PER + i] = k ? (n[t] * hout + oy) * wout + ox : 0;
      live_in |= (k ? 1u : 0u) << (t * PER + i);
    }

  // ---- staging: slot tid + 256 * i is 8 channels of a pixel of a tile's 10x10 window ---------------------------------------
  const int q8 = EPS * (tid & 7);
  int st_po[NLD], st_lds[NLD];
  unsigned inb = 0u, ok1 = 0u, ok2 = 0u;
#pragma unroll
  for (int i = 0; i < NLD; ++i) {
    const int s = (tid + 256 * i) >> 3, t = NT == 2 && s >= IT * IT ? 1 : 0, pix = s - t * (IT * IT);
    const int row = pix / IT, col = pix - row * IT;
    st_lds[i] = t * STAGE + row * RP + col * LS + q8;
    const int iy = (t ? y0[1] : y0[0]) - a.pad + row, ix = (t ? x0[1] : x0[0]) - a.pad + col;
    const bool in = s < NT * IT * IT && iy >= 0 && iy < a.h_in && ix >= 0 && ix < a.w_in && (t == 0 || second);
    st_po[i] = in ? ((t ? n[1] : n[0]) * a.h_in + iy) * a.w_in + ix : 0;
    inb |= (in ? 1u : 0u) << i;
  }
  const int nch1 = a.c1 / CC, nch = nch1 + (a.x2 != nullptr ? a.c2 / CC : 0);
  float4 st[NLD];
  unsigned st_ok = 0u;                                       // which of them count
  // (unconditional loads; slots that do not count read pixel 0)
  auto load_slot = [&](int i, const T* xin, unsigned cs, unsigned ci) {
    const unsigned o = ((st_ok >> i) & 1u) ? (unsigned)st_po[i] * cs : 0u;
    st[i] = *reinterpret_cast<const float4*>(reinterpret_cast<const char*>(xin) + 2u * (o + ci));
  };
  auto store_slots = [&]() {
#pragma unroll
    for (int i = 0; i < NLD; ++i)
      if (tid + 256 * i < NSLOT) {
        const bool k = (st_ok >> i) & 1u;
        *reinterpret_cast<float4*>(sbuf + st_lds[i]) = make_float4(k ? st[i].x : 0.f, k ? st[i].y : 0.f, k ? st[i].z : 0.f, k ? st[i].w : 0.f);
      }
  };

  // ---- operands -----------------------------------------------------------------------------------------------------------
  const unsigned b_lane = (unsigned)((half * cout + co0 + 32 * wave + l32) * EPS) * 2u;
  // units of a chunk in the order of the filter copy: 16 channels x (tap after tap)
  unsigned unit_b = (unsigned)cout * (2 * 2 * EPS);          // bytes of one
  auto load_b = [&](const char* ub, int u) { return *reinterpret_cast<const float4*>(ub + u * unit_b + b_lane); };
  const T* const a0 = sbuf + ((l32 >> 3) * RP + (l32 & 7) * LS + EPS * half);
  auto load_a = [&](int u, float4 (&x)[2 * NT]) {
    const int tap = u % (K * K), q = u / (K * K);
#pragma unroll
    for (int mb = 0; mb < 2 * NT; ++mb)
      x[mb] = *reinterpret_cast<const float4*>(a0 + (mb >> 1) * STAGE + (4 * (mb & 1) + tap / K) * RP + tap % K * LS + SUB * q);
  };
  v16f acc[2 * NT];
#pragma unroll
  for (int mb = 0; mb < 2 * NT; ++mb)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[mb][r] = 0.f;

  // first chunk: where at least four follow, its loads go out for every pixel, before the mask bytes are there
  const bool early = nch >= 4;
  if (early) {
    st_ok = inb;
#pragma unroll
    for (int i = 0; i < NLD; ++i) load_slot(i, a.x, a.c1, q8);
  }
  {
    const uint8_t* const x2m = a.x2 != nullptr ? a.x2m : nullptr;
    unsigned b1[NLD], b2[NLD];
    mie_mask_ask(a.xm, a.filt_mc, st_po, b1);
    mie_mask_ask(x2m, a.filt_mc, st_po, b2);
    mie_mask_asked();
    ok1 = mie_mask_take(a.xm, b1, inb);
    ok2 = mie_mask_take(x2m, b2, a.x2 != nullptr ? inb : 0u);
  }
  st_ok = ok1;
  if (!early) {
#pragma unroll
    for (int i = 0; i < NLD; ++i) load_slot(i, a.x, a.c1, q8);
  }
  const char* ub = reinterpret_cast<const char*>(a.filt_mc);      // (x2's channels lie behind x's there)
  float4 ring[RING];
#pragma unroll
  for (int u = 0; u < PD; ++u) ring[u] = load_b(ub, u);
  const uint8_t* const cp_m = a.g_cpd != nullptr ? a.g_cpm : nullptr;
  unsigned live_b[NT * PER], cp_b[NT * PER];
  mie_mask_ask(a.ts.pixmask, a.filt_mc, live_at, live_b);
  mie_mask_ask(cp_m, a.filt_mc, live_at, cp_b);
  mie_mask_asked();
  store_slots();
  __syncthreads();
  const unsigned live = mie_mask_take(a.ts.pixmask, live_b, live_in);
  const unsigned cp_live = mie_mask_take(cp_m, cp_b, a.g_cpd != nullptr ? live : 0u);
  // the reservoir values of a tile's two items, asked for long before they are needed (lanes without any read one fixed address)
  GateItem item[2];
  auto item_at = [&](int t, int i, long long& ho, long long& go) {
    const int idx = tid + 256 * i, p = idx >> 3, g4 = idx & 7;
    const long long pix = ((long long)n[t] * hout + (y0[t] + (p >> 3))) * wout + x0[t] + (p & 7);
    ho = pix * a.hid + co0 / 4 + 4 * g4;
    go = pix * cout + co0 + 16 * g4;
  };
  auto item_load = [&](int t, int i) {
    long long ho, go;
    item_at(t, i, ho, go);
    conv_gates_load<T>(a, (live >> (t * PER + i)) & 1u, (cp_live >> (t * PER + i)) & 1u, ho, go, item[i]);
  };
  // one chunk; with the next one's slots, or (LAST) the first tile's reservoirs, asked for between its first units
  auto chunk = [&](const char* ub_next, const T* xin, unsigned cs, unsigned ci, auto LAST) {
    constexpr bool last = decltype(LAST)::value;
    float4 av[2][2 * NT];
    load_a(0, av[0]);
#pragma unroll
    for (int u = 0; u < UPC; ++u) {
      const int up = u + PD;
      if (up < UPC) ring[up % RING] = load_b(ub, up);
      else if (!last) ring[up % RING] = load_b(ub_next, up - UPC);
      if (!last && u < NLD) load_slot(u, xin, cs, ci);
      if (last && (u == 2 || u == 8)) item_load(0, u == 8 ? 1 : 0);
      if (u + 1 < UPC) load_a(u + 1, av[(u + 1) & 1]);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int mb = 0; mb < 2 * NT; ++mb) mma_unit(acc[mb], av[u & 1][mb], ring[u % RING], T());
      __builtin_amdgcn_sched_barrier(0);
    }
    __syncthreads();
  };
  for (int c = 1; c < nch; ++c) {
    asm volatile("" : "+s"(unit_b));      // (else 36 multiples of it are kept)
    const bool sec = c >= nch1;
    st_ok = sec ? ok2 : ok1;
    chunk(ub + UPC * unit_b, sec ? a.x2 : a.x, sec ? a.c2 : a.c1, (sec ? c - nch1 : c) * CC + q8, std::false_type{});
    store_slots();
    __syncthreads();
    ub += UPC * unit_b;
  }
  asm volatile("" : "+s"(unit_b));
  chunk(ub, a.x, 0, 0, std::true_type{});

  // ---- epilogue, a tile at a time: sums to LDS, then as in k_conv_mfma ------------------------------------------------------
  auto epilogue = [&](auto TT) {
    constexpr int t = decltype(TT)::value;
#pragma unroll
    for (int mb = 0; mb < 2; ++mb)
#pragma unroll
      for (int r = 0; r < 16; ++r) smem[(mb * 32 + 8 * (r >> 2) + 4 * half + (r & 3)) * COLS + 32 * wave + l32] = acc[2 * t + mb][r];
    __syncthreads();
    float4 dg[2][4];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) dg[i][j] = *reinterpret_cast<const float4*>(&smem[((tid + 256 * i) >> 3) * COLS + 16 * (tid & 7) + 4 * j]);
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      long long ho, go;
      item_at(t, i, ho, go);
      GateItem g = item[i];
      if constexpr (NT == 2 && t == 0) item_load(1, i);      // (this item's registers are free)
      if ((live_in >> (t * PER + i)) & 1u)
        conv_gates_item<T>(a, (live >> (t * PER + i)) & 1u, (cp_live >> (t * PER + i)) & 1u, ho, go, dg[i], g);
    }
  };
  epilogue(std::integral_constant<int, 0>{});
  if constexpr (NT == 2) {
    if (!second) return;
    __syncthreads();
    epilogue(std::integral_constant<int, 1>{});
  }
}

__global__ __launch_bounds__(256, 2) void k_gates_pairs(ConvArgsT<T> a) {
  __shared__ __attribute__((aligned(16))) float smem[SMEM];
  T* const sbuf = reinterpret_cast<T*>(smem);
  const int bx = blockIdx.x + conv_args_entry_zero(a);
  // ---- which pair of list positions and which slab: the order of k_conv_mfma with pairs for tiles -------------------------
  const int cap = a.ts.n * a.ts.tiles_y * a.ts.tiles_x;
  const int n_act = a.ts.counts[MIE_CNT_ACTIVE], n_st = a.ts.counts[MIE_CNT_STALE];
  if (n_act < 0 || n_st < 0 || n_act > cap || n_st > cap) return;
  // few active tiles: one a workgroup (the launcher's grid has room for them)
  const int ns = (int)gridDim.y;
  const bool one = n_act * ns <= ONE_MOST;
  const int p_act = one ? n_act : (n_act + 1) >> 1, p_st = (n_st + 1) >> 1;
  const int w_act = p_act * ns, w_st = p_st * ns;
  const int lg = __builtin_ctz(a.xcd_fs), sh = 3 - lg, up = (1 << sh) - 1, spg = ns >> lg;
  const int g_act = w_act >> lg, g_st = w_st >> lg;            // of a group of slabs
  const int c_act = (g_act + up) >> sh, c_st = (g_st + up) >> sh;
  const int xcd = bx & 7, k = xcd & up, slot = (int)blockIdx.y * ((int)gridDim.x >> 3) + (bx >> 3);
  const bool active = slot < c_act;
  const int v = active ? k * c_act + slot : k * c_st + (slot - c_act);
  if (v >= (active ? g_act : g_st) || (!active && slot - c_act >= c_st)) return;
  const int pair = mie_tile_div(v, spg, a.xcd_m);
  const int co0 = ((xcd >> sh) * spg + (v - pair * spg)) * COLS;
  const int count = active ? n_act : n_st, at = one && active ? pair : 2 * pair;
  const int32_t* const list = active ? a.ts.tiles : a.ts.stale;
  const int tiles[2] = {list[at], list[at + 1 < count ? at + 1 : at]};
  const bool second = at + 1 < count && !(one && active);
  int n[2], y0[2], x0[2];
#pragma unroll
  for (int t = 0; t < 2; ++t) {
    if (tiles[t] < 0 || tiles[t] >= cap) return;      // corrupt list entry: skip rather than touch memory
    const int ty = mie_tile_div(tiles[t], a.ts.tiles_x, a.ts.mx);
    x0[t] = (tiles[t] - ty * a.ts.tiles_x) * MIE_TILE;
    n[t] = mie_tile_div(ty, a.ts.tiles_y, a.ts.my);
    y0[t] = (ty - n[t] * a.ts.tiles_y) * MIE_TILE;
  }
  if (!active) {
    auto zero = [&](int n, int y0, int x0) {
      for (int idx = threadIdx.x; idx < 64 * (COLS / 16); idx += 256) {
        const int p = idx >> 3, g4 = idx & 7, oy = y0 + (p >> 3), ox = x0 + (p & 7);
        if (oy >= a.ts.h || ox >= a.ts.w) continue;
        const long long o = (((long long)n * a.ts.h + oy) * a.ts.w + ox) * a.hid + co0 / 4 + 4 * g4;
        mie_st4(a.g_dh, o, make_float4(0.f, 0.f, 0.f, 0.f));
        mie_st4(a.g_dc, o, make_float4(0.f, 0.f, 0.f, 0.f));
      }
    };
    zero(n[0], y0[0], x0[0]);
    if (second) zero(n[1], y0[1], x0[1]);
    return;
  }
  if (one) gates_tiles<1>(a, sbuf, smem, n, y0, x0, false, co0);
  else gates_tiles<2>(a, sbuf, smem, n, y0, x0, second, co0);
}

}  // namespace

// From 256 workgroups (one a CU) on: at 168 (256+256->1024 at 2x25x35) one tile a workgroup is ahead, 35.5 us against 38.6; at
// 256 (2x50x70, above) two are.
bool mie_launch_gates_pairs(const ConvArgsT<mie_bf16>& a0, unsigned cap, hipStream_t st) {
  static const int least = [] { const char* e = getenv("MIE_GATES_PAIRS"); return e ? atoi(e) : 256; }();      // tuning knob
  ConvArgsT<T> a = a0;
  if (a.hid <= 0 || a.cout != 4 * a.hid || a.cout % COLS != 0 || a.c1 % CC != 0 || a.c2 % CC != 0 || a.pad != 1 || forced_slab() != 0) return false;
  if ((long long)a.ts.n * a.h_in * a.w_in * (a.c1 > a.c2 ? a.c1 : a.c2) >= 1LL << 31) return false;      // 32-bit offsets
  const unsigned pairs = cap / 2 + 1;
  if (least == 0 || (long long)pairs * (a.cout / COLS) < least) return false;
  // (of at most ONE_MOST workgroups of one tile half are more than the pairs have)
  const unsigned gx = xcd_plan(a, pairs + ONE_MOST / 2 / (a.cout / COLS) + 1, a.cout / COLS, K);
  if (a.xcd_fs == 0) return false;
  hipLaunchKernelGGL(k_gates_pairs, dim3(gx, a.cout / COLS), dim3(256), 0, st, a);
  return true;
}
