// Shared host/device helpers of libmie_hip.so (gfx950 only).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <stdio.h>
#include <stdarg.h>

#include <mutex>

// The C ABI is the only thing exported from the library.
#pragma GCC visibility push(default)
#include "../../include/mie.h"
#pragma GCC visibility pop

#define MIE_WAVE 64

// bf16 deltas (MIE_DTYPE_BF16): the compiler's native type; conversions from fp32 round to
// nearest even (v_cvt_pk_bf16_f32 on gfx950), conversions to fp32 are exact.
typedef __bf16 mie_bf16;
typedef __bf16 mie_bf16x4 __attribute__((ext_vector_type(4)));
typedef __bf16 mie_bf16x8 __attribute__((ext_vector_type(8)));

// Scalar load / store of a delta element as fp32.
static __device__ __forceinline__ float mie_ld(const float* p, long long i) { return p[i]; }
static __device__ __forceinline__ float mie_ld(const mie_bf16* p, long long i) { return (float)p[i]; }
static __device__ __forceinline__ void mie_st(float* p, long long i, float v) { p[i] = v; }
static __device__ __forceinline__ void mie_st(mie_bf16* p, long long i, float v) { p[i] = (mie_bf16)v; }
// Four adjacent elements at once (i a multiple of 4, p + i 16-byte / 8-byte aligned).
static __device__ __forceinline__ float4 mie_ld4(const float* p, long long i) { return *reinterpret_cast<const float4*>(p + i); }
static __device__ __forceinline__ float4 mie_ld4(const mie_bf16* p, long long i) {
  const mie_bf16x4 b = *reinterpret_cast<const mie_bf16x4*>(p + i);
  return make_float4((float)b[0], (float)b[1], (float)b[2], (float)b[3]);
}
static __device__ __forceinline__ void mie_st4(float* p, long long i, const float4& v) { *reinterpret_cast<float4*>(p + i) = v; }
static __device__ __forceinline__ void mie_st4(mie_bf16* p, long long i, const float4& v) {
  mie_bf16x4 b;
  b[0] = (mie_bf16)v.x; b[1] = (mie_bf16)v.y; b[2] = (mie_bf16)v.z; b[3] = (mie_bf16)v.w;
  *reinterpret_cast<mie_bf16x4*>(p + i) = b;
}

// Bytes of a mask (NULL: every one set) at N places, all of them readable: asked for by mie_mask_ask, taken as bits, of those
// in `want`, by mie_mask_take.  The loads are unconditional, from a pointer chosen beforehand (`any`: an address that can be
// read), and a kernel puts mie_mask_asked between all that it asks for and what it takes.  Behind a condition, or left to
// the compiler's order, each byte is waited for before the next is asked for, and 8 to 20 trips to L2 one after the other
// are several microseconds of every workgroup.  Measured over whole passes: fp32 1x64x96 196 -> 187 us, 1x264x352 469 ->
// 457; bf16 2x200x280 314 -> 301, 8x480x640 2663 -> 2561; optical flow 1x256x256 506 -> 480.
template <int N>
__device__ __forceinline__ void mie_mask_ask(const uint8_t* m, const void* any, const int (&at)[N], unsigned (&b)[N]) {
  typedef const __attribute__((address_space(1))) uint8_t* global_bytes;
  const global_bytes p = (global_bytes)(m == nullptr ? static_cast<const uint8_t*>(any) : m);
  const int keep = m == nullptr ? 0 : -1;
#pragma unroll
  for (int i = 0; i < N; ++i) b[i] = p[at[i] & keep];
}
__device__ __forceinline__ void mie_mask_asked() { __builtin_amdgcn_sched_barrier(0); }
template <int N>
__device__ __forceinline__ unsigned mie_mask_take(const uint8_t* m, const unsigned (&b)[N], unsigned want) {
  unsigned bits = 0u;
#pragma unroll
  for (int i = 0; i < N; ++i) {
    unsigned v = b[i];
    asm volatile("" : "+v"(v));      // (here, not where it was asked for)
    bits |= (v != 0u ? 1u : 0u) << i;
  }
  return (m == nullptr ? ~0u : bits) & want;
}

// Between what lanes of one wave write to LDS and what others of it read: LDS requests of a wave are served in order, so
// only the compiler has to keep it, which the barrier alone (it touches no memory) does not ask of it.
__device__ __forceinline__ void mie_wave_order() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// ---- host side: launches that share a workspace ----------------------------
// The two launches of a split form belong together: between them the workspace holds the partial sums.  Threads that
// enqueue on one stream with one workspace take turns pair by pair (the lock is held while two launches are enqueued).
inline std::mutex& mie_split_launches() {
  static std::mutex m;
  return m;
}

// ---- host side: error reporting -------------------------------------------
void mie_set_error(const char* fmt, ...);
void mie_clear_error();

#define MIE_REQUIRE(cond, code, ...)        \
  do {                                      \
    if (!(cond)) {                          \
      mie_set_error(__VA_ARGS__);           \
      return (code);                        \
    }                                       \
  } while (0)

// Status of the launch that was just enqueued.
static inline int mie_check_launch(const char* what) {
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) {
    mie_set_error("%s: launch failed: %s", what, hipGetErrorString(e));
    return MIE_ERR_LAUNCH;
  }
  return MIE_OK;
}

static inline bool mie_aligned(const void* p, size_t a) {
  return (reinterpret_cast<uintptr_t>(p) & (a - 1)) == 0;
}

// Validates the pointers and geometry of a tile set (host side only).
int mie_check_tileset(const mie_tileset* ts, const char* who);

static inline int mie_div_up(int a, int b) { return (a + b - 1) / b; }

// ---- device side ------------------------------------------------------------
// Plain-old-data view of a tile set passed to kernels by value.
struct TileSetDev {
  int n, h, w;
  int tiles_y, tiles_x;
  unsigned my, mx;                // mie_tile_div
  const uint8_t* pixmask;
  const int32_t* tiles;
  const int32_t* stale;
  const int32_t* counts;
};

// t / d for a tile number t: a multiply by what the host worked out instead of a division by a run-time value, 30 instructions in
// a chain of which every workgroup had two ahead of its first load.  floor((2 t + 1) m / 2^32) with m = ceil(2^31 / d): (2 t + 1) /
// (2 d) has the floor of t / d and is at least 1 / (2 d) below the next whole number, and what m is too large by adds less
// than (2 t + 1) / 2^32.  m = 0 (a plane so large that this is not below 1 / (2 d)): the division.
static inline unsigned mie_tile_magic(long long tiles, int d) {
  return (2 * tiles + 1) * 2 * d < (1LL << 32) ? (unsigned)(((1LL << 31) + d - 1) / d) : 0u;
}
__device__ __forceinline__ int mie_tile_div(int t, int d, unsigned m) {
  return m != 0u ? (int)__umulhi(2u * (unsigned)t + 1u, m) : t / d;
}

static inline TileSetDev mie_dev_tileset(const mie_tileset* ts) {
  TileSetDev d;
  d.n = ts->n; d.h = ts->h; d.w = ts->w;
  d.tiles_y = mie_div_up(ts->h, MIE_TILE);
  d.tiles_x = mie_div_up(ts->w, MIE_TILE);
  const long long tiles = (long long)d.n * d.tiles_y * d.tiles_x;
  d.my = mie_tile_magic(tiles, d.tiles_y);
  d.mx = mie_tile_magic(tiles, d.tiles_x);
  d.pixmask = ts->pixmask; d.tiles = ts->tiles; d.stale = ts->stale;
  d.counts = ts->counts;
  return d;
}

// Which tile block `b` of a capacity-sized grid works on.
//   returns 0: nothing to do (b beyond active + stale)
//           1: active tile   2: stale tile (zero its delta)
// (n, y0, x0) = batch index and top-left output pixel of the tile.
// The same with the counts and the list entry tiles[b] already loaded by the caller (`spec`; any value
// if b is not an active position).
__device__ __forceinline__ int mie_pick_tile_loaded(const TileSetDev& ts, int b, int spec, int n_active,
                                                    int n_stale, int& n, int& y0, int& x0) {
  const int cap = ts.n * ts.tiles_y * ts.tiles_x;
  if (n_active < 0 || n_stale < 0 || n_active > cap || n_stale > cap) return 0;   // corrupt counts
  int tile, kind;
  if (b < 0) {
    return 0;
  } else if (b < n_active) {
    tile = spec;
    kind = 1;
  } else if (b < n_active + n_stale) {
    tile = ts.stale[b - n_active];
    kind = 2;
  } else {
    return 0;
  }
  if (tile < 0 || tile >= cap) return 0;    // corrupt list entry: skip rather than touch memory
  const int t2 = mie_tile_div(tile, ts.tiles_x, ts.mx), tx = tile - t2 * ts.tiles_x;
  n = mie_tile_div(t2, ts.tiles_y, ts.my);
  const int ty = t2 - n * ts.tiles_y;
  y0 = ty * MIE_TILE;
  x0 = tx * MIE_TILE;
  return kind;
}

// The list entry is fetched together with the counts (one memory round trip instead of two); whether it is valid is decided
// afterwards.  Asked for by mie_tile_ask, and taken by mie_tile_take: a kernel may put other loads between the two.
// (With this, the divisions by mie_tile_div and the arguments in one batch, whole passes: fp32 1x64x96 169.1 -> 163.1 us, 1x128x128
// 237.5 -> 231.1, optical flow 1x256x256 362.0 -> 355.2 and 450.9 -> 444.6; planes of many tiles as before.)
struct TileAsk {
  int spec, n_active, n_stale;
};
__device__ __forceinline__ TileAsk mie_tile_ask(const TileSetDev& ts, int b) {
  const int cap = ts.n * ts.tiles_y * ts.tiles_x;
  TileAsk k;
  k.spec = __builtin_amdgcn_readfirstlane(ts.tiles[(b >= 0 && b < cap) ? b : 0]);
  k.n_active = __builtin_amdgcn_readfirstlane(ts.counts[MIE_CNT_ACTIVE]);
  k.n_stale = __builtin_amdgcn_readfirstlane(ts.counts[MIE_CNT_STALE]);
  return k;
}
__device__ __forceinline__ int mie_tile_take(const TileSetDev& ts, int b, TileAsk& k, int& n, int& y0, int& x0) {
  // (all three taken here: left to itself the compiler moves the entry's load behind the test of the counts)
  asm("" : "+s"(k.spec), "+s"(k.n_active), "+s"(k.n_stale));
  return mie_pick_tile_loaded(ts, b, k.spec, k.n_active, k.n_stale, n, y0, x0);
}
__device__ __forceinline__ int mie_pick_tile(const TileSetDev& ts, int b, int& n, int& y0, int& x0) {
  TileAsk k = mie_tile_ask(ts, b);
  return mie_tile_take(ts, b, k, n, y0, x0);
}

// Whether block `b` of a capacity-sized grid is beyond the active and the stale tiles.
__device__ __forceinline__ bool mie_no_tile(const TileSetDev& ts, int b) {
  return b >= ts.counts[MIE_CNT_ACTIVE] + ts.counts[MIE_CNT_STALE];
}

// Masks first: whether a kernel of little else than loads waits for its mask bytes before it asks for values, so that masked
// pixels are not fetched.  It is a trip to memory more.  That pays where what could be fetched is more than the L2s keep from one
// layer to the next -- known to the launcher, which then takes a kernel with both forms: where there is nothing to gain, the
// branch alone costs 4 to 6 % of a small plane's few microseconds -- and where the step is in between: 4 MB and more
// (`per_tile` bytes each) in active tiles, or latency is all there is, and fewer than 7 of 8 tiles active, or the masks of the
// active ones tend to be full.  Figures stand beside the launchers.
__device__ __forceinline__ bool mie_masks_first(const TileSetDev& ts, int per_tile) {
  const long long n_act = ts.counts[MIE_CNT_ACTIVE];
  return n_act * per_tile >= 4LL << 20 && 8 * n_act < 7LL * ts.n * ts.tiles_y * ts.tiles_x;
}

__device__ __forceinline__ float mie_act(int kind, float slope, float v) {
  switch (kind) {
    case MIE_ACT_RELU: return v > 0.f ? v : 0.f;
    // __fmul_rn: keep the product from being contracted into the caller's
    // subtraction, so act(r1) - act(r0) rounds like two separate IEEE ops
    case MIE_ACT_LEAKY_RELU: return v > 0.f ? v : __fmul_rn(v, slope);
    case MIE_ACT_SIGMOID: return 1.f / (1.f + expf(-v));
    case MIE_ACT_TANH: return tanhf(v);
    default: return v;
  }
}

template <int N>
__device__ __forceinline__ void mie_act_select(int kind, float slope, float (&v)[N]) {      // none, ReLU, leaky ReLU
  const bool none = kind == MIE_ACT_NONE, leaky = kind == MIE_ACT_LEAKY_RELU;
#pragma unroll
  for (int i = 0; i < N; ++i) {
    const float low = none ? v[i] : leaky ? __fmul_rn(v[i], slope) : 0.f;
    v[i] = v[i] > 0.f ? v[i] : low;
  }
}

// mie_act of N values, for a kind that is not known at compile time.  Inlined once per value, the two transcendental
// kinds made 55 of the 70 KB of a kernel with 64 values a thread, and a workgroup that took neither still had to fetch the
// lines it jumped between; the instruction cache holds 64 KB for two CUs, and starts cold.  So the other kinds are selects,
// and those two are one loop over the values, which move up a place each time round (19 KB).  Measured over whole passes:
// fp32 1x64x96 201 -> 196 us, 1x264x352 461 -> 449; bf16 2x200x280 320 -> 314, 8x480x640 2740 -> 2590.
template <int N>
__device__ __forceinline__ void mie_act_n(int kind, float slope, float (&v)[N]) {
  if (__builtin_expect(kind <= MIE_ACT_LEAKY_RELU, 1)) {
    mie_act_select(kind, slope, v);
    return;
  }
#pragma unroll 1
  for (int k = 0; k < N; ++k) {
    const float y = kind == MIE_ACT_SIGMOID ? 1.f / (1.f + expf(-v[0])) : tanhf(v[0]);
#pragma unroll
    for (int i = 0; i + 1 < N; ++i) v[i] = v[i + 1];
    v[N - 1] = y;
  }
}
