// Pixel masks and ordered active-tile compaction (gfx950).
//
// mie_build_mask_tiles is two launches on the caller's stream: every wave of
// the first derives the 64 output-mask bits of one 8x8 tile from the input
// mask footprint and records whether the tile holds any active pixel (wave
// ballot); the second turns the per-tile flags into the ascending tile lists
// with a two-level ballot + popcount prefix scan (one block per 4096 tiles,
// each counting the flags below its chunk itself), so the list order is
// deterministic and nothing is communicated between workgroups inside a
// kernel (device-wide fences cost tens of microseconds on this chip).
#include "mie_common.h"

#include <string.h>

// ---- error string -----------------------------------------------------------
static thread_local char g_err[512] = "";

void mie_set_error(const char* fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(g_err, sizeof(g_err), fmt, ap);
  va_end(ap);
}
void mie_clear_error() { g_err[0] = 0; }

extern "C" const char* mie_last_error_string(void) { return g_err; }
extern "C" int mie_version(void) { return 100; }

extern "C" int mie_tile_capacity(int n, int h, int w) {
  if (n <= 0 || h <= 0 || w <= 0) return 0;
  long long cap = (long long)n * mie_div_up(h, MIE_TILE) * mie_div_up(w, MIE_TILE);
  if (cap > 0x3fffffff) return 0;
  return (int)cap;
}

int mie_check_tileset(const mie_tileset* ts, const char* who) {
  MIE_REQUIRE(ts != nullptr, MIE_ERR_INVALID_ARG, "%s: tile set is NULL", who);
  MIE_REQUIRE(ts->n > 0 && ts->h > 0 && ts->w > 0, MIE_ERR_INVALID_ARG,
              "%s: tile set geometry (%d,%d,%d) must be positive", who, ts->n, ts->h, ts->w);
  MIE_REQUIRE(mie_tile_capacity(ts->n, ts->h, ts->w) > 0, MIE_ERR_CAPACITY,
              "%s: tile set geometry (%d,%d,%d) too large", who, ts->n, ts->h, ts->w);
  MIE_REQUIRE((long long)ts->n * ts->h * ts->w < 0x7fffffffLL, MIE_ERR_CAPACITY,
              "%s: more than 2^31 pixels", who);
  MIE_REQUIRE(ts->pixmask && ts->tiles && ts->stale && ts->counts && ts->flags,
              MIE_ERR_INVALID_ARG, "%s: tile set has a NULL buffer", who);
  MIE_REQUIRE(mie_aligned(ts->tiles, 4) && mie_aligned(ts->stale, 4) &&
                  mie_aligned(ts->counts, 4) && mie_aligned(ts->flags, 16),
              MIE_ERR_INVALID_ARG, "%s: tile set buffers must be 4-byte aligned (flags: 16-byte)", who);
  return MIE_OK;
}

// ---- mask from delta ----------------------------------------------------------
// One thread per pixel walks its channel vector; C is small (<= 1024) and the
// vector is contiguous, float4 when the row is 16-byte aligned.
template <typename T>
__global__ __launch_bounds__(256) void k_mask_from_delta(
    const T* __restrict__ delta, long long npix, int c, float thr,
    uint8_t* __restrict__ pixmask) {
  const long long p = (long long)blockIdx.x * 256 + threadIdx.x;
  if (p >= npix) return;
  const T* row = delta + p * c;
  int any = 0;
  if constexpr (sizeof(T) == 4) {
    if ((c & 3) == 0) {
      const float4* r4 = reinterpret_cast<const float4*>(row);
      for (int i = 0; i < (c >> 2); ++i) {
        const float4 v = r4[i];
        any |= (fabsf(v.x) > thr) | (fabsf(v.y) > thr) | (fabsf(v.z) > thr) | (fabsf(v.w) > thr);
      }
    } else {
      for (int i = 0; i < c; ++i) any |= (fabsf(mie_ld(row, i)) > thr);
    }
  } else {
    for (int i = 0; i < c; ++i) any |= (fabsf(mie_ld(row, i)) > thr);
  }
  pixmask[p] = (uint8_t)any;
}

// Few channels that are no multiple of 4 (a network's input: 5 event bins): a pixel's row is 10 or 20 bytes, and one
// thread per pixel reads it in 2- or 4-byte pieces at a stride of that many bytes.  Here a wave takes the 64 * c elements
// of its 64 pixels as ONE contiguous span in 16-byte loads (the span starts at a multiple of 64 * c * sizeof(T) bytes,
// so every load is aligned), tests its elements and marks their pixels -- element e of the span belongs to pixel e / c
// -- in LDS; lane p then writes the byte of pixel p.  8x480x640x5 bf16: 35 -> 10 us on its own.
constexpr int MFD_SMALL_C = 16;      // channels up to which this form is taken
template <typename T>
__global__ __launch_bounds__(256) void k_mask_from_delta_span(
    const T* __restrict__ delta, long long npix, int c, float thr, uint8_t* __restrict__ pixmask) {
  constexpr int EPL = 16 / (int)sizeof(T);      // elements per 16-byte load
  __shared__ unsigned s_any[4][64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const long long p0 = ((long long)blockIdx.x * 4 + wave) * 64;      // first pixel of this wave
  s_any[wave][lane] = 0u;
  if (p0 < npix) {      // uniform over the wave
    const long long total = npix * c;                 // elements of the whole delta
    const long long e0 = p0 * c;                      // first element of the span
    const int span = 64 * c;                          // elements of a full span
    const unsigned inv_c = (65536u + (unsigned)c - 1u) / (unsigned)c;      // e / c for e < 64 * 16, c <= 16
    for (int ch = lane; ch * EPL < span; ch += 64) {
      const long long e = e0 + (long long)ch * EPL;
      if (e >= total) break;
      float f[EPL];
      if (e + EPL <= total) {
        const float4 raw = *reinterpret_cast<const float4*>(delta + e);
        if constexpr (sizeof(T) == 4) {
          f[0] = raw.x; f[1] = raw.y; f[2] = raw.z; f[3] = raw.w;
        } else {
          const unsigned w4[4] = {__float_as_uint(raw.x), __float_as_uint(raw.y), __float_as_uint(raw.z), __float_as_uint(raw.w)};
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            f[2 * j] = __uint_as_float(w4[j] << 16);
            f[2 * j + 1] = __uint_as_float(w4[j] & 0xffff0000u);
          }
        }
      } else {      // the last load of the delta would run past its end
#pragma unroll
        for (int j = 0; j < EPL; ++j) f[j] = (e + j < total) ? mie_ld(delta, e + j) : 0.f;
      }
#pragma unroll
      for (int j = 0; j < EPL; ++j) {
        if (fabsf(f[j]) > thr) {
          const unsigned le = (unsigned)(ch * EPL + j);      // element of the span
          s_any[wave][(le * inv_c) >> 16] = 1u;
        }
      }
    }
  }
  __syncthreads();
  if (p0 + lane < npix) pixmask[p0 + lane] = (uint8_t)s_any[wave][lane];
}

extern "C" int mie_mask_from_delta(const void* delta, int n, int h, int w, int c,
                                   float threshold, uint8_t* pixmask, int dtype, void* stream) {
  mie_clear_error();
  MIE_REQUIRE(delta && pixmask, MIE_ERR_INVALID_ARG, "mie_mask_from_delta: NULL pointer");
  MIE_REQUIRE(dtype == MIE_DTYPE_F32 || dtype == MIE_DTYPE_BF16, MIE_ERR_UNSUPPORTED,
              "mie_mask_from_delta: unknown delta dtype %d", dtype);
  MIE_REQUIRE(n > 0 && h > 0 && w > 0 && c > 0, MIE_ERR_INVALID_ARG,
              "mie_mask_from_delta: sizes must be positive (n=%d h=%d w=%d c=%d)", n, h, w, c);
  MIE_REQUIRE(threshold >= 0.f, MIE_ERR_INVALID_ARG, "mie_mask_from_delta: threshold < 0");
  MIE_REQUIRE(mie_aligned(delta, 16), MIE_ERR_INVALID_ARG,
              "mie_mask_from_delta: delta must be 16-byte aligned");
  const long long npix = (long long)n * h * w;
  MIE_REQUIRE(npix < 0x7fffffffLL, MIE_ERR_CAPACITY, "mie_mask_from_delta: too many pixels");
  const unsigned blocks = (unsigned)((npix + 255) / 256);
  const bool span = (c & 3) != 0 && c <= MFD_SMALL_C;
  if (dtype == MIE_DTYPE_BF16) {
    if (span)
      hipLaunchKernelGGL(k_mask_from_delta_span<mie_bf16>, dim3(blocks), dim3(256), 0, (hipStream_t)stream,
                         (const mie_bf16*)delta, npix, c, threshold, pixmask);
    else
      hipLaunchKernelGGL(k_mask_from_delta<mie_bf16>, dim3(blocks), dim3(256), 0, (hipStream_t)stream,
                         (const mie_bf16*)delta, npix, c, threshold, pixmask);
  } else {
    if (span)
      hipLaunchKernelGGL(k_mask_from_delta_span<float>, dim3(blocks), dim3(256), 0, (hipStream_t)stream,
                         (const float*)delta, npix, c, threshold, pixmask);
    else
      hipLaunchKernelGGL(k_mask_from_delta<float>, dim3(blocks), dim3(256), 0, (hipStream_t)stream,
                         (const float*)delta, npix, c, threshold, pixmask);
  }
  return mie_check_launch("mie_mask_from_delta");
}

// ---- footprint + tile flags + ordered compaction ----------------------------
struct BuildArgs {
  const uint8_t* in;
  const uint8_t* in2;
  int n, h_in, w_in;
  int foot, k, s, p;
  uint8_t* out;
  int h_out, w_out, tiles_y, tiles_x, cap;
  int32_t* tiles;
  int32_t* stale;
  int32_t* counts;
  uint32_t* flags;
};

__device__ __forceinline__ int mask_at(const BuildArgs& a, int n, int iy, int ix) {
  if (iy < 0 || iy >= a.h_in || ix < 0 || ix >= a.w_in) return 0;
  const long long o = ((long long)n * a.h_in + iy) * a.w_in + ix;
  int v = a.in[o];
  if (a.in2) v |= a.in2[o];
  return v != 0;
}

// Source index pair of bilinear x2 (align_corners = False) with non-zero weight.
__device__ __forceinline__ void up2x_src(int o, int in_size, int& i0, int& i1) {
  const int j = o >> 1;
  if (o & 1) {
    i0 = j;
    i1 = (j + 1 < in_size) ? j + 1 : j;
  } else {
    i0 = (j > 0) ? j - 1 : 0;
    i1 = j;
  }
}

// k x k window of a conv with the window size known at compile time: every load is issued from a clamped
// address and masked afterwards, so the K * K loads of a lane are independent and go out back to back.
template <int K>
__device__ __forceinline__ int conv_window_bit(const BuildArgs& a, int n, int iy0, int ix0) {
  const uint8_t* base = a.in + (long long)n * a.h_in * a.w_in;
  const uint8_t* base2 = a.in2 ? a.in2 + (long long)n * a.h_in * a.w_in : nullptr;
  int bit = 0;
#pragma unroll
  for (int ky = 0; ky < K; ++ky) {
    const int iy = iy0 + ky;
    const bool oky = iy >= 0 && iy < a.h_in;
    const int row = (oky ? iy : 0) * a.w_in;
#pragma unroll
    for (int kx = 0; kx < K; ++kx) {
      const int ix = ix0 + kx;
      const bool ok = oky && ix >= 0 && ix < a.w_in;
      const int o = row + (ok ? ix : 0);
      int v = base[o];
      if (base2) v |= base2[o];
      bit |= ok ? v : 0;
    }
  }
  return bit != 0;
}

__device__ int footprint_bit(const BuildArgs& a, int n, int oy, int ox) {
  if (a.in == nullptr) return 1;
  int bit = 0;
  if (a.foot == MIE_FOOT_CONV) {
    const int iy0 = oy * a.s - a.p, ix0 = ox * a.s - a.p;
    if (a.k == 5) return conv_window_bit<5>(a, n, iy0, ix0);
    if (a.k == 3) return conv_window_bit<3>(a, n, iy0, ix0);
    if (a.k == 1) return conv_window_bit<1>(a, n, iy0, ix0);
    for (int ky = 0; ky < a.k; ++ky)
      for (int kx = 0; kx < a.k; ++kx) bit |= mask_at(a, n, iy0 + ky, ix0 + kx);
  } else if (a.foot == MIE_FOOT_UP2X) {
    int r0, r1, c0, c1;
    up2x_src(oy, a.h_in, r0, r1);
    up2x_src(ox, a.w_in, c0, c1);
    bit = mask_at(a, n, r0, c0) | mask_at(a, n, r0, c1) | mask_at(a, n, r1, c0) |
          mask_at(a, n, r1, c1);
  } else {  // MIE_FOOT_TCONV
    for (int ky = 0; ky < a.k; ++ky) {
      const int ty = oy + a.p - ky;
      if (ty < 0 || (ty % a.s) != 0) continue;
      for (int kx = 0; kx < a.k; ++kx) {
        const int tx = ox + a.p - kx;
        if (tx < 0 || (tx % a.s) != 0) continue;
        bit |= mask_at(a, n, ty / a.s, tx / a.s);
      }
    }
  }
  return bit;
}

// Kernel 1: one wave per output tile.  Lane = pixel of the 8x8 tile: derives its mask bit
// from the input footprint, writes the output pixel mask, and a wave ballot tells whether
// the tile holds any active pixel.
__device__ __forceinline__ bool tile_footprint(const BuildArgs& a, int tile, int lane) {
  const int tx = tile % a.tiles_x;
  const int t2 = tile / a.tiles_x;
  const int ty = t2 % a.tiles_y;
  const int n = t2 / a.tiles_y;
  const int oy = ty * MIE_TILE + (lane >> 3), ox = tx * MIE_TILE + (lane & 7);
  int bit = 0;
  if (oy < a.h_out && ox < a.w_out) {
    bit = footprint_bit(a, n, oy, ox);
    a.out[((long long)n * a.h_out + oy) * a.w_out + ox] = (uint8_t)bit;
  }
  return __ballot(bit != 0) != 0ull;
}

// flags[tile]: bit 0 = the tile holds an active pixel after this build, bit 1 = it did after the
// previous build of this tile set (what makes a tile stale).  A lane reads and writes its own word only.
__device__ __forceinline__ uint32_t next_flag(uint32_t old, bool any) { return ((old & 1u) << 1) | (any ? 1u : 0u); }

__global__ __launch_bounds__(256) void k_mask_footprint(BuildArgs a) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int tile = blockIdx.x * 4 + wave;
  if (tile >= a.cap) return;
  const uint32_t old = a.flags[tile];          // issued ahead of the footprint's mask loads
  const bool any = tile_footprint(a, tile, lane);
  if (lane == 0) a.flags[tile] = next_flag(old, any);
}

// Ordered compaction of the tile flags into the active list (bit 0 set) and the stale list (bit 1
// set, bit 0 clear), both ascending, by a grid of COMPACT_THREADS-thread blocks without atomics or
// fences: block b owns the COMPACT_CHUNK flags [b * CHUNK, (b + 1) * CHUNK).  It first counts the two
// kinds over every flag below its chunk (16-byte loads; at most a few dozen per thread even for tens of
// thousands of tiles) -- that is its base in either list -- and then ranks its own flags: per wave a
// ballot gives 64 keep-bits, popcount below the lane the rank inside the wave, and the wave totals
// meet in LDS.  The last block also writes the two totals.
constexpr int COMPACT_THREADS = 1024;
constexpr int COMPACT_WAVES = COMPACT_THREADS / 64;
constexpr int COMPACT_ITEMS = 4;      // element j * COMPACT_THREADS + tid of the chunk, j < COMPACT_ITEMS
constexpr int COMPACT_CHUNK = COMPACT_THREADS * COMPACT_ITEMS;

__device__ __forceinline__ int wave_sum(int v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
  return v;
}

// flag(t) returns the flag word of tile t (from memory or, for the one-block build, from LDS).
template <typename FlagFn>
__device__ void compact_lists(const BuildArgs& a, FlagFn flag, int chunk, int base_act, int base_st, bool last,
                              int* s_tot) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  bool ka[COMPACT_ITEMS], ks[COMPACT_ITEMS];
  int ra[COMPACT_ITEMS], rs[COMPACT_ITEMS];
#pragma unroll
  for (int j = 0; j < COMPACT_ITEMS; ++j) {
    const int t = chunk * COMPACT_CHUNK + j * COMPACT_THREADS + threadIdx.x;
    const uint32_t f = (t < a.cap) ? flag(t) : 0u;
    ka[j] = (f & 1u) != 0u;
    ks[j] = (f & 3u) == 2u;
    const unsigned long long ba = __ballot(ka[j]), bs = __ballot(ks[j]);
    const unsigned long long below = (1ull << lane) - 1ull;
    ra[j] = __popcll(ba & below);
    rs[j] = __popcll(bs & below);
    if (lane == 0) {
      s_tot[j * COMPACT_WAVES + wave] = __popcll(ba);
      s_tot[COMPACT_ITEMS * COMPACT_WAVES + j * COMPACT_WAVES + wave] = __popcll(bs);
    }
  }
  __syncthreads();
  // exclusive prefix over the (j, wave) totals in element order: j major, wave minor
  int run_a = base_act, run_s = base_st;
#pragma unroll
  for (int j = 0; j < COMPACT_ITEMS; ++j) {
    int off_a = run_a, off_s = run_s;
#pragma unroll
    for (int wv = 0; wv < COMPACT_WAVES; ++wv) {
      const int ta = s_tot[j * COMPACT_WAVES + wv];
      const int tst = s_tot[COMPACT_ITEMS * COMPACT_WAVES + j * COMPACT_WAVES + wv];
      if (wv < wave) off_a += ta, off_s += tst;
      run_a += ta;
      run_s += tst;
    }
    const int t = chunk * COMPACT_CHUNK + j * COMPACT_THREADS + threadIdx.x;
    if (ka[j]) a.tiles[off_a + ra[j]] = t;
    if (ks[j]) a.stale[off_s + rs[j]] = t;
  }
  if (last && threadIdx.x == 0) {
    a.counts[MIE_CNT_ACTIVE] = run_a;
    a.counts[MIE_CNT_STALE] = run_s;
  }
}

// One chunk of the compaction of a tile set: block `chunk` of `nchunks`.
__device__ void compact_chunk(const BuildArgs& a, int chunk, int nchunks, int* s_tot, int* s_base) {
  const uint32_t* flags = a.flags;
  // base = number of active / stale tiles below this chunk (its start is a multiple of 4096 flags)
  int na = 0, ns = 0;
  const uint4* f4 = reinterpret_cast<const uint4*>(flags);
  const int n4 = chunk * (COMPACT_CHUNK / 4);
  for (int i = threadIdx.x; i < n4; i += COMPACT_THREADS) {
    const uint4 v = f4[i];
    na += (int)(v.x & 1u) + (int)(v.y & 1u) + (int)(v.z & 1u) + (int)(v.w & 1u);
    ns += (int)((v.x & 3u) == 2u) + (int)((v.y & 3u) == 2u) + (int)((v.z & 3u) == 2u) + (int)((v.w & 3u) == 2u);
  }
  int base_act = 0, base_st = 0;
  if (chunk > 0) {      // uniform over the block
    na = wave_sum(na);
    ns = wave_sum(ns);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    if (lane == 0) s_base[wave] = na, s_base[COMPACT_WAVES + wave] = ns;
    __syncthreads();
#pragma unroll
    for (int wv = 0; wv < COMPACT_WAVES; ++wv) base_act += s_base[wv], base_st += s_base[COMPACT_WAVES + wv];
  }
  compact_lists(a, [&](int t) { return flags[t]; }, chunk, base_act, base_st, chunk == nchunks - 1, s_tot);
}

__global__ __launch_bounds__(COMPACT_THREADS) void k_compact_tiles(BuildArgs a) {
  __shared__ int s_tot[2 * COMPACT_WAVES * COMPACT_ITEMS];
  __shared__ int s_base[2 * COMPACT_WAVES];
  compact_chunk(a, blockIdx.x, (int)gridDim.x, s_tot, s_base);
}

// Planes of at most SMALL_CAP tiles (the 33x44 plane of a 264x352 frame: 30 tiles): footprint
// and compaction in ONE block, tile flags handed over through LDS -- one launch instead of two.
constexpr int SMALL_CAP = 32;

__global__ __launch_bounds__(COMPACT_THREADS) void k_build_small(BuildArgs a) {
  __shared__ int s_tot[2 * COMPACT_WAVES * COMPACT_ITEMS];
  __shared__ unsigned s_flag[SMALL_CAP];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  for (int tile = wave; tile < a.cap; tile += COMPACT_WAVES) {
    const uint32_t old = a.flags[tile];
    const bool any = tile_footprint(a, tile, lane);
    if (lane == 0) {
      const uint32_t f = next_flag(old, any);
      s_flag[tile] = f;
      a.flags[tile] = f;
    }
  }
  __syncthreads();
  compact_lists(a, [&](int t) { return s_flag[t]; }, 0, 0, 0, true, s_tot);
}

// ---- one launch for planes of up to TICKET_CAP tiles ----------------------------------------------
// The footprint kernel's workgroups take a ticket from counts[MIE_CNT_TICKET] when their flags are written; the one
// that draws the last ticket puts the counter back to zero and ranks the two lists from the flags of all of them.
// Nobody waits for anybody: every other workgroup has left by then.  The lists are what k_compact_tiles writes.
// Flags are stored and, by the last workgroup, loaded as device-scope atomics, which go through to the level the
// XCDs share; a workgroup waits for its flag stores to complete before it draws its ticket.  (A device-scope
// release / acquire fence pair would order ordinary stores as well, but it writes back and invalidates the whole L2
// of the XCD -- with a step's deltas in it that cost 8 us per build, more than the launch it saves.)  The pixel masks
// are ordinary stores: nothing in the kernel reads another workgroup's.
constexpr int TICKET_CAP = 4096;
constexpr int TICKET_THREADS = 256;

__device__ __forceinline__ void store_flag(uint32_t* flags, int tile, uint32_t f) {
  __hip_atomic_store(flags + tile, f, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// true in exactly one workgroup of the grid: the one whose ticket is the last
__device__ __forceinline__ bool last_workgroup(int32_t* counts, int* s_last) {
  // This thread's flag stores have completed.  (A release fence of the workgroup does not say so: the caches a workgroup
  // shares need no such wait, and the compiler leaves it out.)
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  if (threadIdx.x == 0) {
    const int t = __hip_atomic_fetch_add(&counts[MIE_CNT_TICKET], 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const bool last = t == (int)gridDim.x - 1;
    if (last) __hip_atomic_store(&counts[MIE_CNT_TICKET], 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);   // all drawn
    *s_last = last ? 1 : 0;
  }
  __syncthreads();
  return *s_last != 0;
}

// the two lists of a set of at most TICKET_CAP tiles, by the first TICKET_THREADS threads of one workgroup (all of its
// threads call): flag j * TICKET_THREADS + tid in round j, ranked by ballots -- a wave's round is 64 tiles in a row, and the
// rounds' counts, active and stale in the halves of a word, meet in LDS for one scan.  (With sixteen consecutive flags
// per thread and two scans over the threads by shuffles, the mask and lists of 374 tiles took 1.0 us more.)
template <int ROUNDS>
__device__ __forceinline__ void compact_rounds(const BuildArgs& a, int* s_w) {
  constexpr int WAVES = TICKET_THREADS / 64, WORDS = ROUNDS * WAVES;
  static_assert(WORDS <= 64, "a wave scans the words");
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  uint32_t f[ROUNDS];
  if (wave < WAVES) {
#pragma unroll
    for (int j = 0; j < ROUNDS; ++j) {      // every load goes out, from a clamped address
      const int t = j * TICKET_THREADS + tid;
      f[j] = __hip_atomic_load(a.flags + (t < a.cap ? t : a.cap - 1), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
#pragma unroll
    for (int j = 0; j < ROUNDS; ++j) {
      if (j * TICKET_THREADS + tid >= a.cap) f[j] = 0u;
      const int na = __popcll(__ballot(f[j] & 1u)), ns = __popcll(__ballot((f[j] & 3u) == 2u));
      if (lane == 0) s_w[j * WAVES + wave] = na | ns << 16;
    }
  }
  __syncthreads();
  if (wave >= WAVES) return;      // a wider workgroup: its other waves only meet the barrier
  int sum = lane < WORDS ? s_w[lane] : 0;
  const int own = sum;
#pragma unroll
  for (int o = 1; o < WORDS; o <<= 1) {
    const int u = __shfl_up(sum, o);
    if (lane >= o) sum += u;
  }
  const int before = sum - own, all = __builtin_amdgcn_readlane(sum, WORDS - 1);
#pragma unroll
  for (int j = 0; j < ROUNDS; ++j) {
    const unsigned long long ba = __ballot(f[j] & 1u), bs = __ballot((f[j] & 3u) == 2u);
    const int at = __builtin_amdgcn_readlane(before, j * WAVES + __builtin_amdgcn_readfirstlane(wave));
    const unsigned long long below = (1ull << lane) - 1ull;
    const int t = j * TICKET_THREADS + tid;
    if (f[j] & 1u) a.tiles[(at & 0xffff) + __popcll(ba & below)] = t;
    if ((f[j] & 3u) == 2u) a.stale[(at >> 16) + __popcll(bs & below)] = t;
  }
  if (tid == 0) {
    a.counts[MIE_CNT_ACTIVE] = all & 0xffff;
    a.counts[MIE_CNT_STALE] = all >> 16;
  }
}
__device__ __forceinline__ void compact_by_one(const BuildArgs& a, int* s_w) {
  if (a.cap <= 2 * TICKET_THREADS) compact_rounds<2>(a, s_w);
  else compact_rounds<TICKET_CAP / TICKET_THREADS>(a, s_w);
}

// k_mask_footprint + k_compact_tiles for sets of up to TICKET_CAP tiles
__global__ __launch_bounds__(TICKET_THREADS) void k_mask_footprint_lists(BuildArgs a) {
  __shared__ int s_w[64];
  __shared__ int s_last;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int tile = blockIdx.x * 4 + wave;
  if (tile < a.cap) {
    const uint32_t old = a.flags[tile];
    const bool any = tile_footprint(a, tile, lane);
    if (lane == 0) store_flag(a.flags, tile, next_flag(old, any));
  }
  if (last_workgroup(a.counts, &s_last)) compact_by_one(a, s_w);
}

// ---- threshold mask + footprint (+ lists) in one launch -------------------------------------------
// What mie_mask_from_delta followed by mie_build_mask_tiles (conv footprint) leave, for the thresholded masks of
// the lossy networks: one workgroup per output tile tests the input pixels of its tile's windows against the
// threshold itself, straight from the delta, keeps the bits in LDS, writes the bytes of the input pixels it owns (the
// 8s x 8s block under its tile; the last row / column of tiles owns through the plane's edge) and forms the footprint
// from LDS.  Pixels in the halo of a window are tested by up to four workgroups; a delta plane of these networks is
// at most a few MB and the launch is bound by latency -- so the test is a flat loop over (pixel, 4-channel group)
// pairs with eight loads in flight per thread and no exchange between lanes (a hit sets the pixel's byte in LDS).
struct ThrArgs {
  BuildArgs b;          // b.in is unused (the mask comes from delta); b.in2 as in mie_build_mask_tiles
  const void* delta;
  uint8_t* thr_mask;    // [n, h_in, w_in]: the thresholded mask, as mie_mask_from_delta writes it
  int c;
  int vec_shift;        // log2(c / 4) when c / 4 is a power of two, else -1
  float thr;
  int lists;            // 1: the last workgroup ranks the lists
};
constexpr int THR_EDGE = 24;      // largest region edge: 7 * s + k (+ the rows no window reaches)
constexpr int THR_UNROLL = 8;
constexpr int TICKET_MAX_WGS = 128;      // more workgroups than this queue up at the ticket counter: two launches then

template <typename T>
__global__ __launch_bounds__(1024) void k_build_thresholded(ThrArgs a) {
  __shared__ uint8_t s_in[THR_EDGE * THR_EDGE];
  __shared__ int s_w[64];
  __shared__ int s_last;
  const BuildArgs& b = a.b;
  const int tid = threadIdx.x, nthr = blockDim.x, lane = tid & 63;
  const int tile = blockIdx.x;                    // the grid is one workgroup per tile
  const int tx = tile % b.tiles_x, t2 = tile / b.tiles_x, ty = t2 % b.tiles_y, n = t2 / b.tiles_y;
  uint32_t old = 0;
  if (tid == 0) old = b.flags[tile];
  const int r0 = ty * MIE_TILE * b.s - b.p, c0 = tx * MIE_TILE * b.s - b.p;
  const int own_r0 = ty * MIE_TILE * b.s, own_c0 = tx * MIE_TILE * b.s;
  const int own_r1 = (ty == b.tiles_y - 1) ? b.h_in : own_r0 + MIE_TILE * b.s;
  const int own_c1 = (tx == b.tiles_x - 1) ? b.w_in : own_c0 + MIE_TILE * b.s;
  const int win = 7 * b.s + b.k;
  const int rows = max(r0 + win, own_r1) - r0, cols = max(c0 + win, own_c1) - c0;
  const int npx = rows * cols;
  const unsigned col_magic = (65536u + (unsigned)cols - 1u) / (unsigned)cols;      // p / cols for p < 576, cols <= 24
  const T* plane = static_cast<const T*>(a.delta) + (long long)n * b.h_in * b.w_in * a.c;
  for (int i = tid; i < npx; i += nthr) s_in[i] = 0;
  __syncthreads();
  if ((a.c & 3) == 0) {
    const int nvec = a.c >> 2, total = npx * nvec;
    for (int base = tid; base < total; base += THR_UNROLL * nthr) {
      float4 v[THR_UNROLL];
      int pp[THR_UNROLL];
#pragma unroll
      for (int u = 0; u < THR_UNROLL; ++u) {
        const int idx = base + u * nthr;
        const int p = a.vec_shift >= 0 ? (idx >> a.vec_shift) : idx / nvec;
        const int q = idx - p * nvec;
        const int ry = (int)(((unsigned)p * col_magic) >> 16), rx = p - ry * cols;
        const int iy = r0 + ry, ix = c0 + rx;
        const bool inside = idx < total && iy >= 0 && iy < b.h_in && ix >= 0 && ix < b.w_in;
        pp[u] = inside ? p : -1;
        // every load goes out, from a clamped address: eight independent loads, no branch between them
        v[u] = mie_ld4(plane + (inside ? ((long long)iy * b.w_in + ix) * a.c + 4 * q : 0ll), 0);
      }
#pragma unroll
      for (int u = 0; u < THR_UNROLL; ++u) {
        const bool hit = (fabsf(v[u].x) > a.thr) | (fabsf(v[u].y) > a.thr) | (fabsf(v[u].z) > a.thr) | (fabsf(v[u].w) > a.thr);
        if (pp[u] >= 0 && hit) s_in[pp[u]] = 1;
      }
    }
  } else {      // channel counts that are no multiple of 4 (a network's input): one thread per pixel
    for (int p = tid; p < npx; p += nthr) {
      const int ry = (int)(((unsigned)p * col_magic) >> 16), rx = p - ry * cols;
      const int iy = r0 + ry, ix = c0 + rx;
      if (iy < 0 || iy >= b.h_in || ix < 0 || ix >= b.w_in) continue;
      const T* row = plane + ((long long)iy * b.w_in + ix) * a.c;
      int any = 0;
      for (int i = 0; i < a.c; ++i) any |= (fabsf(mie_ld(row, i)) > a.thr);
      if (any) s_in[p] = 1;
    }
  }
  __syncthreads();
  for (int p = tid; p < npx; p += nthr) {
    const int ry = (int)(((unsigned)p * col_magic) >> 16), rx = p - ry * cols;
    const int iy = r0 + ry, ix = c0 + rx;
    if (iy >= own_r0 && iy < min(own_r1, b.h_in) && ix >= own_c0 && ix < min(own_c1, b.w_in))
      a.thr_mask[((long long)n * b.h_in + iy) * b.w_in + ix] = s_in[p];
  }
  if (tid < 64) {
    const int py = lane >> 3, px = lane & 7;
    const int oy = ty * MIE_TILE + py, ox = tx * MIE_TILE + px;
    int bit = 0;
    if (oy < b.h_out && ox < b.w_out) {
      for (int ky = 0; ky < b.k; ++ky)
        for (int kx = 0; kx < b.k; ++kx) bit |= s_in[(py * b.s + ky) * cols + px * b.s + kx];
      if (b.in2) {
        const uint8_t* m2 = b.in2 + (long long)n * b.h_in * b.w_in;
        for (int ky = 0; ky < b.k; ++ky) {
          const int iy = oy * b.s - b.p + ky;
          if (iy < 0 || iy >= b.h_in) continue;
          for (int kx = 0; kx < b.k; ++kx) {
            const int ix = ox * b.s - b.p + kx;
            if (ix >= 0 && ix < b.w_in) bit |= m2[iy * b.w_in + ix];
          }
        }
      }
      bit = bit != 0;
      b.out[((long long)n * b.h_out + oy) * b.w_out + ox] = (uint8_t)bit;
    }
    const bool any = __ballot(bit != 0) != 0ull;
    if (lane == 0) {
      if (a.lists) store_flag(b.flags, tile, next_flag(old, any));
      else b.flags[tile] = next_flag(old, any);
    }
  }
  if (a.lists && last_workgroup(b.counts, &s_last)) compact_by_one(b, s_w);
}

extern "C" int mie_build_mask_tiles(const uint8_t* in_mask, const uint8_t* in_mask2,
                                    int h_in, int w_in, int foot, int k, int stride,
                                    int pad, const mie_tileset* out, void* stream) {
  mie_clear_error();
  int rc = mie_check_tileset(out, "mie_build_mask_tiles");
  if (rc != MIE_OK) return rc;
  MIE_REQUIRE(h_in > 0 && w_in > 0, MIE_ERR_INVALID_ARG,
              "mie_build_mask_tiles: input size (%d,%d) must be positive", h_in, w_in);
  MIE_REQUIRE(in_mask != nullptr || in_mask2 == nullptr, MIE_ERR_INVALID_ARG,
              "mie_build_mask_tiles: in_mask2 given without in_mask");
  MIE_REQUIRE((long long)out->n * h_in * w_in < 0x7fffffffLL, MIE_ERR_CAPACITY,
              "mie_build_mask_tiles: more than 2^31 input pixels");
  if (foot == MIE_FOOT_CONV) {
    MIE_REQUIRE(k >= 1 && k <= 15 && stride >= 1 && stride <= 4 && pad >= 0 && pad < 16,
                MIE_ERR_UNSUPPORTED, "mie_build_mask_tiles: conv footprint k=%d stride=%d pad=%d",
                k, stride, pad);
    const int ho = (h_in + 2 * pad - k) / stride + 1, wo = (w_in + 2 * pad - k) / stride + 1;
    MIE_REQUIRE(h_in + 2 * pad >= k && w_in + 2 * pad >= k && ho == out->h && wo == out->w,
                MIE_ERR_INVALID_ARG,
                "mie_build_mask_tiles: conv output of (%d,%d) k=%d s=%d p=%d is (%d,%d), tile set is (%d,%d)",
                h_in, w_in, k, stride, pad, ho, wo, out->h, out->w);
  } else if (foot == MIE_FOOT_UP2X) {
    MIE_REQUIRE(out->h == 2 * h_in && out->w == 2 * w_in, MIE_ERR_INVALID_ARG,
                "mie_build_mask_tiles: up2x of (%d,%d) is not (%d,%d)", h_in, w_in, out->h, out->w);
  } else if (foot == MIE_FOOT_TCONV) {
    MIE_REQUIRE(k >= 1 && k <= 15 && stride >= 1 && stride <= 4 && pad >= 0 && pad < 16,
                MIE_ERR_UNSUPPORTED, "mie_build_mask_tiles: tconv footprint k=%d stride=%d pad=%d",
                k, stride, pad);
    const int hmin = (h_in - 1) * stride - 2 * pad + k, wmin = (w_in - 1) * stride - 2 * pad + k;
    MIE_REQUIRE(out->h >= hmin && out->h < hmin + stride && out->w >= wmin && out->w < wmin + stride,
                MIE_ERR_INVALID_ARG,
                "mie_build_mask_tiles: tconv output (%d,%d) not in [(%d,%d), +stride)", out->h,
                out->w, hmin, wmin);
  } else {
    MIE_REQUIRE(false, MIE_ERR_UNSUPPORTED, "mie_build_mask_tiles: unknown footprint %d", foot);
  }
  // A lane reads the mask bytes of its footprint while other lanes write theirs: only the 1x1 stride-1
  // identity footprint (own pixel in, own pixel out) may be built in place.
  const bool identity = foot == MIE_FOOT_CONV && k == 1 && stride == 1 && pad == 0;
  MIE_REQUIRE(identity || ((const uint8_t*)out->pixmask != in_mask && (const uint8_t*)out->pixmask != in_mask2),
              MIE_ERR_INVALID_ARG,
              "mie_build_mask_tiles: out->pixmask aliases an input mask (allowed for the 1x1 stride-1 footprint only)");
  BuildArgs a;
  a.in = in_mask; a.in2 = in_mask2;
  a.n = out->n; a.h_in = h_in; a.w_in = w_in;
  a.foot = foot; a.k = k; a.s = stride; a.p = pad;
  a.out = out->pixmask; a.h_out = out->h; a.w_out = out->w;
  a.tiles_y = mie_div_up(out->h, MIE_TILE); a.tiles_x = mie_div_up(out->w, MIE_TILE);
  a.cap = mie_tile_capacity(out->n, out->h, out->w);
  a.tiles = out->tiles; a.stale = out->stale; a.counts = out->counts; a.flags = out->flags;
  if (a.cap <= SMALL_CAP) {
    hipLaunchKernelGGL(k_build_small, dim3(1), dim3(COMPACT_THREADS), 0, (hipStream_t)stream, a);
    return mie_check_launch("mie_build_mask_tiles");
  }
  const unsigned blocks = (unsigned)mie_div_up(a.cap, 4);
  static const int ticket_wgs = [] { const char* e = getenv("MIE_BUILD_TICKET"); return e ? atoi(e) : TICKET_MAX_WGS; }();   // tuning knob
  if ((int)blocks <= ticket_wgs && a.cap <= TICKET_CAP) {
    hipLaunchKernelGGL(k_mask_footprint_lists, dim3(blocks), dim3(TICKET_THREADS), 0, (hipStream_t)stream, a);
    return mie_check_launch("mie_build_mask_tiles");
  }
  hipLaunchKernelGGL(k_mask_footprint, dim3(blocks), dim3(256), 0, (hipStream_t)stream, a);
  rc = mie_check_launch("mie_build_mask_tiles");
  if (rc != MIE_OK) return rc;
  hipLaunchKernelGGL(k_compact_tiles, dim3((unsigned)mie_div_up(a.cap, COMPACT_CHUNK)), dim3(COMPACT_THREADS), 0,
                     (hipStream_t)stream, a);
  return mie_check_launch("mie_build_mask_tiles");
}

extern "C" int mie_build_mask_tiles_thresholded(const void* delta, int c, int dtype, float threshold, uint8_t* thr_mask,
                                                const uint8_t* in_mask2, int h_in, int w_in, int k, int stride, int pad,
                                                const mie_tileset* out, void* stream) {
  const char* who = "mie_build_mask_tiles_thresholded";
  mie_clear_error();
  int rc = mie_check_tileset(out, who);
  if (rc != MIE_OK) return rc;
  MIE_REQUIRE(delta && thr_mask, MIE_ERR_INVALID_ARG, "%s: NULL pointer", who);
  MIE_REQUIRE(dtype == MIE_DTYPE_F32 || dtype == MIE_DTYPE_BF16, MIE_ERR_UNSUPPORTED, "%s: unknown delta dtype %d", who, dtype);
  MIE_REQUIRE(h_in > 0 && w_in > 0 && c > 0, MIE_ERR_INVALID_ARG, "%s: sizes must be positive (h=%d w=%d c=%d)", who, h_in, w_in, c);
  MIE_REQUIRE(threshold >= 0.f, MIE_ERR_INVALID_ARG, "%s: threshold < 0", who);
  MIE_REQUIRE(mie_aligned(delta, 16), MIE_ERR_INVALID_ARG, "%s: delta must be 16-byte aligned", who);
  MIE_REQUIRE((long long)out->n * h_in * w_in < 0x7fffffffLL, MIE_ERR_CAPACITY, "%s: more than 2^31 input pixels", who);
  MIE_REQUIRE(k >= 1 && stride >= 1 && pad >= 0, MIE_ERR_UNSUPPORTED, "%s: conv footprint k=%d stride=%d pad=%d", who, k, stride, pad);
  // a workgroup owns the input block under its tile and must find it inside its tile's windows
  MIE_REQUIRE(stride + pad <= k && 7 * stride + k + (stride - 1 - pad > 0 ? stride - 1 - pad : 0) <= THR_EDGE,
              MIE_ERR_UNSUPPORTED, "%s: no one-launch form for k=%d stride=%d pad=%d (mie_mask_from_delta + mie_build_mask_tiles take it)",
              who, k, stride, pad);
  const int ho = (h_in + 2 * pad - k) / stride + 1, wo = (w_in + 2 * pad - k) / stride + 1;
  MIE_REQUIRE(h_in + 2 * pad >= k && w_in + 2 * pad >= k && ho == out->h && wo == out->w, MIE_ERR_INVALID_ARG,
              "%s: conv output of (%d,%d) k=%d s=%d p=%d is (%d,%d), tile set is (%d,%d)", who, h_in, w_in, k, stride, pad,
              ho, wo, out->h, out->w);
  MIE_REQUIRE(thr_mask != out->pixmask && in_mask2 != out->pixmask && in_mask2 != thr_mask, MIE_ERR_INVALID_ARG,
              "%s: thr_mask, in_mask2 and out->pixmask must be three buffers", who);
  ThrArgs a;
  memset(&a, 0, sizeof(a));
  BuildArgs& b = a.b;
  b.in = nullptr; b.in2 = in_mask2;
  b.n = out->n; b.h_in = h_in; b.w_in = w_in;
  b.foot = MIE_FOOT_CONV; b.k = k; b.s = stride; b.p = pad;
  b.out = out->pixmask; b.h_out = out->h; b.w_out = out->w;
  b.tiles_y = mie_div_up(out->h, MIE_TILE); b.tiles_x = mie_div_up(out->w, MIE_TILE);
  b.cap = mie_tile_capacity(out->n, out->h, out->w);
  b.tiles = out->tiles; b.stale = out->stale; b.counts = out->counts; b.flags = out->flags;
  a.delta = delta; a.thr_mask = thr_mask; a.c = c; a.thr = threshold;
  a.vec_shift = -1;
  if ((c & 3) == 0 && ((c >> 2) & ((c >> 2) - 1)) == 0)
    for (a.vec_shift = 0; (1 << a.vec_shift) < (c >> 2); ++a.vec_shift) {}
  static const int ticket_wgs = [] { const char* e = getenv("MIE_BUILD_TICKET"); return e ? atoi(e) : TICKET_MAX_WGS; }();   // tuning knob
  a.lists = b.cap <= ticket_wgs && b.cap <= TICKET_CAP ? 1 : 0;
  // deep planes of few tiles (fewer workgroups than CUs): more threads per tile, so that a thread's loads go out in one
  // round (thresholded 264x352 frame, cap 0 / 128 / 512 / 2048: 0.504 / 0.485 / 0.490 / 0.501 ms)
  static const int wide_cap = [] { const char* e = getenv("MIE_THR_WIDE_CAP"); return e ? atoi(e) : 128; }();      // tuning knob
  const int threads = (b.cap <= wide_cap && (long long)(7 * stride + k) * (7 * stride + k) * (c / 4) > THR_UNROLL * 256) ? 1024 : 256;
  if (dtype == MIE_DTYPE_BF16)
    hipLaunchKernelGGL(k_build_thresholded<mie_bf16>, dim3((unsigned)b.cap), dim3(threads), 0, (hipStream_t)stream, a);
  else
    hipLaunchKernelGGL(k_build_thresholded<float>, dim3((unsigned)b.cap), dim3(threads), 0, (hipStream_t)stream, a);
  rc = mie_check_launch(who);
  if (rc != MIE_OK || a.lists) return rc;
  hipLaunchKernelGGL(k_compact_tiles, dim3((unsigned)mie_div_up(b.cap, COMPACT_CHUNK)), dim3(COMPACT_THREADS), 0,
                     (hipStream_t)stream, b);
  return mie_check_launch(who);
}

// ---- every tile set of a network in one or two launches ------------------------------------------
// mie_build_mask_plan runs a sequence of mie_build_mask_tiles calls -- every structural mask of a network is a chain
// of footprints of the input pixel mask.  A workgroup keeps the pixel masks of one sample's chain as BITMAPS in LDS (a
// 264x352 plane is 11.6 KB): a footprint is then a handful of word operations per 32 pixels -- the window of a conv is
// the OR of the rows it covers, shifted left and right (stride 2: the even bits of that, compressed); bilinear x2 and
// the stride-2 transposed conv interleave two such ORs bit by bit -- instead of k*k byte loads per pixel, and no launch
// or memory round trip separates one mask of the chain from the next.  Several workgroups per sample each walk the whole
// chain on their own and share only what goes to memory.
//
// What bounds it is the chain: one step after the other, a barrier between them, next to no work in the small planes.
// A step costs the latency of the instructions of one wave (some 1100 clocks, hardly fewer for a plane of 16 words than
// for one of 700), so there are few of them and each does little:
//  * a same-size conv window over the result of another is one wider window over what that one read (both padded by half
//    their size: every pixel between two pixels of the plane is in the plane), so the host lets a step read its input's
//    input where the wider window has a form below: the four convs of a bottleneck are one level, and so are a conv and
//    the stride-2 conv behind it;
//  * steps that do not depend on each other share a level (a barrier interval), each on waves of its own;
//  * a wave finds its step's parameters in one register, a word per lane, asked for a level ahead; a wave without a
//    step goes straight to the barrier;
//  * rows outside the plane are read from words of zeros, by address, instead of being masked after the load;
//  * where all bitmaps fit the LDS together nothing is written between the levels: the pixel masks of all sets go to
//    memory at the end, 16 pixels a thread, a slice per workgroup.  Where they do not, a bitmap is dropped after its last
//    reader and waves of their own write the masks of a level beside the next one's bitmaps.
// With one sample (all bitmaps resident, sets of at most 4096 tiles) a workgroup OWNS sets: it alone reads and writes their
// flags, and ranks their lists itself at the end, so the plan is one launch.  With a batch the lists run over all samples:
// a workgroup writes the flags of its slice of every set and k_plan_compact ranks the lists behind it, one block per 4096
// tiles.  Slots of LDS are handed out on the host by lifetime in levels.
// Measured, both kernels together (before: one step a level, 28 words of parameters read by all 16 waves in every step, the
// masks written between the steps, two launches): E2Depth-incr 64x96 25.8 -> 17.0 us, 264x352 37.2 -> 24.5, EVFlowNet-incr
// 256x256 45.1 -> 23.7, 8x480x640 75.8 -> 58.6.  (Windows over up-samplings in one level: whole passes 1x64x96 146.6 -> 144.6 us, 1x128x128
// 220.3 -> 218.9, 1x264x352 470.5 -> 468.6.  Tried: the code of the later levels fetched during level 0 by waves that it leaves over: the first
// level 1.2 us shorter, level 0 2.5 longer.)
namespace {

constexpr int PLAN_THREADS = 1024;
constexpr int PLAN_WAVES = PLAN_THREADS / 64;
constexpr int PLAN_COMPUTE_WAVES = 12;                 // of a level's bitmaps where the others write the level before it
constexpr int PLAN_WRITE_WAVES = PLAN_WAVES - PLAN_COMPUTE_WAVES;
constexpr int PLAN_UP_WORDS = PLAN_THREADS;            // of a plane whose window over an up-sampling is read from below that
constexpr int PLAN_LEVEL_STEPS = 8;                    // steps of a level (not resident: at least one writing wave each)
constexpr int PLAN_MAX_SHARES = 64;                    // workgroups per sample
constexpr int PLAN_PIXELS_PER_SHARE = 8192;            // of the plan's largest plane
constexpr int PLAN_OWNED_TILES = 4096;                 // largest set a workgroup ranks by itself
constexpr int PLAN_KIND_LOAD = 0, PLAN_KIND_FOOT = 1;
constexpr unsigned PLAN_IN_NONE = 0xffffu;             // instead of an LDS word offset (at most 40960)
constexpr int PLAN_IDLE = 255;                         // task table: nothing to do for this wave in this level

// A step's words (lane l of a wave that works on it holds word l).
enum {
  PS_IN,            // LDS word offsets of the input bitmaps: in1 | in2 << 16
  PS_OUT_WIN,       // LDS word offset of the bitmap it makes | input width << 16
  PS_HIN, PS_HOUT,
  PS_WOUT_KEY,      // output width | PLAN_KEY_* << 16 | kind << 24 | size of its accesses to the mask in memory << 28 (2: 16 bytes, 1: 4, 0: 1)
  PS_GEOM,          // foot | k << 8 | stride << 16 | pad << 24
  PS_MWORDS,        // plan_magic of the words per row
  PS_MUNITS,        // plan_magic of the 16-pixel units per row
  PS_WAVES,         // computing waves: first | number << 8; writing waves: first << 16 | number << 24
  PS_UBASE,         // 16-pixel units of the sets before it
  PS_FL,            // byte offset of its tiles in the workgroup's flag area
  PS_OWN,           // sets owned: the next set of the same owner, or PLAN_IDLE; else tiles of the set per share
  PS_MTILES,        // plan_magic of the tiles per row
  PS_PIX, PS_PIX_HI,          // pixel mask in memory (LOAD: the mask to read)
  PS_FLAGS, PS_FLAGS_HI, PS_TILES, PS_TILES_HI, PS_STALE, PS_STALE_HI, PS_COUNTS, PS_COUNTS_HI,
  PS_WORDS
};

struct PlanArgs {
  int n_steps, n_levels, n_loads;         // steps are in level order; the first n_loads are the masks from memory of level 0
  int first_last;                         // the first step of the last level
  int resident;                           // all bitmaps stay: everything is written at the end
  int owned;                              // a workgroup owns sets and ranks them (resident only); 0: slices, lists by k_plan_compact
  int units, pad_;                        // 16-pixel units of all sets
  int zero_off, flag_off;                 // LDS: words of zeros; a byte per tile (owned: old state; not resident: new state)
  uint32_t st[MIE_PLAN_MAX_STEPS * PS_WORDS];
  uint8_t task[(MIE_PLAN_MAX_STEPS + 3) * PLAN_WAVES];     // [level][wave] -> step
  uint8_t head[PLAN_MAX_SHARES];          // the first set each share owns, or PLAN_IDLE
};
constexpr int PLAN_ZERO_WORDS = 8;

// (To be called where every lane of the wave is active: a load that feeds it may move down to it, and the lanes that a
// branch around both has switched off would not have loaded their word.)
__device__ __forceinline__ uint32_t plan_word(uint32_t pw, int i) { return (uint32_t)__builtin_amdgcn_readlane((int)pw, i); }
template <typename P>
__device__ __forceinline__ P* plan_ptr(uint32_t pw, int i) {
  const unsigned long long v = ((unsigned long long)plan_word(pw, i + 1) << 32) | plan_word(pw, i);
  return reinterpret_cast<P*>(v);
}
__device__ __forceinline__ int plan_kind(uint32_t pw) { return (int)((plan_word(pw, PS_WOUT_KEY) >> 24) & 15u); }

__device__ __forceinline__ uint32_t plan_dot4(uint32_t a, uint32_t b, uint32_t c) { return __builtin_amdgcn_udot4(a, b, c, false); }

// bit x of the result = bit (x + t) of the row whose words around the current one are prev, cur, next (|t| < 32):
// 32 bits out of the middle of two adjacent words (v_alignbit_b32), no branch on the sign of t
__device__ __forceinline__ uint32_t plan_shift(uint32_t prev, uint32_t cur, uint32_t next, int t) {
  const uint32_t hi = t >= 0 ? next : cur, lo = t >= 0 ? cur : prev;
  return __builtin_amdgcn_alignbit(hi, lo, (uint32_t)t & 31u);
}
// bits 0, 2, 4, ... of x packed into the low half
__device__ __forceinline__ uint32_t plan_even_bits(uint32_t x) {
  x &= 0x55555555u;
  x = (x | (x >> 1)) & 0x33333333u;
  x = (x | (x >> 2)) & 0x0f0f0f0fu;
  x = (x | (x >> 4)) & 0x00ff00ffu;
  x = (x | (x >> 8)) & 0x0000ffffu;
  return x;
}
// bit i of the low half of x moved to bit 2i
__device__ __forceinline__ uint32_t plan_spread(uint32_t x) {
  x &= 0x0000ffffu;
  x = (x | (x << 8)) & 0x00ff00ffu;
  x = (x | (x << 4)) & 0x0f0f0f0fu;
  x = (x | (x << 2)) & 0x33333333u;
  x = (x | (x << 1)) & 0x55555555u;
  return x;
}
// eight mask bytes -> eight bits (a byte counts when it is not zero): 0 / 1 in every byte, then the dot product with the
// bits' places
__device__ __forceinline__ uint32_t plan_ones(uint32_t v) {
  return ((((v & 0x7f7f7f7fu) + 0x7f7f7f7fu) | v) >> 7) & 0x01010101u;
}
__device__ __forceinline__ uint32_t plan_octet(uint32_t a, uint32_t b) {
  return plan_dot4(plan_ones(a), 0x08040201u, plan_dot4(plan_ones(b), 0x80402010u, 0u));
}
// four mask bytes, or the four bytes of a word of a bitmap -> four bits
__device__ __forceinline__ uint32_t plan_nibble(uint32_t v) { return plan_dot4(plan_ones(v), 0x08040201u, 0u); }
// four bits -> four bytes of 0 / 1 (bit i to bit 8 i: a copy shifted by 7 i each, then the one bit of each byte)
__device__ __forceinline__ uint32_t plan_bytes(uint32_t nib) {
  return __umul24(nib, 0x204081u) & 0x01010101u;
}

// floor(a / d) with m = plan_magic(d) = ceil(2^32 / d) worked out on the host: one multiply instead of a division by a
// run-time value.  Exact while a * d < 2^32 (the excess of m over 2^32 / d is below one, so the quotient is off by less
// than a / 2^32 < 1 / d); the planes of a plan are held to 2^20 pixels per sample and 2^11 per row for that.  d = 1
// has no 32-bit magic number: a itself, by a select.
inline unsigned plan_magic(int d) { return d <= 1 ? 0u : (unsigned)(0xffffffffu / (unsigned)d + 1u); }
__device__ __forceinline__ int plan_div(int a, unsigned m) {
  const int q = (int)__umulhi((unsigned)a, m);
  return m == 0u ? a : q;
}
// the bits of word j of a row of w pixels that are pixels
__device__ __forceinline__ uint32_t plan_valid(int w, int j) {
  const int left = w - 32 * j;
  return left >= 32 ? 0xffffffffu : ((1u << left) - 1u);
}

// specialised forms of the footprint (kernel size, stride and "same" padding K / 2 at compile time)
enum { PLAN_KEY_GENERIC = 0, PLAN_KEY_C11, PLAN_KEY_C31, PLAN_KEY_C51, PLAN_KEY_C71, PLAN_KEY_C91, PLAN_KEY_C111, PLAN_KEY_C32, PLAN_KEY_C52,
       PLAN_KEY_C72, PLAN_KEY_C92, PLAN_KEY_UP, PLAN_KEY_UP3, PLAN_KEY_UP5, PLAN_KEY_T32, PLAN_KEY_T52, PLAN_KEY_ALL };
constexpr int PLAN_MAX_K1 = 11, PLAN_MAX_K2 = 9;       // widest windows of stride 1 and 2 among them
constexpr int plan_key_size(int key) {
  return key == PLAN_KEY_C31 || key == PLAN_KEY_C32 || key == PLAN_KEY_T32 ? 3 : key == PLAN_KEY_C51 || key == PLAN_KEY_C52 || key == PLAN_KEY_T52 ? 5
         : key == PLAN_KEY_C71 || key == PLAN_KEY_C72 ? 7 : key == PLAN_KEY_C91 || key == PLAN_KEY_C92 ? 9 : key == PLAN_KEY_C111 ? 11 : 1;
}

// What the computing waves of a step know of it.
struct PlanIn {
  const uint32_t* lds;
  int in1, in2;             // LDS word offsets (in2: that of in1 where there is one input)
  int zero;                 // LDS word offset of the words of zeros
  int ww, h;                // words per row and rows of the input
};

// The K rows of a window, and of the windows of the R - 1 output rows below it (R = 1 or 2, S input rows apart): v[r][q] is
// the OR of word j0 + q of the rows first + r * S ... first + r * S + K - 1.  Rows that both windows hold are read once.
// Rows outside the plane come from the words of zeros.  A word left or right of the row is a word of a neighbouring row
// (or of the header): the caller drops those.
template <int K, int N, int S, int R, bool TWO>
__device__ __forceinline__ void plan_rows(const PlanIn& in, int first, int j0, uint32_t (&v)[R][N]) {
  int off = first * in.ww + j0;
  uint32_t both[N];
#pragma unroll
  for (int q = 0; q < N; ++q) {
    both[q] = 0u;
#pragma unroll
    for (int r = 0; r < R; ++r) v[r][q] = 0u;
  }
#pragma unroll
  for (int ky = 0; ky < K + (R - 1) * S; ++ky) {
    const bool ok = (unsigned)(first + ky) < (unsigned)in.h;
    const uint32_t* p1 = in.lds + (ok ? in.in1 + off : in.zero);
    const uint32_t* p2 = in.lds + (ok ? in.in2 + off : in.zero);
#pragma unroll
    for (int q = 0; q < N; ++q) {
      const uint32_t x = TWO ? p1[q] | p2[q] : p1[q];
      if (R == 2 && ky < S) v[0][q] |= x;
      else if (R == 2 && ky >= K) v[R - 1][q] |= x;
      else both[q] |= x;
    }
    off += in.ww;
  }
#pragma unroll
  for (int q = 0; q < N; ++q)
#pragma unroll
    for (int r = 0; r < R; ++r) v[r][q] |= both[q];
}

// Output words j of rows y .. y + R - 1 of a specialised footprint (pixels 32*j .. 32*j+31; R = 2: y is even).
template <int KEY, bool TWO, int R>
__device__ __forceinline__ void plan_foot_words(const PlanIn& in, int y, int j, uint32_t (&r)[R]) {
  constexpr int K = plan_key_size(KEY);
  constexpr int P = K / 2;
  if constexpr (KEY == PLAN_KEY_C11) {
    uint32_t v[R][1];
    plan_rows<1, 1, 1, R, TWO>(in, y, j, v);
#pragma unroll
    for (int i = 0; i < R; ++i) r[i] = v[i][0];
  } else if constexpr (KEY >= PLAN_KEY_C31 && KEY <= PLAN_KEY_C111) {
    uint32_t v[R][3];
    plan_rows<K, 3, 1, R, TWO>(in, y - P, j - 1, v);
#pragma unroll
    for (int i = 0; i < R; ++i) {
      const uint32_t vp = j > 0 ? v[i][0] : 0u, vn = j + 1 < in.ww ? v[i][2] : 0u;
      r[i] = 0u;
#pragma unroll
      for (int t = 0; t < K; ++t) r[i] |= plan_shift(vp, v[i][1], vn, t - P);
    }
  } else if constexpr (KEY >= PLAN_KEY_C32 && KEY <= PLAN_KEY_C92) {
    // the window OR at input positions 64*j .. 64*j+63, of which the even ones are the outputs
    uint32_t v[R][4];
    plan_rows<K, 4, 2, R, TWO>(in, 2 * y - P, 2 * j - 1, v);
#pragma unroll
    for (int i = 0; i < R; ++i) {
      const uint32_t v0 = j > 0 ? v[i][0] : 0u, v2 = 2 * j + 1 < in.ww ? v[i][2] : 0u, v3 = 2 * j + 2 < in.ww ? v[i][3] : 0u;
      uint32_t d0 = 0u, d1 = 0u;
#pragma unroll
      for (int t = 0; t < K; ++t) {
        d0 |= plan_shift(v0, v[i][1], v2, t - P);
        d1 |= plan_shift(v[i][1], v2, v3, t - P);
      }
      r[i] = plan_even_bits(d0) | (plan_even_bits(d1) << 16);
    }
  } else {
    const int js = j >> 1, sh = 16 * (j & 1), e = y & 1, m = y >> 1;
    const bool okp = js > 0, okn = js + 1 < in.ww;
    uint32_t v[R][3];
    if constexpr (KEY == PLAN_KEY_UP) {
      // out[2m] = in[m-1] | in[m], out[2m+1] = in[m] | in[m+1], rows and columns alike (clamping at the border adds
      // nothing: the clamped neighbour is the pixel itself)
      plan_rows<2, 3, 1, R, TWO>(in, m - 1 + e, js - 1, v);
    } else if constexpr (KEY == PLAN_KEY_UP3) {
      // ... and a 3x3 window over that: in[m-1 .. m+1], for both
      plan_rows<3, 3, 0, R, TWO>(in, m - 1, js - 1, v);
    } else if constexpr (KEY == PLAN_KEY_UP5) {
      // ... and a 5x5 window: in[m-2 .. m+1], in[m-1 .. m+2]
      plan_rows<4, 3, 1, R, TWO>(in, m - 2 + e, js - 1, v);
    } else {
      // transposed conv, stride 2: output 2m + e sees input m + (e + P - kk) / 2 for the taps kk with e + P - kk even:
      // K = 3: {m} for e = 0, {m, m+1} for e = 1;  K = 5: {m-1, m, m+1}, {m, m+1}
      uint32_t w[1][3];
      if constexpr (K == 3) {
        plan_rows<1, 3, 1, 1, TWO>(in, m, js - 1, v);
        plan_rows<1, 3, 1, 1, TWO>(in, e ? m + 1 : -1, js - 1, w);
      } else {
        plan_rows<2, 3, 1, 1, TWO>(in, m, js - 1, v);
        plan_rows<1, 3, 1, 1, TWO>(in, e ? -1 : m - 1, js - 1, w);
      }
#pragma unroll
      for (int q = 0; q < 3; ++q) v[0][q] |= w[0][q];
    }
#pragma unroll
    for (int i = 0; i < R; ++i) {
      const uint32_t vp = okp ? v[i][0] : 0u, vn = okn ? v[i][2] : 0u;
      uint32_t ev = 0u, od = 0u;
      if constexpr (KEY == PLAN_KEY_UP) {
        ev = v[i][1] | plan_shift(vp, v[i][1], vn, -1);
        od = v[i][1] | plan_shift(vp, v[i][1], vn, 1);
      } else if constexpr (KEY == PLAN_KEY_UP3 || KEY == PLAN_KEY_UP5) {
        ev = od = v[i][1] | plan_shift(vp, v[i][1], vn, -1) | plan_shift(vp, v[i][1], vn, 1);
        if (KEY == PLAN_KEY_UP5) ev |= plan_shift(vp, v[i][1], vn, -2), od |= plan_shift(vp, v[i][1], vn, 2);
      } else {
#pragma unroll
        for (int kx = 0; kx < K; ++kx) {
          const int d2 = P - kx;
          if (d2 & 1) od |= plan_shift(vp, v[i][1], vn, (d2 + 1) >> 1);
          else ev |= plan_shift(vp, v[i][1], vn, d2 >> 1);
        }
      }
      r[i] = plan_spread(ev >> sh) | (plan_spread(od >> sh) << 1);
    }
  }
}

// The general form: any kernel size and padding, conv of stride 1 or 2, transposed conv of stride 2.  Output word j of
// row oy; words and rows outside the input count as zero.
__device__ uint32_t plan_foot_general(const PlanIn& in, int geom, int oy, int j) {
  const int foot = geom & 255, k = (geom >> 8) & 255, s = (geom >> 16) & 255, p = (geom >> 24) & 255;
  auto word = [&](int y, int jj) -> uint32_t {
    const bool ok = (unsigned)y < (unsigned)in.h && (unsigned)jj < (unsigned)in.ww;
    const int o = y * in.ww + jj;
    return in.lds[ok ? in.in1 + o : in.zero] | in.lds[ok ? in.in2 + o : in.zero];
  };
  if (foot == MIE_FOOT_CONV && s == 1) {
    uint32_t vp = 0u, vc = 0u, vn = 0u, r = 0u;
    for (int ky = 0; ky < k; ++ky) {
      vp |= word(oy - p + ky, j - 1);
      vc |= word(oy - p + ky, j);
      vn |= word(oy - p + ky, j + 1);
    }
    for (int t = 0; t < k; ++t) r |= plan_shift(vp, vc, vn, t - p);
    return r;
  }
  if (foot == MIE_FOOT_CONV) {
    uint32_t v[4] = {0u, 0u, 0u, 0u}, d0 = 0u, d1 = 0u;
    for (int ky = 0; ky < k; ++ky)
      for (int q = 0; q < 4; ++q) v[q] |= word(2 * oy - p + ky, 2 * j - 1 + q);
    for (int t = 0; t < k; ++t) {
      d0 |= plan_shift(v[0], v[1], v[2], t - p);
      d1 |= plan_shift(v[1], v[2], v[3], t - p);
    }
    return plan_even_bits(d0) | (plan_even_bits(d1) << 16);
  }
  const int js = j >> 1, sh = 16 * (j & 1), e = oy & 1, m = oy >> 1;
  uint32_t vp = 0u, vc = 0u, vn = 0u, ev = 0u, od = 0u;
  for (int ky = 0; ky < k; ++ky) {
    const int d2 = e + p - ky;
    if (d2 & 1) continue;
    vp |= word(m + (d2 >> 1), js - 1);
    vc |= word(m + (d2 >> 1), js);
    vn |= word(m + (d2 >> 1), js + 1);
  }
  for (int kx = 0; kx < k; ++kx) {
    const int d2 = p - kx;
    if (d2 & 1) od |= plan_shift(vp, vc, vn, (d2 + 1) >> 1);
    else ev |= plan_shift(vp, vc, vn, d2 >> 1);
  }
  return plan_spread(ev >> sh) | (plan_spread(od >> sh) << 1);
}

// R = 2: a thread makes the words of two rows, where there are more words than threads (fewer reads a word, a longer step).
template <int KEY, bool TWO, int R>
__device__ __forceinline__ void plan_foot_all(const PlanIn& in, uint32_t* out, int ho, int wo, uint32_t m_words, int geom, int r,
                                              int nthr) {
  const int wwo = (wo + 31) >> 5, total = (R == 2 ? (ho + 1) >> 1 : ho) * wwo;
  for (int wd = r; wd < total; wd += nthr) {
    const int y = R * plan_div(wd, m_words), j = wd - (R == 2 ? y >> 1 : y) * wwo;
    uint32_t v[R];
    if constexpr (KEY == PLAN_KEY_ALL) v[0] = 0xffffffffu;
    else if constexpr (KEY == PLAN_KEY_GENERIC) v[0] = plan_foot_general(in, geom, y, j);
    else plan_foot_words<KEY, TWO, R>(in, y, j, v);
    const uint32_t valid = plan_valid(wo, j);
    out[y * wwo + j] = v[0] & valid;
    if (R == 2 && y + 1 < ho) out[(y + 1) * wwo + j] = v[R - 1] & valid;
  }
}

// The bitmap of a footprint step: thread r of nthr takes words r, r + nthr, ...
__device__ void plan_compute(uint32_t pw, uint32_t* lds, int zero, int r, int nthr) {
  const uint32_t io = plan_word(pw, PS_IN), ow = plan_word(pw, PS_OUT_WIN), wk = plan_word(pw, PS_WOUT_KEY);
  const int ho = (int)plan_word(pw, PS_HOUT), wo = (int)(wk & 0xffffu), key = (int)((wk >> 16) & 0xffu);
  const uint32_t mw = plan_word(pw, PS_MWORDS);
  const int geom = (int)plan_word(pw, PS_GEOM);
  uint32_t* out = lds + (ow & 0xffffu);
  PlanIn in;
  in.lds = lds;
  in.zero = zero;
  in.in1 = (int)(io & 0xffffu);
  const bool two = (io >> 16) != PLAN_IN_NONE;
  in.in2 = two ? (int)(io >> 16) : in.in1;
  in.ww = ((int)(ow >> 16) + 31) >> 5;
  in.h = (int)plan_word(pw, PS_HIN);
  const bool many = ho * ((wo + 31) >> 5) > nthr;
  switch (key) {       // uniform over the wave
#define PLAN_CASE(KEY)                                                                          \
    case KEY:                                                                                   \
      if (two) plan_foot_all<KEY, true, 1>(in, out, ho, wo, mw, geom, r, nthr);                 \
      else plan_foot_all<KEY, false, 1>(in, out, ho, wo, mw, geom, r, nthr);                    \
      break
#define PLAN_CASE_R(KEY)                                                                        \
    case KEY:                                                                                   \
      if (two) plan_foot_all<KEY, true, 1>(in, out, ho, wo, mw, geom, r, nthr);                 \
      else if (many) plan_foot_all<KEY, false, 2>(in, out, ho, wo, mw, geom, r, nthr);          \
      else plan_foot_all<KEY, false, 1>(in, out, ho, wo, mw, geom, r, nthr);                    \
      break
    PLAN_CASE(PLAN_KEY_C11);
    PLAN_CASE_R(PLAN_KEY_C31);
    PLAN_CASE_R(PLAN_KEY_C51);
    PLAN_CASE(PLAN_KEY_C71);
    PLAN_CASE(PLAN_KEY_C91);
    PLAN_CASE(PLAN_KEY_C111);
    PLAN_CASE_R(PLAN_KEY_C32);
    PLAN_CASE_R(PLAN_KEY_C52);
    PLAN_CASE_R(PLAN_KEY_C72);
    PLAN_CASE_R(PLAN_KEY_C92);
    case PLAN_KEY_UP:
      if (two && many) plan_foot_all<PLAN_KEY_UP, true, 2>(in, out, ho, wo, mw, geom, r, nthr);
      else if (many) plan_foot_all<PLAN_KEY_UP, false, 2>(in, out, ho, wo, mw, geom, r, nthr);
      else if (two) plan_foot_all<PLAN_KEY_UP, true, 1>(in, out, ho, wo, mw, geom, r, nthr);
      else plan_foot_all<PLAN_KEY_UP, false, 1>(in, out, ho, wo, mw, geom, r, nthr);
      break;
    PLAN_CASE(PLAN_KEY_UP3);
    PLAN_CASE(PLAN_KEY_UP5);
    PLAN_CASE(PLAN_KEY_T32);
    PLAN_CASE(PLAN_KEY_T52);
#undef PLAN_CASE_R
#undef PLAN_CASE
    case PLAN_KEY_ALL: plan_foot_all<PLAN_KEY_ALL, false, 1>(in, out, ho, wo, mw, geom, r, nthr); break;
    default: plan_foot_all<PLAN_KEY_GENERIC, true, 1>(in, out, ho, wo, mw, geom, r, nthr);
  }
}

// A mask in memory -> bitmap: two words a thread asked for together where rows allow 16-byte loads.
__device__ __forceinline__ void plan_load(uint32_t pw, uint32_t* lds, int n, int r, int nthr) {
  const uint32_t ow = plan_word(pw, PS_OUT_WIN), wk = plan_word(pw, PS_WOUT_KEY);
  const int ho = (int)plan_word(pw, PS_HOUT), wo = (int)(wk & 0xffffu), wwo = (wo + 31) >> 5, total = ho * wwo;
  const uint32_t mw = plan_word(pw, PS_MWORDS);
  const uint8_t* src = plan_ptr<const uint8_t>(pw, PS_PIX) + (long long)n * ho * wo;
  uint32_t* out = lds + (ow & 0xffffu);
  const int unit = (int)(wk >> 28);
  if (unit == 2) {
    constexpr int U = 2;
    for (int w0 = r; w0 < total; w0 += U * nthr) {
      uint4 v[U][2];
      bool half[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int wd = w0 + u * nthr < total ? w0 + u * nthr : w0;
        const int y = plan_div(wd, mw), j = wd - y * wwo;
        const uint4* p = reinterpret_cast<const uint4*>(src + (long long)y * wo + 32 * j);
        half[u] = wo - 32 * j <= 16;
        v[u][0] = p[0];
        v[u][1] = p[half[u] ? 0 : 1];
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        uint32_t b[2];
#pragma unroll
        for (int q = 0; q < 2; ++q)
          b[q] = plan_octet(v[u][q].x, v[u][q].y) | (plan_octet(v[u][q].z, v[u][q].w) << 8);
        if (w0 + u * nthr < total) out[w0 + u * nthr] = b[0] | (half[u] ? 0u : b[1] << 16);
      }
    }
    return;
  }
  for (int wd = r; wd < total; wd += nthr) {
    const int y = plan_div(wd, mw), j = wd - y * wwo;
    const int x0 = 32 * j, nb = (wo - x0 < 32) ? wo - x0 : 32;
    const uint8_t* row = src + (long long)y * wo + x0;
    uint32_t bits = 0u;
    if (unit == 1) {
      const uint32_t* r4 = reinterpret_cast<const uint32_t*>(row);
      const int nq = nb >> 2;
      uint32_t v[8];
#pragma unroll
      for (int q = 0; q < 8; ++q) v[q] = r4[q < nq ? q : 0];
#pragma unroll
      for (int q = 0; q < 8; ++q) bits |= q < nq ? plan_nibble(v[q]) << (4 * q) : 0u;
    } else {
      for (int b0 = 0; b0 < nb; b0 += 8) {
        uint8_t v[8];
#pragma unroll
        for (int q = 0; q < 8; ++q) v[q] = row[b0 + q < nb ? b0 + q : 0];
#pragma unroll
        for (int q = 0; q < 8; ++q) bits |= (b0 + q < nb && v[q] != 0) ? 1u << (b0 + q) : 0u;
      }
    }
    out[wd] = bits;
  }
}

// 16 pixels of a row of a mask: bits -> bytes, as wide as the rows allow.
__device__ __forceinline__ void plan_put16(uint8_t* p, uint32_t b16, int left, int unit) {
  const uint4 v = make_uint4(plan_bytes(b16 & 15u), plan_bytes((b16 >> 4) & 15u), plan_bytes((b16 >> 8) & 15u), plan_bytes((b16 >> 12) & 15u));
  if (unit == 2) {
    *reinterpret_cast<uint4*>(p) = v;
  } else if (unit == 1) {
    uint32_t* p4 = reinterpret_cast<uint32_t*>(p);
    p4[0] = v.x;
    if (left > 4) p4[1] = v.y;
    if (left > 8) p4[2] = v.z;
    if (left > 12) p4[3] = v.w;
  } else {
    for (int q = 0; q < 16 && q < left; ++q) p[q] = (uint8_t)((b16 >> q) & 1u);
  }
}

__device__ __forceinline__ int plan_tiles(uint32_t pw) {
  const int ho = (int)plan_word(pw, PS_HOUT), wo = (int)(plan_word(pw, PS_WOUT_KEY) & 0xffffu);
  return ((ho + MIE_TILE - 1) / MIE_TILE) * ((wo + MIE_TILE - 1) / MIE_TILE);
}
// The tiles of a set whose flags a workgroup writes where it does not own sets: [lo, hi).
__device__ __forceinline__ void plan_slice(uint32_t pw, int share, int& lo, int& hi) {
  const int tiles = plan_tiles(pw), own = (int)plan_word(pw, PS_OWN);
  lo = share * own;
  hi = lo + own < tiles ? lo + own : tiles;
}
// Whether tile t of a set holds an active pixel.
__device__ __forceinline__ bool plan_tile_any(const uint32_t* bitmap, int t, int ho, int wo, uint32_t mt) {
  const int wwo = (wo + 31) >> 5, tiles_x = (wo + MIE_TILE - 1) / MIE_TILE, ty = plan_div(t, mt), tx = t - ty * tiles_x;
  uint32_t any = 0u;
#pragma unroll
  for (int q = 0; q < MIE_TILE; ++q) {
    const int y = ty * MIE_TILE + q;
    any |= bitmap[(y < ho ? y : ho - 1) * wwo + (tx >> 2)];       // the last row again where a tile ends below the plane
  }
  return ((any >> (8 * (tx & 3))) & 0xffu) != 0u;
}

// Not resident: what a step leaves in memory, from its bitmap, by threads r of nthr.  The pixel mask, this workgroup's
// slice (share of shares), and, in LDS, the state of the tiles it writes the flags of: byte t - lo of the step's part of
// the flag area.
__device__ void plan_write(uint32_t pw, const uint32_t* lds, uint8_t* fl, int n, int share, int shares, int r, int nthr) {
  const int ho = (int)plan_word(pw, PS_HOUT), wo = (int)(plan_word(pw, PS_WOUT_KEY) & 0xffffu), wwo = (wo + 31) >> 5;
  const uint32_t* out = lds + (plan_word(pw, PS_OUT_WIN) & 0xffffu);
  const uint32_t mu = plan_word(pw, PS_MUNITS), mt = plan_word(pw, PS_MTILES);
  const int unit = (int)(plan_word(pw, PS_WOUT_KEY) >> 28), per_row = (wo + 15) >> 4, units = ho * per_row;
  uint8_t* pm = plan_ptr<uint8_t>(pw, PS_PIX) + (long long)n * ho * wo;
  for (int u = share * nthr + r; u < units; u += shares * nthr) {
    const int y = plan_div(u, mu), q = u - y * per_row;
    plan_put16(pm + (long long)y * wo + 16 * q, out[y * wwo + (q >> 1)] >> (16 * (q & 1)), wo - 16 * q, unit);
  }
  int lo, hi;
  plan_slice(pw, share, lo, hi);
  uint8_t* bits = fl + plan_word(pw, PS_FL);
  for (int t = lo + r; t < hi; t += nthr) bits[t - lo] = plan_tile_any(out, t, ho, wo, mt) ? 1 : 0;
}

// Resident: a thread's 16-pixel unit u of all sets' units -- its set is the last step whose units start at or below it --
// as the place of its bits in LDS and of its bytes in memory.
// (bits: LDS word | upper half << 16 | pixels of it that the row has << 17 | width of the stores << 22)
struct PlanPut { uint8_t* dst; uint32_t bits; };
__device__ __forceinline__ PlanPut plan_find(const uint32_t* lds, int n_steps, int n, int u) {
  int i = 0;
#pragma unroll
  for (int b = 32; b > 0; b >>= 1) {
    const int at = i + b < n_steps ? i + b : i;
    i = (int)lds[at * PS_WORDS + PS_UBASE] <= u ? at : i;
  }
  const uint32_t* p = lds + i * PS_WORDS;
  const int ho = (int)p[PS_HOUT], wo = (int)(p[PS_WOUT_KEY] & 0xffffu), wwo = (wo + 31) >> 5, per_row = (wo + 15) >> 4;
  const int q0 = u - (int)p[PS_UBASE], y = plan_div(q0, p[PS_MUNITS]), q = q0 - y * per_row;
  PlanPut r;
  r.dst = reinterpret_cast<uint8_t*>(((unsigned long long)p[PS_PIX_HI] << 32) | p[PS_PIX]) + ((long long)n * ho + y) * wo + 16 * q;
  const int left = wo - 16 * q < 16 ? wo - 16 * q : 16;
  r.bits = ((p[PS_OUT_WIN] & 0xffffu) + (uint32_t)(y * wwo + (q >> 1))) | (uint32_t)(q & 1) << 16 | (uint32_t)left << 17 | (p[PS_WOUT_KEY] >> 28) << 22;
  return r;
}
__device__ __forceinline__ void plan_put(const uint32_t* lds, const PlanPut& p) {
  plan_put16(p.dst, lds[p.bits & 0xffffu] >> ((p.bits >> 12) & 16u), (int)((p.bits >> 17) & 31u), (int)(p.bits >> 22));
}

// The lists, counts and flags of a set the workgroup owns, from its bitmap and its tiles' old state: by all threads.
// `par` alternates from set to set (and chunk to chunk) so that one barrier a chunk is enough.
__device__ __forceinline__ void plan_rank(uint32_t pw, const uint32_t* lds, const uint8_t* old, int* s_tot, int& par, int tid) {
  const int ho = (int)plan_word(pw, PS_HOUT), wo = (int)(plan_word(pw, PS_WOUT_KEY) & 0xffffu), tiles = plan_tiles(pw);
  const uint32_t mt = plan_word(pw, PS_MTILES);
  const uint8_t* o_tiles = old + plan_word(pw, PS_FL);
  const uint32_t* bitmap = lds + (plan_word(pw, PS_OUT_WIN) & 0xffffu);
  uint32_t* flags = plan_ptr<uint32_t>(pw, PS_FLAGS);
  int32_t* act = plan_ptr<int32_t>(pw, PS_TILES);
  int32_t* stale = plan_ptr<int32_t>(pw, PS_STALE);
  int32_t* counts = plan_ptr<int32_t>(pw, PS_COUNTS);
  const int wave = tid >> 6;
  int run_a = 0, run_s = 0;
  for (int t0 = 0; t0 < tiles; t0 += PLAN_THREADS) {
    const int t = t0 + tid;
    bool a = false, s = false;
    if (t < tiles) {
      a = plan_tile_any(bitmap, t, ho, wo, mt);
      const uint32_t o = o_tiles[t];
      s = !a && (o & 1u) != 0u;
      flags[t] = next_flag(o, a);
    }
    const unsigned long long ba = __ballot(a), bs = __ballot(s);
    int* tot = s_tot + par * PLAN_WAVES;
    par ^= 1;
    if ((tid & 63) == 0) tot[wave] = __popcll(ba) | (__popcll(bs) << 16);        // at most 64 each
    __syncthreads();
    int before = 0, all = 0;
#pragma unroll
    for (int w = 0; w < PLAN_WAVES; ++w) {
      const int v = tot[w];
      before += w < wave ? v : 0;
      all += v;                                              // at most 1024 in either half
    }
    const int ra = run_a + (before & 0xffff), rs = run_s + (before >> 16);
    if (a) act[__builtin_amdgcn_mbcnt_hi((uint32_t)(ba >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)ba, (uint32_t)ra))] = t;
    if (s) stale[__builtin_amdgcn_mbcnt_hi((uint32_t)(bs >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)bs, (uint32_t)rs))] = t;
    run_a += all & 0xffff;
    run_s += all >> 16;
  }
  if (tid == 0) {
    counts[MIE_CNT_ACTIVE] = run_a;
    counts[MIE_CNT_STALE] = run_s;
  }
}

// (64 registers: beside a plan made ahead there is room for a conv's workgroup on the same CU)
__global__ __launch_bounds__(PLAN_THREADS, 8) void k_plan_bits(PlanArgs a) {
  extern __shared__ __attribute__((aligned(16))) uint32_t plan_lds[];
  uint32_t* lds = plan_lds;
  const int n = blockIdx.y, tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int share = blockIdx.x, shares = gridDim.x;
  const int step_words = a.n_steps * PS_WORDS, lw = lane < PS_WORDS ? lane : 0;
  uint8_t* task = reinterpret_cast<uint8_t*>(lds + step_words);
  uint8_t* fl = reinterpret_cast<uint8_t*>(lds + a.flag_off);
  int* s_tot = reinterpret_cast<int*>(lds + a.zero_off + PLAN_ZERO_WORDS);        // 2 * PLAN_WAVES
  {
    // The steps and the task table go from the argument block to LDS in one batch: read where they are used, every
    // step's words would be a cache miss of their own in a chain where nothing else hides it.
    const uint32_t* tsrc = reinterpret_cast<const uint32_t*>(a.task);
    const int tw = (a.n_levels + 2) * (PLAN_WAVES / 4);
    for (int i = tid; i < step_words + tw; i += PLAN_THREADS) lds[i] = i < step_words ? a.st[i] : tsrc[i - step_words];
    if (tid < PLAN_ZERO_WORDS) lds[a.zero_off + tid] = 0u;
  }
  const int first = a.owned ? a.head[share] : PLAN_IDLE;
  __syncthreads();
  // The old state of the tiles of the first set this workgroup owns is asked for, then the masks that level 0 loads; while
  // those are on their way a thread finds the place of its first unit of the pixel masks.
  uint32_t f0 = 0u, fl0 = 0u;
  int tiles0 = 0;
  if (first != PLAN_IDLE) {
    const uint32_t q = lds[first * PS_WORDS + lw];
    tiles0 = plan_tiles(q);
    fl0 = plan_word(q, PS_FL);
    f0 = plan_ptr<const uint32_t>(q, PS_FLAGS)[tid < tiles0 ? tid : 0];
  }
  const int load = __builtin_amdgcn_readfirstlane((int)task[wave]);       // level 0: masks from memory, by all waves
  if (load < a.n_loads) {
    const uint32_t q = lds[load * PS_WORDS + lw], wv = plan_word(q, PS_WAVES);
    plan_load(q, lds, n, (wave - (int)(wv & 255u)) * 64 + lane, (int)((wv >> 8) & 255u) * 64);
  }
  PlanPut put = {nullptr, 0u};
  const int u0 = share * PLAN_THREADS + tid;
  if (a.resident) put = plan_find(lds, a.n_steps, n, u0 < a.units ? u0 : 0);
  if (first != PLAN_IDLE) {
    if (tid < tiles0) fl[fl0 + tid] = (uint8_t)(f0 & 1u);
    // what is left: tiles beyond the first 1024, further sets
    for (int i = first; i != PLAN_IDLE;) {
      const uint32_t p = lds[i * PS_WORDS + lw];
      const int tiles = plan_tiles(p);
      const uint32_t* flags = plan_ptr<const uint32_t>(p, PS_FLAGS);
      uint8_t* o = fl + plan_word(p, PS_FL);
      for (int t = tid + (i == first ? PLAN_THREADS : 0); t < tiles; t += PLAN_THREADS) o[t] = (uint8_t)(flags[t] & 1u);
      i = (int)plan_word(p, PS_OWN);
    }
  }
  __syncthreads();
  const int compute_waves = a.resident ? PLAN_WAVES : PLAN_COMPUTE_WAVES;
  int idx = __builtin_amdgcn_readfirstlane((int)task[PLAN_WAVES + wave]);
  int next = task[2 * PLAN_WAVES + wave];
  uint32_t pw = lds[(idx == PLAN_IDLE ? 0 : idx) * PS_WORDS + lw];
  for (int lv = 1; lv < a.n_levels; ++lv) {
    // the step of the next level and the number of the one after it
    const int nidx = __builtin_amdgcn_readfirstlane(next);
    const uint32_t npw = lds[(nidx == PLAN_IDLE ? 0 : nidx) * PS_WORDS + lw];
    next = task[(lv + 2 <= a.n_levels ? lv + 2 : 0) * PLAN_WAVES + wave];
    if (idx != PLAN_IDLE) {
      const uint32_t wv = plan_word(pw, PS_WAVES);
      if (wave < compute_waves) {
        int r = (wave - (int)(wv & 255u)) * 64 + lane;
        const int nthr = (int)((wv >> 8) & 255u) * 64;
        asm volatile("" : "+v"(r));        // or a dozen multiples of it are kept in registers through the whole chain
        if (plan_kind(pw) == PLAN_KIND_LOAD) plan_load(pw, lds, n, r, nthr);
        else plan_compute(pw, lds, a.zero_off, r, nthr);
      } else {
        // (the writing waves read the slots of the level before while this level's are written: the host keeps them
        // apart -- a slot is handed on one level after its last reader)
        plan_write(pw, lds, fl, n, share, shares, (wave - (int)((wv >> 16) & 255u)) * 64 + lane, (int)(wv >> 24) * 64);
      }
    }
    __syncthreads();
    idx = nidx;
    pw = npw;
  }
  if (a.resident) {
    // the pixel masks of all sets: this workgroup's slice of their units
    for (int u = u0; u < a.units; u += shares * PLAN_THREADS) {
      if (u != u0) put = plan_find(lds, a.n_steps, n, u);
      plan_put(lds, put);
    }
  } else {
    for (int i = a.first_last; i < a.n_steps; ++i)       // the last level, by everybody
      plan_write(lds[i * PS_WORDS + lw], lds, fl, n, share, shares, tid, PLAN_THREADS);
    __syncthreads();
  }
  if (a.owned) {
    int par = 0;
    for (int i = first; i != PLAN_IDLE;) {
      const uint32_t q = lds[i * PS_WORDS + lw];
      plan_rank(q, lds, fl, s_tot, par, tid);
      i = (int)plan_word(q, PS_OWN);
    }
    return;
  }
  // one wave a set: the flags of this workgroup's slice, old state asked for here
  for (int i = wave; i < a.n_steps; i += PLAN_WAVES) {
    const uint32_t q = lds[i * PS_WORDS + lw];
    if (plan_kind(q) != PLAN_KIND_FOOT) continue;
    int lo, hi;
    plan_slice(q, share, lo, hi);
    const int ho = (int)plan_word(q, PS_HOUT), wo = (int)(plan_word(q, PS_WOUT_KEY) & 0xffffu);
    const uint32_t mt = plan_word(q, PS_MTILES);
    const uint8_t* now = fl + plan_word(q, PS_FL);
    const uint32_t* bitmap = lds + (plan_word(q, PS_OUT_WIN) & 0xffffu);
    uint32_t* flags = plan_ptr<uint32_t>(q, PS_FLAGS) + (long long)n * plan_tiles(q);
    for (int t = lo + lane; t < hi; t += 64) {
      const uint32_t o = flags[t];
      flags[t] = next_flag(o, a.resident ? plan_tile_any(bitmap, t, ho, wo, mt) : now[t - lo] != 0);
    }
  }
}

// The lists of every set of a plan: block b is chunk b - first_chunk[i] of the compaction of set i (as
// k_compact_tiles).  The table of first chunks is a few cache lines read in one go; a block then touches only the
// line of its own set.
struct PlanCompactSet {
  int32_t* tiles;
  int32_t* stale;
  int32_t* counts;
  uint32_t* flags;
  int cap, pad_;
};
struct PlanCompactArgs {
  int n_sets, pad_;
  int first_chunk[MIE_PLAN_MAX_STEPS + 2];     // first_chunk[n_sets] = number of blocks
  PlanCompactSet set[MIE_PLAN_MAX_STEPS];
};

__global__ __launch_bounds__(COMPACT_THREADS) void k_plan_compact(PlanCompactArgs a) {
  __shared__ int s_tot[2 * COMPACT_WAVES * COMPACT_ITEMS];
  __shared__ int s_base[2 * COMPACT_WAVES];
  const int b = blockIdx.x;
  int i = 0;
#pragma unroll 1
  for (int q = 1; q < a.n_sets; ++q)
    if (a.first_chunk[q] <= b) i = q;
  const PlanCompactSet& st = a.set[i];
  BuildArgs ba;
  ba.cap = st.cap;
  ba.tiles = st.tiles; ba.stale = st.stale; ba.counts = st.counts; ba.flags = st.flags;
  compact_chunk(ba, b - a.first_chunk[i], a.first_chunk[i + 1] - a.first_chunk[i], s_tot, s_base);
}

// LDS a workgroup may use on the current device.
int plan_lds_limit(int* bytes, const char* who) {
  static int limit[64];
  int dev = -1;
  hipError_t e = hipGetDevice(&dev);
  MIE_REQUIRE(e == hipSuccess && dev >= 0 && dev < 64, MIE_ERR_LAUNCH, "%s: no current device (%s)", who, hipGetErrorString(e));
  if (limit[dev] == 0) {
    int v = 0;
    e = hipDeviceGetAttribute(&v, hipDeviceAttributeMaxSharedMemoryPerBlock, dev);
    MIE_REQUIRE(e == hipSuccess && v > 0, MIE_ERR_LAUNCH, "%s: cannot read the LDS size of device %d (%s)", who, dev, hipGetErrorString(e));
    limit[dev] = v;
  }
  *bytes = limit[dev];
  return MIE_OK;
}

// Whether a plan's LDS is there, and the opt-in for more than 64 KB of it (once per process).
int plan_lds_take(long long need_bytes, int limit, const char* who) {
  static long long opted[64];
  int dev = -1;
  hipError_t e = hipGetDevice(&dev);
  MIE_REQUIRE(e == hipSuccess && dev >= 0 && dev < 64, MIE_ERR_LAUNCH, "%s: no current device (%s)", who, hipGetErrorString(e));
  MIE_REQUIRE(need_bytes <= limit, MIE_ERR_CAPACITY,
              "%s: the masks of this plan need %lld bytes of LDS at once, the device offers %d per workgroup; "
              "build the plan in parts, or with mie_build_mask_tiles", who, need_bytes, limit);
  if (need_bytes > 65536 && need_bytes > opted[dev]) {
    e = hipFuncSetAttribute(reinterpret_cast<const void*>(k_plan_bits), hipFuncAttributeMaxDynamicSharedMemorySize, limit);
    MIE_REQUIRE(e == hipSuccess, MIE_ERR_CAPACITY, "%s: the device refuses %d bytes of dynamic LDS (%s)", who, limit,
                hipGetErrorString(e));
    opted[dev] = limit;
  }
  return MIE_OK;
}

// Host side of a plan: its steps (masks loaded from memory and ops), the level each runs in and the LDS its bitmap takes.
struct PlanHost {
  static constexpr int MAX = MIE_PLAN_MAX_STEPS;
  struct Step {
    int op;                     // the op, or -1: a mask loaded from memory
    int in[2];                  // steps whose bitmaps it reads, -1: none
    int k;                      // its window over them (conv windows of stride 1 and 2 that may have been widened)
    int src[2];                 // as in[], as the op says it
    const uint8_t* ptr;         // its mask in memory
    int h, w;
    long long words;
    int level, last;            // when its bitmap is made, and the last level that reads it (writing waves included)
    int rec;                    // the allocation its bitmap lies in
    bool up;                    // a window over an up-sampling, read from that one's inputs
  };
  struct Alloc { long long words, off; int born, rel; };
  Step st[MAX];
  int n_steps = 0, n_levels = 0;
  Alloc rec[MAX];
  int n_rec = 0;
  long long top = 0;            // words of LDS of all bitmaps

  // A conv window with "same" padding over the result of a stride-1 window with "same" padding is one wider window over
  // that one's input: read that, where the wide window has a form of its own.  So is a 3x3 or 5x5 window over a bilinear
  // up-sampling one over what that read: a decoder layer is one level and not two, while it and the up-sampling's own set have a
  // thread for every word (264x352: 1.1 us for 1.3 + 0.85 at a quarter of the resolution, 1.8 for 1.3 + 1.3 at half, 4.1 for 1.9 + 1.8 at the full one).
  void widen(const mie_plan_op* ops) {
    auto same = [&](const Step& s, int stride) {
      if (s.op < 0 || s.src[0] < 0) return false;
      const mie_plan_op& op = ops[s.op];
      return op.foot == MIE_FOOT_CONV && op.stride == stride && (op.k & 1) && op.pad == op.k / 2;
    };
    for (int i = 0; i < n_steps; ++i) {
      Step& s = st[i];
      const bool one = same(s, 1);
      if (!(one || same(s, 2)) || s.src[1] >= 0) continue;
      const Step& m = st[s.src[0]];
      if (one && (s.k == 3 || s.k == 5) && m.op >= 0 && ops[m.op].foot == MIE_FOOT_UP2X && m.src[0] >= 0 && s.words <= PLAN_UP_WORDS) {
        s.in[0] = m.src[0];
        s.in[1] = m.src[1];
        s.up = true;
        continue;
      }
      const int k = s.k + m.k - 1;
      if (m.up || !same(m, 1) || k > (one ? PLAN_MAX_K1 : PLAN_MAX_K2)) continue;
      s.in[0] = m.in[0];
      s.in[1] = m.in[1];
      s.k = k;
    }
  }
  void as_given(const mie_plan_op* ops) {
    for (int i = 0; i < n_steps; ++i) {
      st[i].in[0] = st[i].src[0];
      st[i].in[1] = st[i].src[1];
      st[i].k = st[i].op >= 0 ? ops[st[i].op].k : 0;
      st[i].up = false;
    }
  }

  // What a word of a step costs, roughly: the words it reads (R = 1) and some twenty instructions more.
  long long cost(int i, const mie_plan_op* ops) const {
    if (st[i].op < 0) return 20;
    const mie_plan_op& op = ops[st[i].op];
    const int rows = st[i].up ? (st[i].k == 5 ? 4 : 3) : op.foot == MIE_FOOT_CONV ? st[i].k : 2, words = op.foot == MIE_FOOT_CONV && op.stride == 2 ? 4 : 3;
    return rows * words * (st[i].in[1] >= 0 ? 2 : 1) + 20;
  }

  // Level 0 holds masks from memory only; they are there before the chain starts.  serial: one step after the other, a mask from memory right before the op that reads it first (the form
  // that needs least LDS).  Otherwise a step runs as soon as what it reads is there, at most so many a level.
  // resident: every bitmap is held to the end.
  void schedule(bool serial, bool resident, const mie_plan_op* ops) {
    int count[MAX + 2] = {0};
    n_levels = 1;
    for (int i = 0; i < n_steps; ++i) {
      int lv = st[i].op >= 0 ? 1 : 0;
      for (int q = 0; q < 2; ++q)
        if (st[i].in[q] >= 0 && st[st[i].in[q]].level + 1 > lv) lv = st[st[i].in[q]].level + 1;
      // a set or a mask that is written twice: in the order of the ops, and after it was loaded
      for (int j = 0; j < i && st[i].op >= 0; ++j)
        if (st[j].ptr == st[i].ptr || (st[j].op >= 0 && ops[st[j].op].out.flags == ops[st[i].op].out.flags))
          if (st[j].level + 1 > lv) lv = st[j].level + 1;
      if (serial) lv = i + (i > 0 || st[i].op >= 0 ? 1 : 0);
      else
        while (count[lv] >= (resident ? PLAN_LEVEL_STEPS : PLAN_WRITE_WAVES)) ++lv;
      ++count[lv];
      st[i].level = lv;
      if (lv + 1 > n_levels) n_levels = lv + 1;
    }
    for (int i = 0; i < n_steps; ++i) st[i].last = st[i].op < 0 ? st[i].level : resident ? n_levels : st[i].level + 1;
    for (int i = 0; i < n_steps; ++i)
      for (int q = 0; q < 2; ++q)
        if (st[i].in[q] >= 0 && st[i].level > st[st[i].in[q]].last) st[st[i].in[q]].last = st[i].level;
  }

  // LDS: an allocation per bitmap, held from its level to its last reader's (both included).  A union (the 1x1
  // footprint of two masks) is a word-by-word OR and may overwrite an input that nothing else reads in its level or
  // later -- the writing waves of the level before are through with it if it is at least two levels old.
  void place(const mie_plan_op* ops) {
    n_rec = 0;
    int order[MAX];              // steps by level
    int no = 0;
    for (int lv = 0; lv < n_levels; ++lv)
      for (int i = 0; i < n_steps; ++i)
        if (st[i].level == lv) order[no++] = i;
    for (int oi = 0; oi < no; ++oi) {
      Step& s = st[order[oi]];
      s.rec = -1;
      if (s.op >= 0 && s.in[0] >= 0 && s.in[1] >= 0) {
        const mie_plan_op& op = ops[s.op];
        if (op.foot == MIE_FOOT_CONV && s.k == 1 && op.stride == 1 && op.pad == 0) {
          for (int q = 1; q >= 0 && s.rec < 0; --q) {
            const Step& m = st[s.in[q]];
            bool alone = m.words == s.words && m.last == s.level && m.level <= s.level - 2 && s.in[0] != s.in[1];
            for (int j = 0; j < n_steps && alone; ++j)
              if (&st[j] != &s && st[j].level == s.level && (st[j].in[0] == s.in[q] || st[j].in[1] == s.in[q])) alone = false;
            if (!alone || rec[m.rec].rel != s.level) continue;      // (rel: the memory was handed to another union already)
            s.rec = m.rec;
            rec[s.rec].rel = s.last;
          }
        }
      }
      if (s.rec < 0) {
        s.rec = n_rec;
        rec[n_rec++] = {s.words, 0, s.level, s.last};
      }
    }
    // two ways of packing, the tighter one counts: in order of birth, and largest first; each allocation at the lowest
    // offset where it meets none whose lifetime overlaps
    long long best[MAX];
    top = -1;
    for (int way = 0; way < 2; ++way) {
      int by[MAX];
      for (int i = 0; i < n_rec; ++i) by[i] = i;
      for (int i = 1; way == 1 && i < n_rec; ++i)
        for (int j = i; j > 0 && rec[by[j]].words > rec[by[j - 1]].words; --j) {
          const int t = by[j]; by[j] = by[j - 1]; by[j - 1] = t;
        }
      long long t = 0;
      for (int oi = 0; oi < n_rec; ++oi) {
        Alloc& r = rec[by[oi]];
        long long off = 0;
        for (bool moved = true; moved;) {
          moved = false;
          for (int oj = 0; oj < oi; ++oj) {
            const Alloc& q = rec[by[oj]];
            if (r.born <= q.rel && q.born <= r.rel && off < q.off + q.words && q.off < off + r.words) {
              off = q.off + q.words;
              moved = true;
            }
          }
        }
        r.off = off;
        if (off + r.words > t) t = off + r.words;
      }
      if (top < 0 || t < top) {
        top = t;
        for (int i = 0; i < n_rec; ++i) best[i] = rec[i].off;
      }
    }
    for (int i = 0; i < n_rec; ++i) rec[i].off = best[i];
  }
};

// `total` waves for the steps of a level by their weights: at least one each, none more than it has work for.
void plan_deal(int total, int n, const long long* weight, const int* most, int* first, int* count) {
  long long sum = 0;
  for (int i = 0; i < n; ++i) sum += weight[i];
  int used = 0;
  for (int i = 0; i < n; ++i) {
    int c = (int)(weight[i] * total / (sum > 0 ? sum : 1));
    c = c < 1 ? 1 : c;
    c = c > most[i] ? most[i] : c;
    count[i] = c;
    used += c;
  }
  while (used > total) {          // the minimum of one each went beyond: from the largest
    int b = 0;
    for (int i = 1; i < n; ++i) b = count[i] > count[b] ? i : b;
    --count[b];
    --used;
  }
  for (bool more = true; more && used < total;) {
    more = false;
    int b = -1;
    for (int i = 0; i < n; ++i)
      if (count[i] < most[i] && (b < 0 || weight[i] * count[b] > weight[b] * count[i])) b = i;
    if (b >= 0) { ++count[b]; ++used; more = true; }
  }
  for (int i = 0, at = 0; i < n; ++i) { first[i] = at; at += count[i]; }
}

}  // namespace

namespace {
int build_mask_plan(const char* who, const mie_plan_op* ops, int n_ops, int wg_cap, void* stream);
}

extern "C" int mie_build_mask_plan(const mie_plan_op* ops, int n_ops, void* stream) {
  return build_mask_plan("mie_build_mask_plan", ops, n_ops, 0, stream);
}

extern "C" int mie_build_mask_plan_wgs(const mie_plan_op* ops, int n_ops, int max_workgroups, void* stream) {
  const char* who = "mie_build_mask_plan_wgs";
  mie_clear_error();
  MIE_REQUIRE(max_workgroups > 0, MIE_ERR_INVALID_ARG, "%s: max_workgroups %d", who, max_workgroups);
  return build_mask_plan(who, ops, n_ops, max_workgroups, stream);
}

namespace {
int build_mask_plan(const char* who, const mie_plan_op* ops, int n_ops, int wg_cap, void* stream) {
  mie_clear_error();
  MIE_REQUIRE(ops != nullptr && n_ops > 0, MIE_ERR_INVALID_ARG, "%s: no ops", who);
  MIE_REQUIRE(n_ops <= MIE_PLAN_MAX_STEPS, MIE_ERR_CAPACITY, "%s: %d ops, at most %d per call", who, n_ops, MIE_PLAN_MAX_STEPS);
  const int n = ops[0].out.n;
  PlanHost ph;
  long long total_chunks = 0, max_pixels = 0;
  bool owned = n == 1;            // one launch: no set with more tiles than a workgroup ranks, none twice
  bool reread = false;            // an op overwrites a mask that the plan also loads from memory
  for (int i = 0; i < n_ops; ++i) {
    const mie_plan_op& op = ops[i];
    int rc = mie_check_tileset(&op.out, who);
    if (rc != MIE_OK) return rc;
    MIE_REQUIRE(op.out.n == n, MIE_ERR_INVALID_ARG, "%s: op %d has batch size %d, op 0 has %d", who, i, op.out.n, n);
    MIE_REQUIRE(op.h_in > 0 && op.w_in > 0, MIE_ERR_INVALID_ARG, "%s: op %d: input size (%d,%d) must be positive", who, i,
                op.h_in, op.w_in);
    MIE_REQUIRE(op.in_mask != nullptr || op.in_mask2 == nullptr, MIE_ERR_INVALID_ARG, "%s: op %d: in_mask2 given without in_mask", who, i);
    MIE_REQUIRE((long long)n * op.h_in * op.w_in < 0x7fffffffLL, MIE_ERR_CAPACITY, "%s: op %d: more than 2^31 input pixels", who, i);
    MIE_REQUIRE(op.w_in <= 2048 && op.out.w <= 2048 && (long long)op.h_in * op.w_in <= (1 << 20) &&
                    (long long)op.out.h * op.out.w <= (1 << 20),
                MIE_ERR_CAPACITY, "%s: op %d: planes of up to 2048 pixels per row and 2^20 pixels per sample (use mie_build_mask_tiles)", who, i);
    const int k = op.k, st = op.stride, pad = op.pad;
    if (op.foot == MIE_FOOT_CONV) {
      MIE_REQUIRE(k >= 1 && k <= 15 && (st == 1 || st == 2) && pad >= 0 && pad < 16, MIE_ERR_UNSUPPORTED,
                  "%s: op %d: conv footprint k=%d stride=%d pad=%d (strides 1 and 2 only)", who, i, k, st, pad);
      const int ho = (op.h_in + 2 * pad - k) / st + 1, wo = (op.w_in + 2 * pad - k) / st + 1;
      MIE_REQUIRE(op.h_in + 2 * pad >= k && op.w_in + 2 * pad >= k && ho == op.out.h && wo == op.out.w, MIE_ERR_INVALID_ARG,
                  "%s: op %d: conv output of (%d,%d) k=%d s=%d p=%d is (%d,%d), tile set is (%d,%d)", who, i, op.h_in, op.w_in, k,
                  st, pad, ho, wo, op.out.h, op.out.w);
    } else if (op.foot == MIE_FOOT_UP2X) {
      MIE_REQUIRE(op.out.h == 2 * op.h_in && op.out.w == 2 * op.w_in, MIE_ERR_INVALID_ARG,
                  "%s: op %d: up2x of (%d,%d) is not (%d,%d)", who, i, op.h_in, op.w_in, op.out.h, op.out.w);
    } else if (op.foot == MIE_FOOT_TCONV) {
      MIE_REQUIRE(k >= 1 && k <= 15 && st == 2 && pad >= 0 && pad < 16, MIE_ERR_UNSUPPORTED,
                  "%s: op %d: tconv footprint k=%d stride=%d pad=%d (stride 2 only)", who, i, k, st, pad);
      const int hmin = (op.h_in - 1) * st - 2 * pad + k, wmin = (op.w_in - 1) * st - 2 * pad + k;
      MIE_REQUIRE(op.out.h >= hmin && op.out.h < hmin + st && op.out.w >= wmin && op.out.w < wmin + st, MIE_ERR_INVALID_ARG,
                  "%s: op %d: tconv output (%d,%d) not in [(%d,%d), +stride)", who, i, op.out.h, op.out.w, hmin, wmin);
    } else {
      MIE_REQUIRE(false, MIE_ERR_UNSUPPORTED, "%s: op %d: unknown footprint %d", who, i, op.foot);
    }
    // (as in mie_build_mask_tiles: only the identity footprint may be built in place)
    const bool identity = op.foot == MIE_FOOT_CONV && k == 1 && st == 1 && pad == 0;
    MIE_REQUIRE(identity || ((const uint8_t*)op.out.pixmask != op.in_mask && (const uint8_t*)op.out.pixmask != op.in_mask2),
                MIE_ERR_INVALID_ARG, "%s: op %d: out.pixmask aliases an input mask (allowed for the 1x1 stride-1 footprint only)", who, i);
    // inputs: the mask an earlier op of this plan left at this address last; any other is loaded from memory, once
    int in[2] = {-1, -1};
    const uint8_t* ins[2] = {op.in_mask, op.in_mask2};
    for (int q = 0; q < 2; ++q) {
      if (ins[q] == nullptr) continue;
      for (int j = ph.n_steps - 1; j >= 0 && in[q] < 0; --j)
        if (ph.st[j].ptr == ins[q]) in[q] = j;
      if (in[q] < 0) {
        MIE_REQUIRE(ph.n_steps < MIE_PLAN_MAX_STEPS, MIE_ERR_CAPACITY,
                    "%s: more than %d steps (ops plus masks loaded from memory); build the plan in parts", who, MIE_PLAN_MAX_STEPS);
        PlanHost::Step& ld = ph.st[ph.n_steps];
        ld = {-1, {-1, -1}, 0, {-1, -1}, ins[q], op.h_in, op.w_in, (long long)op.h_in * ((op.w_in + 31) / 32), 0, 0, -1};
        in[q] = ph.n_steps++;
        for (int j = i; j < n_ops; ++j) reread |= (const uint8_t*)ops[j].out.pixmask == ins[q];
      }
      const PlanHost::Step& m = ph.st[in[q]];
      MIE_REQUIRE(m.h == op.h_in && m.w == op.w_in, MIE_ERR_INVALID_ARG,
                  "%s: op %d reads a mask of (%d,%d) as (%d,%d)", who, i, m.h, m.w, op.h_in, op.w_in);
    }
    MIE_REQUIRE(ph.n_steps < MIE_PLAN_MAX_STEPS, MIE_ERR_CAPACITY,
                "%s: more than %d steps (ops plus masks loaded from memory); build the plan in parts", who, MIE_PLAN_MAX_STEPS);
    PlanHost::Step& ft = ph.st[ph.n_steps++];
    ft = {i, {in[0], in[1]}, k, {in[0], in[1]}, op.out.pixmask, op.out.h, op.out.w, (long long)op.out.h * ((op.out.w + 31) / 32), 0, 0, -1};
    const int cap = mie_tile_capacity(n, op.out.h, op.out.w);
    total_chunks += mie_div_up(cap, COMPACT_CHUNK);
    if ((long long)op.out.h * op.out.w > max_pixels) max_pixels = (long long)op.out.h * op.out.w;
    owned = owned && cap <= PLAN_OWNED_TILES;
    for (int j = 0; j < i; ++j) owned = owned && ops[j].out.flags != op.out.flags;
  }
  // workgroups per sample: a slice of the largest plane's stores each, and with one sample a set or two to rank
  long long shares = (max_pixels + PLAN_PIXELS_PER_SHARE - 1) / PLAN_PIXELS_PER_SHARE;
  // Every workgroup walks the whole chain of its sample (and loads every mask that comes from memory): with a batch of
  // samples there are workgroups enough without many per sample, and more than one per CU would only queue (a
  // workgroup of a large plane takes most of a CU's LDS).
  static const int max_wgs = [] { const char* e = getenv("MIE_PLAN_WGS"); return e ? atoi(e) : 256; }();      // tuning knob
  const int wgs = (wg_cap > 0 && wg_cap < max_wgs) ? wg_cap : max_wgs;     // a caller's cap: the plan runs beside other kernels
  if (shares * n > wgs) shares = wgs / n > 0 ? wgs / n : 1;
  MIE_REQUIRE(shares <= PLAN_MAX_SHARES, MIE_ERR_CAPACITY,
              "%s: a plane of %lld pixels per sample is beyond the plan's %d workgroups per sample; use "
              "mie_build_mask_tiles", who, max_pixels, PLAN_MAX_SHARES);
  if (reread) shares = 1;         // a workgroup that lags must not load what another has already overwritten
  const long long shares_in_slices = shares;
  // (a plan held to some workgroups runs beside other kernels: no more of them than its stores need)
  if (owned && !reread && wg_cap == 0 && shares < n_ops) shares = n_ops < wgs ? n_ops : wgs;
  if (shares > PLAN_MAX_SHARES) shares = PLAN_MAX_SHARES;
  int limit = 0;
  int rc = plan_lds_limit(&limit, who);
  if (rc != MIE_OK) return rc;
  PlanArgs a;
  long long lds_words = 0;
  // The first form that fits: everything resident; bitmaps dropped after their last reader; step by step.
  for (int form = 0; form < 3; ++form) {
    const bool resident = form == 0, serial = form == 2;
    owned = owned && resident;
    if (!owned) shares = shares_in_slices;
    ph.as_given(ops);
    if (!serial) ph.widen(ops);
    ph.schedule(serial, resident, ops);
    ph.place(ops);
    memset(&a, 0, sizeof(a));
    memset(a.task, PLAN_IDLE, sizeof(a.task));
    memset(a.head, PLAN_IDLE, sizeof(a.head));
    a.n_steps = ph.n_steps;
    a.n_levels = ph.n_levels;
    a.resident = resident ? 1 : 0;
    a.owned = owned ? 1 : 0;
    const int compute_waves = resident ? PLAN_WAVES : PLAN_COMPUTE_WAVES;
    // flags: who owns which set (largest first, to whoever has least), or how much of each a workgroup writes
    int own[PlanHost::MAX];
    long long fl[PlanHost::MAX], flag_bytes = 0;
    auto set_tiles = [&](int i) { return (long long)mie_div_up(ph.st[i].h, MIE_TILE) * mie_div_up(ph.st[i].w, MIE_TILE); };
    int owner[PlanHost::MAX];
    for (int i = 0; i < ph.n_steps; ++i) {
      if (ph.st[i].op < 0) continue;
      own[i] = (int)((set_tiles(i) + shares - 1) / shares);
      fl[i] = flag_bytes;
      if (!resident) flag_bytes += own[i];
    }
    if (owned) {
      long long load[PLAN_MAX_SHARES] = {0};
      bool done[PlanHost::MAX] = {false};
      for (int c = 0; c < n_ops; ++c) {
        int b = -1, to = 0;
        for (int i = 0; i < ph.n_steps; ++i)
          if (ph.st[i].op >= 0 && !done[i] && (b < 0 || set_tiles(i) > set_tiles(b))) b = i;
        for (int s = 1; s < shares; ++s) to = load[s] < load[to] ? s : to;
        owner[b] = to;
        fl[b] = load[to];
        load[to] += set_tiles(b);
        done[b] = true;
        flag_bytes = load[to] > flag_bytes ? load[to] : flag_bytes;
      }
    }
    flag_bytes = (flag_bytes + 15) / 16 * 16;
    // LDS: steps, task table, zeros and wave totals, tile bits, bitmaps, and the words a load right of the last row reaches
    a.zero_off = ph.n_steps * PS_WORDS + (ph.n_levels + 2) * (PLAN_WAVES / 4);
    a.flag_off = a.zero_off + PLAN_ZERO_WORDS + 2 * PLAN_WAVES;
    const long long base = a.flag_off + flag_bytes / 4;
    lds_words = base + ph.top + 4;
    int at = 0;                   // a step's place in the level order
    for (int lv = 0; lv < ph.n_levels; ++lv) {
      int id[PLAN_LEVEL_STEPS], ns = 0, most[PLAN_LEVEL_STEPS], cf[PLAN_LEVEL_STEPS], cn[PLAN_LEVEL_STEPS], wf[PLAN_LEVEL_STEPS], wn[PLAN_LEVEL_STEPS];
      long long weight[PLAN_LEVEL_STEPS];
      if (lv == ph.n_levels - 1) a.first_last = at;
      for (int i = 0; i < ph.n_steps; ++i)
        if (ph.st[i].level == lv) id[ns++] = i;
      for (int q = 0; q < ns; ++q) {
        weight[q] = ph.st[id[q]].words * ph.cost(id[q], ops);
        most[q] = (int)(ph.st[id[q]].words + 63) / 64;
        if (most[q] > (lv == 0 ? PLAN_WAVES : compute_waves)) most[q] = lv == 0 ? PLAN_WAVES : compute_waves;
      }
      // level 0 holds masks from memory only: by all waves, before the chain starts
      if (lv == 0) a.n_loads = ns;
      plan_deal(lv == 0 ? PLAN_WAVES : compute_waves, ns, weight, most, cf, cn);
      for (int q = 0; q < ns; ++q) most[q] = PLAN_WRITE_WAVES, wf[q] = wn[q] = 0;
      if (!resident) plan_deal(PLAN_WRITE_WAVES, ns, weight, most, wf, wn);
      for (int q = 0; q < ns; ++q) {
        const int i = id[q];
        const PlanHost::Step& s = ph.st[i];
        if (owned && s.op >= 0) {        // in front of its owner's list
          own[i] = a.head[owner[i]];
          a.head[owner[i]] = (uint8_t)at;
        }
        wf[q] += PLAN_COMPUTE_WAVES;
        for (int w = cf[q]; w < cf[q] + cn[q]; ++w) a.task[lv * PLAN_WAVES + w] = (uint8_t)at;
        if (!resident && s.op >= 0 && lv + 1 < ph.n_levels)
          for (int w = wf[q]; w < wf[q] + wn[q]; ++w) a.task[(lv + 1) * PLAN_WAVES + w] = (uint8_t)at;
        uint32_t* p = a.st + at * PS_WORDS;
        ++at;
        auto offset = [&](int j) { return (uint32_t)(base + ph.rec[ph.st[j].rec].off); };
        auto pointer = [&](int word, const void* v) {
          const unsigned long long b = reinterpret_cast<unsigned long long>(v);
          p[word] = (uint32_t)b;
          p[word + 1] = (uint32_t)(b >> 32);
        };
        if (lds_words > 0xfff0) continue;       // refused below; the offsets would not fit their fields
        int key = PLAN_KEY_GENERIC, unit = 0, h_in = s.h, w_in = s.w;
        if (mie_aligned(s.ptr, 16) && s.w % 16 == 0) unit = 2;        // rows of whole 16-byte (4-byte) groups, on such boundaries
        else if (mie_aligned(s.ptr, 4) && s.w % 4 == 0) unit = 1;
        p[PS_IN] = (s.in[0] < 0 ? PLAN_IN_NONE : offset(s.in[0])) | (s.in[1] < 0 ? PLAN_IN_NONE : offset(s.in[1])) << 16;
        if (s.op >= 0) {
          const mie_plan_op& op = ops[s.op];
          h_in = s.up ? s.h / 2 : op.h_in;
          w_in = s.up ? s.w / 2 : op.w_in;
          // the specialised forms have kernel size, stride and the padding k / 2 built in
          if (op.in_mask == nullptr) key = PLAN_KEY_ALL;
          else if (op.foot == MIE_FOOT_UP2X) key = PLAN_KEY_UP;
          else if (s.up) key = s.k == 3 ? PLAN_KEY_UP3 : PLAN_KEY_UP5;
          else if (op.pad == op.k / 2) {
            const int k = s.k;
            if (op.foot == MIE_FOOT_CONV && op.stride == 1 && (k & 1) && k <= PLAN_MAX_K1) key = PLAN_KEY_C11 + k / 2;
            if (op.foot == MIE_FOOT_CONV && op.stride == 2 && (k & 1) && k >= 3 && k <= PLAN_MAX_K2) key = PLAN_KEY_C32 + k / 2 - 1;
            if (op.foot == MIE_FOOT_TCONV) key = k == 3 ? PLAN_KEY_T32 : k == 5 ? PLAN_KEY_T52 : PLAN_KEY_GENERIC;
          }
          p[PS_GEOM] = (uint32_t)op.foot | (uint32_t)op.k << 8 | (uint32_t)op.stride << 16 | (uint32_t)op.pad << 24;
          p[PS_FL] = (uint32_t)fl[i];
          p[PS_OWN] = (uint32_t)own[i];
          pointer(PS_FLAGS, op.out.flags);
          pointer(PS_TILES, op.out.tiles);
          pointer(PS_STALE, op.out.stale);
          pointer(PS_COUNTS, op.out.counts);
        }
        p[PS_OUT_WIN] = offset(i) | (uint32_t)w_in << 16;
        p[PS_HIN] = (uint32_t)h_in;
        p[PS_HOUT] = (uint32_t)s.h;
        p[PS_WOUT_KEY] = (uint32_t)s.w | (uint32_t)key << 16 | (uint32_t)(s.op < 0 ? PLAN_KIND_LOAD : PLAN_KIND_FOOT) << 24 | (uint32_t)unit << 28;
        p[PS_MWORDS] = plan_magic(mie_div_up(s.w, 32));
        p[PS_MUNITS] = plan_magic(mie_div_up(s.w, 16));
        p[PS_MTILES] = plan_magic(mie_div_up(s.w, MIE_TILE));
        p[PS_UBASE] = (uint32_t)a.units;
        if (s.op >= 0) a.units += s.h * mie_div_up(s.w, 16);
        p[PS_WAVES] = (uint32_t)cf[q] | (uint32_t)cn[q] << 8 | (uint32_t)wf[q] << 16 | (uint32_t)wn[q] << 24;
        pointer(PS_PIX, s.ptr);
      }
    }
    if (lds_words * 4 <= limit) break;
  }
  rc = plan_lds_take(lds_words * 4, limit, who);
  if (rc != MIE_OK) return rc;
  hipLaunchKernelGGL(k_plan_bits, dim3((unsigned)shares, (unsigned)n), dim3(PLAN_THREADS), (size_t)lds_words * 4,
                     (hipStream_t)stream, a);
  rc = mie_check_launch(who);
  if (rc != MIE_OK || owned) return rc;
  PlanCompactArgs c;
  memset(&c, 0, sizeof(c));
  for (int i = 0; i < n_ops; ++i) {
    const mie_tileset& ts = ops[i].out;
    PlanCompactSet& st = c.set[c.n_sets];
    st.tiles = ts.tiles; st.stale = ts.stale; st.counts = ts.counts; st.flags = ts.flags;
    st.cap = mie_tile_capacity(ts.n, ts.h, ts.w);
    c.first_chunk[c.n_sets + 1] = c.first_chunk[c.n_sets] + mie_div_up(st.cap, COMPACT_CHUNK);
    ++c.n_sets;
  }
  hipLaunchKernelGGL(k_plan_compact, dim3((unsigned)total_chunks), dim3(COMPACT_THREADS), 0, (hipStream_t)stream, c);
  return mie_check_launch(who);
}
}  // namespace
