// Stride-2 transposed conv of a delta on the matrix cores (gfx950): kernel size K in {3, 5}, padding
// K/2, output exactly twice the input (output_padding 1) -- the decoder layer of the flow and depth
// networks (incr_modules/e2depth_incr.py:243-282).
//
// Sub-pixel decomposition.  Output row 2i + py receives input row i + dy through tap ky iff
// py == (ky - pad) mod 2, with dy = (py + pad - ky) / 2; the same holds for columns.  The four output
// phases (py, px) are therefore four ordinary stride-1 contractions over disjoint tap subsets of the
// same staged input: for K = 3 phase (0,0) has 1 tap, (0,1) and (1,0) two, (1,1) four -- 9 taps for
// 4 output pixels, where the zero-insertion form would multiply 36.  One workgroup takes an 8x8 block
// of INPUT positions (a 16x16 block of output pixels): M = 64 positions per phase, four accumulator sets,
// the input block plus halo staged once per channel chunk exactly as in the conv kernel
// (mie_conv_mfma_impl.h: same LDS layout, operand pairing, filter ring and k-split), each tap's MFMAs
// going to the accumulators of its phase.  No multiplication is wasted on inserted zeros.
//
// Tile sets.  `a.ts` is the output tile set (8x8 output tiles, MIE_FOOT_TCONV); the workgroups walk `pts`,
// the tile set of the 16x16 output blocks at input resolution (built from the output pixel mask with a 2x2
// stride-2 OR): a block is live when any of its four output tiles is.  A live block writes all its 256
// pixels (zeros where no input reaches, their reservoirs left alone), a stale block is zeroed, which covers every stale
// output tile.
// On planes of very few blocks the 3x3 form is another kernel, one launch (k_tconv_deep), for bf16 deltas and fp32 in three terms.
// Of the others, and of fp32 of very many channels, the chunks are split there over up to 8 workgroups that write partial sums to the workspace, and
// k_conv_split_finish (walking the OUTPUT tile set) adds them and runs the epilogue.
#include "mie_conv_mfma_impl.h"
#include <type_traits>

namespace {

__host__ __device__ constexpr int tc_phase(int k, int pad) { return (((k - pad) % 2) + 2) % 2; }
__host__ __device__ constexpr int tc_shift(int k, int pad) { return (tc_phase(k, pad) + pad - k) / 2; }   // numerator is even

// The six significant term products of a unit, the two pixel blocks interleaved (smallest terms first).
__device__ __forceinline__ void mma_tconv_x3(v16f (&acc)[2], const float4 (&A)[2][3], const float4 (&B)[3]) {
  mma_unit(acc[0], A[0][2], B[0], mie_bf16()); mma_unit(acc[1], A[1][2], B[0], mie_bf16());
  mma_unit(acc[0], A[0][1], B[1], mie_bf16()); mma_unit(acc[1], A[1][1], B[1], mie_bf16());
  mma_unit(acc[0], A[0][0], B[2], mie_bf16()); mma_unit(acc[1], A[1][0], B[2], mie_bf16());
  mma_unit(acc[0], A[0][1], B[0], mie_bf16()); mma_unit(acc[1], A[1][1], B[0], mie_bf16());
  mma_unit(acc[0], A[0][0], B[1], mie_bf16()); mma_unit(acc[1], A[1][0], B[1], mie_bf16());
  mma_unit(acc[0], A[0][0], B[0], mie_bf16()); mma_unit(acc[1], A[1][0], B[0], mie_bf16());
}

// X3 (fp32 deltas): the three-term bf16 form of k_conv_mfma -- staged values and weights as hi + mid + lo in bf16, six
// v_mfma_f32_32x32x16_bf16 products per multiply, fp32 accuracy; chunks of 64 channels (four units per tap, so that the
// k-split stays over whole sub-chunks and every tap's phase is known at compile time), three bf16 planes in LDS,
// single-buffered.  With the accumulators of four phases it needs 140-176 registers beside them: one workgroup per CU
// (forcing two makes it spill and costs 1 % of the EVFlowNet frame; as it is the form gains 1-2 % there).
// LEAD: with two more input channels (a.g_cpd with its mask a.g_cpm, filter rows a.g_cpres).  Kernels of up to 64 columns take them
// along by a branch; of 128 that costs registers where there are none (364 -> 408; bf16 128->128 from 2x120x160 96.9 us, with the
// branch 98.3, from 150x170 66.8, 68.1), and they are two forms (with the two channels 79.4, by the branch 81.0; of 64 columns a form of its
// own was slower, 27.3 -> 30.2).
// ARITH: 0 deltas as they are, 1 X3, 2 fp32 deltas in two fp16 terms (F2 of mie_conv_mfma_impl.h): leading products and cross products in
// accumulators of their own, 256 of them, which one wave a SIMD has room for (X3 adds all six to one, as it has no room for two in its
// 128-column form either).  All active, three terms -> two, us, and error against fp64: 64+64->64 from 160x160 38.1 -> 33.7, 1.97 -> 1.19e-7;
// 512->256 from 40x44 34 -> 28, 2.84 -> 1.49e-7; 5x5 128+64->64 from 66x88 29.0 -> 22.4, 2.71 -> 1.47e-7; 64+64->32 from 128x128, two chunks,
// bound by its trips to memory, 14.0 -> 13.7, 1.39 -> 1.07e-7.
template <typename T, int K, int WN, bool SPLIT, int ARITH = 0, bool LEAD = false>
__global__ __launch_bounds__(256, ARITH == 0 && WN <= 2 ? 2 : 1) void k_tconv_mfma(ConvArgsT<T> a, TileSetDev pts) {
  constexpr bool X3 = ARITH != 0, F2 = ARITH == 2;
  static_assert(!X3 || sizeof(T) == 4, "X3: fp32 deltas");
  constexpr bool ANY_LEAD = K == 3 && !SPLIT && (X3 || sizeof(T) == 2) && WN < 4;      // (the types that mie_tconv2x_lead_masked takes)
  using TL = std::conditional_t<X3, mie_bf16, T>;            // element type in LDS and on the matrix cores
  constexpr int PL = F2 ? 2 : X3 ? 3 : 1;                    // operand planes (terms per value)
  constexpr int GPS = X3 ? 2 : 1;                            // 16-byte global loads per staging slot
  constexpr int PAD = K / 2;
  constexpr int LO = (K == 5) ? 1 : 0;                       // halo above / left of the block (shifts reach -LO .. +1)
  constexpr int NBUF = X3 ? 1 : stage_buffers(1, (int)sizeof(T));
  constexpr int EPS = 16 / (int)sizeof(TL);
  constexpr int SUB = 2 * EPS;
  constexpr int WK = 4 / WN;
  constexpr int IT = 8 + LO + 1;
  constexpr int CC = X3 ? 64 : stage_channels(K, 1) * (4 / (int)sizeof(T));
  constexpr int LS = CC + EPS;
  constexpr int NPIX = IT * IT;
  constexpr int Q4 = CC / EPS;
  constexpr int NSLOT = NPIX * Q4;
  constexpr int NLD = (NSLOT + 255) / 256;
  constexpr int RP = row_pitch_dw(IT, LS * (int)sizeof(TL) / 4, 1) * 4 / (int)sizeof(TL);
  constexpr int STAGE = IT * RP;                             // elements per plane of a staging buffer
  constexpr int NQ = CC / SUB;
  static_assert(NQ % WK == 0, "the k-split is over whole sub-chunks");
  constexpr int NQW = NQ / WK;
  constexpr int UPC = K * K * NQW;
  constexpr int RING = (X3 && ring_size(UPC) > 6) ? ring_size(UPC, 3) : ring_size(UPC);
  constexpr int PD = RING - 1;
  constexpr int CO_BLK = 32 * WN;
  constexpr int RED = WK * 64 * CO_BLK;                      // the accumulators of one phase, parked for the epilogue
  constexpr int STAGE_F = (F2 ? 3 : NBUF * PL) * STAGE * (int)sizeof(TL) / 4;      // (F2: three planes for what does not fit)
  constexpr int SMEM = STAGE_F > RED ? STAGE_F : RED;
  static_assert(SMEM * 4 <= 65536, "LDS budget");
  static_assert(!SPLIT || WN == 1, "the split form is the 32-channel slab kernel");
  static_assert(!F2 || NBUF == 1, "two terms: one staging buffer");
  __shared__ __attribute__((aligned(16))) float smem[SMEM];
  __shared__ float s_f2[F2 ? 6 : 1];                         // F2: largest values of the waves' first slots; whether a group of a chunk does not fit
  TL* const sbuf = reinterpret_cast<TL*>(smem);

  int n, y0, x0;                                             // block origin in INPUT coordinates
  int bx = blockIdx.x + conv_args_entry_zero(a), by = blockIdx.y, bz = 0;
  if constexpr (SPLIT) split_order(a, bx, by, bz);
  const int tk = mie_pick_tile(pts, bx, n, y0, x0);
  if (tk == 0) return;
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int l32 = lane & 31, half = lane >> 5;
  const int wn = wave % WN, wk = wave / WN;
  const int co0 = by * CO_BLK;
  const int hout = 2 * a.h_in, wout = 2 * a.w_in;
  const int cout = a.cout;

  if (tk == 2) {                                             // stale block: zero this workgroup's slab of its 16x16 pixels
    if (SPLIT) return;                                       // (the finish kernel zeroes the stale output tiles)
    for (int idx = tid; idx < 64 * CO_BLK; idx += 256) {      // groups of four channels
      const int p = idx / (CO_BLK / 4), col = 4 * (idx - p * (CO_BLK / 4));
      const int oy = 2 * y0 + (p >> 4), ox = 2 * x0 + (p & 15);
      if (oy < hout && ox < wout)
        mie_st4(a.out, (((long long)n * hout + oy) * wout + ox) * cout + co0 + col, make_float4(0.f, 0.f, 0.f, 0.f));
    }
    return;
  }

  v16f acc[4][2], sm[F2 ? 4 : 1][2];
#pragma unroll
  for (int ph = 0; ph < 4; ++ph)
#pragma unroll
    for (int mb = 0; mb < 2; ++mb)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        acc[ph][mb][r] = 0.f;
        if (F2) sm[F2 ? ph : 0][mb][r] = 0.f;
      }
  // F2: the filter's scale and whether it fits, on their way from here on
  const long long weights = (long long)a.cin_total * (K * K) * cout;
  float filt_unscale = 1.f;
  float filt_form = 1.f;
  if constexpr (F2) {
    const float* const end = f2_filter_end(a.filt_mc, weights);
    filt_unscale = end[0];
    filt_form = end[1] - end[2];
  }

  // ---- staging plan (as in k_conv_mfma, stride 1) ------------------------------------------------------
  const int iy0 = y0 - LO, ix0 = x0 - LO;
  int st_po[NLD], st_lds[NLD], st_c4[NLD];
  unsigned inb = 0u;
#pragma unroll
  for (int i = 0; i < NLD; ++i) {
    const int slot = tid + 256 * i;
    const int pix = slot / Q4, q4 = slot - pix * Q4;
    const int lrow = pix / IT;
    st_lds[i] = lrow * RP + (pix - lrow * IT) * LS + EPS * q4;
    st_c4[i] = EPS * q4;
    st_po[i] = 0;
    if (slot < NSLOT) {
      const int iy = iy0 + lrow, ix = ix0 + (pix - lrow * IT);
      if (iy >= 0 && iy < a.h_in && ix >= 0 && ix < a.w_in) {
        st_po[i] = (n * a.h_in + iy) * a.w_in + ix;
        inb |= 1u << i;
      }
    }
  }
  const uint8_t* const x2m = a.x2 != nullptr ? a.x2m : nullptr;
  unsigned b1[NLD], b2[NLD];
  mie_mask_ask(a.xm, a.filt_mc, st_po, b1);
  mie_mask_ask(x2m, a.filt_mc, st_po, b2);
  mie_mask_asked();
  const unsigned ok1 = mie_mask_take(a.xm, b1, inb), ok2 = mie_mask_take(x2m, b2, a.x2 != nullptr ? inb : 0u);
  const int nch1 = a.c1 / CC;
  const int nch = nch1 + (a.x2 != nullptr ? a.c2 / CC : 0);

  float4 st_reg[NLD][GPS];
  F2Groups groups;
  auto stage_load = [&](int c) __attribute__((always_inline)) {
    const bool second = c >= nch1;
    const T* xin = second ? a.x2 : a.x;
    const int cs = second ? a.c2 : a.c1;
    const int ci0 = (second ? c - nch1 : c) * CC;
    const unsigned ok = second ? ok2 : ok1;
    const T* dummy = a.filt_mc;          // masked lanes read one cache-resident address: loads stay unconditional
#pragma unroll
    for (int i = 0; i < NLD; ++i) {
      const bool okb = (ok >> i) & 1u;
      const T* p = xin + (long long)st_po[i] * cs + ci0 + st_c4[i];
      p = okb ? p : dummy;
#pragma unroll
      for (int g = 0; g < GPS; ++g) {
        float4 v = *reinterpret_cast<const float4*>(p + 4 * g);
        v.x = okb ? v.x : 0.f; v.y = okb ? v.y : 0.f; v.z = okb ? v.z : 0.f; v.w = okb ? v.w : 0.f;
        st_reg[i][g] = v;
      }
    }
  };
  auto slots_max = [&](const float4 (&regs)[NLD][GPS]) __attribute__((always_inline)) {
    float m = 0.f;
#pragma unroll
    for (int i = 0; i < NLD; ++i) {
      const float4 u = regs[i][0], v = regs[i][GPS - 1];
      const float f[8] = {u.x, u.y, u.z, u.w, v.x, v.y, v.z, v.w};
      m = __builtin_elementwise_maximum(m, f2_amax8(f));
    }
    return m;
  };
  // (terms: 1 in terms, F2: 2 in three of them, 0 as it is)
  auto stage_store = [&](int buf, auto terms) __attribute__((always_inline)) {
    TL* dst = sbuf + buf * (PL * STAGE);
#pragma unroll
    for (int i = 0; i < NLD; ++i)
      if (tid + 256 * i < NSLOT) {
        if constexpr (F2) {
          const float4 u = st_reg[i][0], v = st_reg[i][GPS - 1];
          const float f[8] = {u.x, u.y, u.z, u.w, v.x, v.y, v.z, v.w};
          constexpr int FORM = decltype(terms)::value;
          float4 pl[FORM == 2 ? 3 : 2];
          pl[0] = u; pl[1] = v;
          if constexpr (FORM == 1) groups.terms(f, pl);
          else groups.note(f);
          if constexpr (FORM == 2) split3(f, pl);
#pragma unroll
          for (int q = 0; q < (FORM == 2 ? 3 : 2); ++q) *reinterpret_cast<float4*>(dst + q * STAGE + st_lds[i]) = pl[q];
        } else if constexpr (X3) {
          const float f[8] = {st_reg[i][0].x, st_reg[i][0].y, st_reg[i][0].z, st_reg[i][0].w,
                              st_reg[i][1].x, st_reg[i][1].y, st_reg[i][1].z, st_reg[i][1].w};
          float4 pl[3];
          split3(f, pl);
#pragma unroll
          for (int q = 0; q < 3; ++q) *reinterpret_cast<float4*>(dst + q * STAGE + st_lds[i]) = pl[q];
        } else {
          *reinterpret_cast<float4*>(dst + st_lds[i]) = st_reg[i][0];
        }
      }
  };

  // ---- operand addressing --------------------------------------------------------------------------------
  const int q0w = wk * NQW;
  const int cob0 = co0 + wn * 32;
  const int b_lane = (half * cout + l32) * EPS;
  int a_lane[2];
#pragma unroll
  for (int mb = 0; mb < 2; ++mb) {
    const int p = mb * 32 + l32;
    a_lane[mb] = (p >> 3) * RP + (p & 7) * LS + SUB * q0w + EPS * half;
  }
  auto chunk_b = [&](int c) -> const TL* {
    const bool second = c >= nch1;
    const int ci0 = (second ? c - nch1 : c) * CC;
    const int fb = second ? a.c1 : 0;
    return reinterpret_cast<const TL*>(a.filt_mc) + ((long long)((fb + ci0) / SUB + q0w) * (K * K) * (PL * 2) * cout + cob0) * EPS;
  };
  float4 bring[RING][PL];
  auto load_b = [&](const TL* ub, int unit, float4 (&bv)[PL]) __attribute__((always_inline)) {
    const int tap = unit / NQW, qi = unit % NQW;
#pragma unroll
    for (int q = 0; q < PL; ++q)
      bv[q] = *reinterpret_cast<const float4*>(ub + ((long long)(((qi * (K * K) + tap) * PL + q) * 2) * cout) * EPS + b_lane);
  };

  const int c_lo = SPLIT ? bz * nch >> a.xcd_fs : 0;
  const int c_hi = SPLIT ? (bz + 1) * nch >> a.xcd_fs : nch;
  const TL* ub_cur = chunk_b(c_lo);
  const TL* ub_next = ub_cur;
  const auto in_terms = std::integral_constant<int, 1>();
  int c_end = c_hi;                         // F2: where the contraction in two terms ends: in front of the first chunk that does not fit
  auto note_misfit = [&]() __attribute__((always_inline)) {
    if constexpr (F2) {
      s_f2[groups.misfit() ? 4 : 5] = 1.f;      // (without a branch)
    }
  };
  // (asked behind the barrier and looked at where the chunk begins; two barriers a chunk: nobody notes the next one before)
  float stop = 0.f;
  auto ask_stop = [&]() __attribute__((always_inline)) {
    if constexpr (F2) stop = s_f2[4];
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
  const bool both = F2 && c_lo < nch1 && nch1 < c_hi;      // (F2: the scale is for both inputs)
  float4 st_two[F2 ? NLD : 1][GPS];
  if constexpr (F2) {
    stage_load(both ? nch1 : c_lo);
#pragma unroll
    for (int i = 0; i < NLD; ++i)
#pragma unroll
      for (int g = 0; g < GPS; ++g) st_two[i][g] = st_reg[i][g];
  }
  stage_load(c_lo);
#pragma unroll
  for (int i = 0; i < (PD > 0 ? PD : 1); ++i) load_b(ub_cur, i, bring[i % RING]);
  if constexpr (F2) {
    const float m = f2_wave_max(__builtin_elementwise_maximum(slots_max(st_two), slots_max(st_reg)));
    if (lane == 0) s_f2[wave] = m;
    if (tid == 0) s_f2[4] = 0.f;
    __syncthreads();
    groups.start(f2_scale(__int_as_float(__builtin_amdgcn_readfirstlane(
        __float_as_int(__builtin_elementwise_maximum(f2_max3(s_f2[0], s_f2[1], s_f2[2]), s_f2[3]))))));
  }
  stage_store(0, in_terms);
  note_misfit();
  __syncthreads();
  if (F2 && filt_form != 1.f) c_end = c_lo;
  ask_stop();

  for (int c = c_lo; c < c_end; ++c) {
    const bool more = c + 1 < c_hi;
    const int cn = more ? c + 1 : c;
    ub_next = chunk_b(cn);
    stage_load(cn);
    const TL* sin = sbuf + ((c - c_lo) % NBUF) * (PL * STAGE);
    float4 av[2][2][PL];
    auto load_a = [&](int unit, float4 (&dst)[2][PL]) {
      const int tap = unit / NQW, qi = unit % NQW;
      const int ky = tap / K, kx = tap - ky * K;
      const int dy = tc_shift(ky, PAD) + LO, dx = tc_shift(kx, PAD) + LO;
#pragma unroll
      for (int mb = 0; mb < 2; ++mb)
#pragma unroll
        for (int q = 0; q < PL; ++q)
          dst[mb][q] = *reinterpret_cast<const float4*>(&sin[q * STAGE + a_lane[mb] + dy * RP + dx * LS + SUB * qi]);
    };
    load_a(0, av[0]);
    if (stops_at(c)) break;
#pragma unroll
    for (int i = 0; i < UPC; ++i) {
      if (PD > 0) {
        const int ip = i + PD;
        if (ip < UPC) load_b(ub_cur, ip, bring[ip % RING]);
        else load_b(ub_next, ip - UPC, bring[ip % RING]);
      }
      if (i + 1 < UPC) load_a(i + 1, av[(i + 1) & 1]);
      __builtin_amdgcn_sched_barrier(0);
      {
        const int tap = i / NQW;
        const int ky = tap / K, kx = tap - ky * K;
        const int ph = tc_phase(ky, PAD) * 2 + tc_phase(kx, PAD);      // compile-time after unrolling
        if constexpr (F2) {
          mma_unit2_f2(acc[ph][0], acc[ph][1], sm[ph][0], sm[ph][1], av[i & 1][0], av[i & 1][1], bring[i % RING]);
        } else if constexpr (X3) {
          mma_tconv_x3(acc[ph], av[i & 1], bring[i % RING]);
        } else {
#pragma unroll
          for (int mb = 0; mb < 2; ++mb) mma_unit(acc[ph][mb], av[i & 1][mb][0], bring[i % RING][0], T());
        }
      }
      __builtin_amdgcn_sched_barrier(0);
      if (PD == 0) load_b(ub_next, 0, bring[0]);
    }
    if (NBUF == 1) __syncthreads();
    if (more) stage_store((c - c_lo + 1) % NBUF, in_terms);
    note_misfit();
    __syncthreads();
    ask_stop();
    ub_cur = ub_next;
  }
  float c0 = 1.f;                      // F2: 1 / scales
  if constexpr (F2) {
    c0 = f2_unscale(groups.scale) * filt_unscale;      // exactly: powers of two, 2^-143 at the least but for sums of zeros
    // a chunk that does not fit: all of it in three bf16 terms of the input and of the fp32 copy of the filter behind the two.  (Not from
    // this chunk on, as in k_conv_mfma: adding up both sets of sums at its place costs the fast path registers.)  us where all fit | later
    // channels 1000 times larger | no chunk fits | three terms: 64+64->64 from 160x160 31.2 | 31.4 | 44 | 36.5, 512->256 from 40x44 26.3 | 49 | 41 | 32,
    // 5x5 128+64->64 from 66x88 20.6 | 20.6 | 33 | 26.5.
    if (__builtin_expect(c_end < c_hi, 0)) {
      auto plainly = [&](auto form) __attribute__((always_inline)) {
        constexpr bool THREE = decltype(form)::value == 2;
        constexpr int PA = THREE ? 3 : 2;
        for (int c = c_lo; c < c_hi; ++c) {
          const TL* ub = chunk_b(c) + 2 * weights;
          stage_load(c);
#pragma unroll
          for (int i = 0; i < RING - 1; ++i) load_b(ub, i, bring[i]);
          __syncthreads();
          stage_store(0, form);
          __syncthreads();
          float4 av[2][2][PA];
          auto read = [&](int i, float4 (&x)[2][PA]) __attribute__((always_inline)) {
            const int tap = i / NQW, ky = tap / K, kx = tap - ky * K;
            const int at = (tc_shift(ky, PAD) + LO) * RP + (tc_shift(kx, PAD) + LO) * LS + SUB * (i % NQW);
#pragma unroll
            for (int mb = 0; mb < 2; ++mb)
#pragma unroll
              for (int q = 0; q < PA; ++q) x[mb][q] = *reinterpret_cast<const float4*>(&sbuf[q * STAGE + a_lane[mb] + at]);
          };
          read(0, av[0]);
#pragma unroll
          for (int i = 0; i < UPC; ++i) {
            const int tap = i / NQW, ky = tap / K, kx = tap - ky * K, ph = tc_phase(ky, PAD) * 2 + tc_phase(kx, PAD);
            asm volatile("" : "+s"(ub));      // (or the units' addresses are all kept in registers)
            if (i + RING - 1 < UPC) load_b(ub, i + RING - 1, bring[(i + RING - 1) % RING]);
            if (i + 1 < UPC) read(i + 1, av[(i + 1) & 1]);
            __builtin_amdgcn_sched_barrier(0);
            const auto& x = av[i & 1];
            if constexpr (THREE) {
              float4 b3[3];
              split3_raw(bring[i % RING], b3);
              mma_tconv_x3(acc[ph], x, b3);
            } else {
#pragma unroll
              for (int q = 0; q < PL; ++q) mma_unit2(acc[ph][0], acc[ph][1], x[0][q], x[1][q], bring[i % RING][q], float());
            }
            __builtin_amdgcn_sched_barrier(0);
          }
        }
      };
      auto clear = [&](v16f (&v)[4][2]) __attribute__((always_inline)) {
#pragma unroll
        for (int ph = 0; ph < 4; ++ph)
#pragma unroll
          for (int mb = 0; mb < 2; ++mb)
#pragma unroll
            for (int r = 0; r < 16; ++r) v[ph][mb][r] = 0.f;
      };
      clear(acc);
      clear(sm);
      c0 = 1.f;
      if (filt_form >= 0.f) plainly(std::integral_constant<int, 2>());
      __syncthreads();
      if (tid == 0) s_f2[4] = filt_form < 0.f ? 1.f : 0.f;
      __syncthreads();
      if (groups.huge()) s_f2[4] = 1.f;
      __syncthreads();
      if (__builtin_amdgcn_readfirstlane(__float_as_int(s_f2[4])) != 0) {      // values that three bf16 terms do not hold: all of it on the fp32 instruction
        clear(acc);
        plainly(std::integral_constant<int, 0>());
        __syncthreads();
      }
    }
  }

  // ---- epilogue, one phase at a time -----------------------------------------------------------------------
  // acc[ph][mb][r] of this lane: input position p = 32*mb + 8*(r/4) + 4*half + r%4 of the block, i.e. output
  // pixel (2*(y0 + p/8) + py, 2*(x0 + p%8) + px), channel column wn*32 + lane%32 of the slab.
  // (a generic lambda called once per phase: the accumulator set is picked at compile time)
  auto epilogue = [&](auto PH) {
    constexpr int ph = decltype(PH)::value;
    constexpr int py = ph >> 1, px = ph & 1;
    // every wave parks the phase's accumulators in LDS; a thread then owns groups of four adjacent output channels
    // of a pixel (16-byte reads of the k-split partial sums, 16-byte reservoir accesses, 16- / 8-byte delta accesses)
    constexpr int QPP = CO_BLK / 4;
    constexpr int PER = 64 * QPP / 256;
    // (the output pixel mask of these groups is asked for before, and taken when the sums and the reservoir are there)
    const uint8_t* const live_m = a.refresh ? nullptr : a.ts.pixmask;
    unsigned live_b[PER];
    if constexpr (!SPLIT) {
      int at[PER];
#pragma unroll
      for (int i = 0; i < PER; ++i) {
        const int p = (tid + 256 * i) / QPP, iy = y0 + (p >> 3), ix = x0 + (p & 7);
        at[i] = iy < a.h_in && ix < a.w_in ? (n * hout + 2 * iy + py) * wout + 2 * ix + px : 0;
      }
      mie_mask_ask(live_m, a.filt_mc, at, live_b);
    }
    float* red = smem + wk * (64 * CO_BLK);
#pragma unroll
    for (int mb = 0; mb < 2; ++mb)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int p = mb * 32 + 8 * (r >> 2) + 4 * half + (r & 3);
        red[p * CO_BLK + wn * 32 + l32] = F2 ? fmaf(sm[F2 ? ph : 0][mb][r], c0 * (1.f / F2_STEP), acc[ph][mb][r] * c0) : acc[ph][mb][r];
      }
    __syncthreads();
    long long off[PER];
    int co[PER];
    bool ok[PER];
    float4 v[PER];
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const int idx = tid + 256 * i;
      const int p = idx / QPP, col = 4 * (idx - p * QPP);
      const int iy = y0 + (p >> 3), ix = x0 + (p & 7);
      ok[i] = iy < a.h_in && ix < a.w_in;
      off[i] = (((long long)n * hout + 2 * iy + py) * wout + 2 * ix + px) * cout + co0 + col;
      co[i] = co0 + col;
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
      for (int i = 0; i < PER; ++i)
        if (ok[i]) *reinterpret_cast<float4*>(plane + off[i]) = v[i];
    } else {
      float4 r0[PER], add[PER];
      conv_epilogue_load4<T, PER>(a, off, ok, r0, add);
      if constexpr (LEAD || ANY_LEAD) {
        // two more input channels, as in k_tconv_deep, in the epilogue's trip (a thread's groups have one column).  Against a launch
        // of their own and an addend, all active, fp32 / bf16: 64+64->32 from 128x128 29.0 -> 20.0 / 21.5 -> 14.7 us, from 2x240x320
        // 238 -> 187 / 111 -> 74, 128->128 from 132x176 115 -> 95 / 70 -> 47.
        if (LEAD || a.g_cpd != nullptr) {
          constexpr int NT = (1 + py) * (1 + px);
          int lat[NT * PER];
          float2 lx[NT * PER];
          float4 lf[NT][2];
          unsigned in = 0u, lb[NT * PER];
#pragma unroll
          for (int q = 0; q < NT; ++q) {
            const int r = px ? q >> 1 : q, c = px ? q & 1 : 0;
            const int ky = r != 0 ? 0 : py ? 2 : 1, kx = c != 0 ? 0 : px ? 2 : 1;
#pragma unroll
            for (int e = 0; e < 2; ++e) lf[q][e] = *reinterpret_cast<const float4*>(a.g_cpres + (long long)(9 * e + 3 * ky + kx) * cout + co[0]);
#pragma unroll
            for (int i = 0; i < PER; ++i) {
              const int p = (tid + 256 * i) / QPP, iy = y0 + (p >> 3) + r, ix = x0 + (p & 7) + c, at = q * PER + i;
              const bool k = ok[i] && iy < a.h_in && ix < a.w_in;
              lat[at] = k ? (n * a.h_in + iy) * a.w_in + ix : 0;
              in |= (k ? 1u : 0u) << at;
              if constexpr (sizeof(T) == 4) {
                lx[at] = *reinterpret_cast<const float2*>(a.g_cpd + 2LL * lat[at]);
              } else {
                const uint32_t b = *reinterpret_cast<const uint32_t*>(a.g_cpd + 2LL * lat[at]);
                lx[at] = make_float2(__uint_as_float(b << 16), __uint_as_float(b & 0xffff0000u));
              }
            }
          }
          mie_mask_ask(a.g_cpm, a.filt_mc, lat, lb);
          const unsigned kk = mie_mask_take(a.g_cpm, lb, in);
#pragma unroll
          for (int q = 0; q < NT; ++q)
#pragma unroll
            for (int i = 0; i < PER; ++i) {
              const int at = q * PER + i;
              const float u = (kk >> at) & 1u ? lx[at].x : 0.f, w = (kk >> at) & 1u ? lx[at].y : 0.f;
              v[i].x += u * lf[q][0].x + w * lf[q][1].x; v[i].y += u * lf[q][0].y + w * lf[q][1].y;
              v[i].z += u * lf[q][0].z + w * lf[q][1].z; v[i].w += u * lf[q][0].w + w * lf[q][1].w;
            }
        }
      }
      const unsigned live_bits = mie_mask_take(live_m, live_b, ~0u);
      bool live[PER];
#pragma unroll
      for (int i = 0; i < PER; ++i) live[i] = ((live_bits >> i) & 1u) != 0u;
      conv_epilogue_store4<T, PER>(a, off, co, ok, v, r0, add, live);
    }
    __syncthreads();                   // the next phase overwrites the parked accumulators
  };
  epilogue(std::integral_constant<int, 0>{});
  epilogue(std::integral_constant<int, 1>{});
  epilogue(std::integral_constant<int, 2>{});
  epilogue(std::integral_constant<int, 3>{});
}

template <typename T, int K, int ARITH = 0>
bool launch_tconv(const ConvArgsT<T>& a0, const TileSetDev& pts, hipStream_t st) {
  constexpr bool X3 = ARITH != 0;
  constexpr int CC = X3 ? 64 : stage_channels(K, 1) * (4 / (int)sizeof(T));
  if (a0.filt_mc == nullptr || a0.c1 % CC != 0 || a0.c2 % CC != 0 || a0.cout % 32 != 0) return false;
  constexpr bool DEEP = K == 3 && (X3 || sizeof(T) == 2);
  const unsigned cap_p = (unsigned)(pts.n * pts.tiles_y * pts.tiles_x);
  const int cout = a0.cout;
  // The one-launch form takes every launch of its types that could be split, but for fp32 of so many channels that the split contraction
  // makes up for its second launch.  One launch over split, three terms in both, 2 to 64 slabs: 1280 channels .89 to 1.05, 1408 .88 to 1.11, 1536 .92 to 1.17,
  // 2048 1.04 to 1.31; 128 slabs of four tiles or fewer, 1536 .97 to 1.18, 2048 1.05 to 1.26, of more .75 to .97 (bf16 of 2048: .5 to 1.0).
  const bool split = !DEEP || (X3 && a0.g_cpd == nullptr && a0.c1 + a0.c2 > 1408 && (long long)cap_p * (cout / 16) <= (cap_p <= 4 ? 128 : 64));
  ConvArgsT<T> a = ARITH == 2 ? f2_args(a0, K) : a0;
  a.xcd_fs = 0; a.xcd_m = 0;
  if constexpr (!DEEP || X3) {
    const unsigned cap_out = (unsigned)(a.ts.n * a.ts.tiles_y * a.ts.tiles_x);
    const long long groups = (long long)cap_p * (cout / 32);
    const int nch = (a.c1 + a.c2) / CC;
    if (split && a.ws != nullptr && !a.refresh && groups <= 128 && nch >= 4) {
      a.ws_plane = (long long)a.ts.n * a.ts.h * a.ts.w * cout;
      int parts = 1;
      while (2 * parts <= 8 && 2 * parts <= nch && groups * (2 * parts) <= 256 && (long long)(2 * parts) * a.ws_plane <= a.ws_floats)
        parts *= 2;
      if (parts >= 2) {
        a.xcd_fs = __builtin_ctz(parts);
        const std::lock_guard<std::mutex> pair(mie_split_launches());
        hipLaunchKernelGGL((k_tconv_mfma<T, K, 1, true, ARITH>), dim3(cout / 32 * parts, cap_p), dim3(256), 0, st, a, pts);
        unsigned ny = (unsigned)((1024 + cap_out - 1) / cap_out);
        if (ny > (unsigned)(cout / 16)) ny = (unsigned)(cout / 16);
        if (ny < 1) ny = 1;
        hipLaunchKernelGGL(k_conv_split_finish<T>, dim3(cap_out, ny), dim3(256), 0, st, a, parts);
        return true;
      }
    }
  }
  if (DEEP && mie_launch_tconv_deep(a0, pts, st)) return true;
  a.ws = nullptr;
  // (the 128-column kernel holds 4 phases x 2 blocks of accumulators and a four-column operand ring: in the three-term
  // form it would spill, so that form stops at 64 columns)
  if (!X3 && cout % 128 == 0 && (long long)cap_p * (cout / 128) >= 400) {
    if (DEEP && a.g_cpd != nullptr)
      hipLaunchKernelGGL((k_tconv_mfma<T, K, 4, false, 0, DEEP && !X3>), dim3(cap_p, cout / 128), dim3(256), 0, st, a, pts);
    else
      hipLaunchKernelGGL((k_tconv_mfma<T, K, 4, false>), dim3(cap_p, cout / 128), dim3(256), 0, st, a, pts);
  } else if (cout % 64 == 0 && (long long)cap_p * (cout / 64) >= 400) {
    hipLaunchKernelGGL((k_tconv_mfma<T, K, 2, false, ARITH>), dim3(cap_p, cout / 64), dim3(256), 0, st, a, pts);
  } else {
    hipLaunchKernelGGL((k_tconv_mfma<T, K, 1, false, ARITH>), dim3(cap_p, cout / 32), dim3(256), 0, st, a, pts);
  }
  return true;
}

template <typename T>
int tconv2x_impl(const char* who, const void* x, const uint8_t* xmask, int c1, const void* x2,
                 const uint8_t* x2mask, int c2, int h_in, int w_in, const float* filter, const void* filter_mc,
                 int cin_total, int k, int cout, const mie_tileset* out, const mie_tileset* blocks,
                 void* out_delta, const void* addend, float* reservoir, int act_kind, float slope, bool refresh,
                 const float* bias, void* workspace, long long workspace_bytes, void* stream, int x3 = 0,
                 const void* lead = nullptr, const uint8_t* lead_mask = nullptr, const float* lead_filter = nullptr) {
  int rc = mie_check_tileset(out, who);
  if (rc != MIE_OK) return rc;
  rc = mie_check_tileset(blocks, who);
  if (rc != MIE_OK) return rc;
  MIE_REQUIRE(x != nullptr && filter != nullptr && filter_mc != nullptr && out_delta != nullptr, MIE_ERR_INVALID_ARG,
              "%s: NULL pointer (x, filter, filter_mc and the output are required)", who);
  MIE_REQUIRE(c1 > 0 && c2 >= 0 && cout > 0 && h_in > 0 && w_in > 0 && (long long)c1 + c2 <= cin_total,
              MIE_ERR_INVALID_ARG, "%s: sizes out of range (c1=%d c2=%d cin_total=%d cout=%d h=%d w=%d)", who, c1, c2,
              cin_total, cout, h_in, w_in);
  MIE_REQUIRE((x2 != nullptr) == (c2 > 0) && (x2 != nullptr || x2mask == nullptr), MIE_ERR_INVALID_ARG,
              "%s: x2, c2 and x2mask must be given together", who);
  MIE_REQUIRE(k == 3 || k == 5, MIE_ERR_UNSUPPORTED, "%s: kernel size %d not implemented (3, 5)", who, k);
  MIE_REQUIRE(!x3 || sizeof(T) == 4, MIE_ERR_INVALID_ARG, "%s: MIE_DTYPE_F32_BF16X3 is a form of fp32 deltas", who);
  const int chunk = x3 ? 64 : 128 / (int)sizeof(T);
  MIE_REQUIRE(c1 % chunk == 0 && c2 % chunk == 0 && cout % 32 == 0 && cin_total % (x3 ? 16 : 32 / (int)sizeof(T)) == 0,
              MIE_ERR_UNSUPPORTED, "%s: needs c1, c2 %% %d == 0 and cout %% 32 == 0 (c1=%d c2=%d cout=%d)", who, chunk,
              c1, c2, cout);
  MIE_REQUIRE(out->h == 2 * h_in && out->w == 2 * w_in && blocks->h == h_in && blocks->w == w_in && blocks->n == out->n,
              MIE_ERR_INVALID_ARG, "%s: the output tile set must be (%d,%d) and the block tile set (%d,%d); got (%d,%d), (%d,%d)",
              who, 2 * h_in, 2 * w_in, h_in, w_in, out->h, out->w, blocks->h, blocks->w);
  MIE_REQUIRE((long long)out->n * out->h * out->w < 0x7fffffffLL && (long long)out->n * h_in * w_in * (c1 > c2 ? c1 : c2) < (1LL << 40),
              MIE_ERR_CAPACITY, "%s: tensor too large", who);
  MIE_REQUIRE(mie_aligned(x, 16) && mie_aligned(x2, 16) && mie_aligned(filter_mc, 16) && mie_aligned(out_delta, 16) &&
                  mie_aligned(addend, 16) && mie_aligned(reservoir, 16) && mie_aligned(bias, 4) && mie_aligned(workspace, 16),
              MIE_ERR_INVALID_ARG, "%s: buffers must be 16-byte aligned (bias: 4)", who);
  MIE_REQUIRE(act_kind >= MIE_ACT_NONE && act_kind <= MIE_ACT_TANH, MIE_ERR_UNSUPPORTED, "%s: unknown activation %d", who,
              act_kind);
  MIE_REQUIRE(refresh || reservoir != nullptr || act_kind == MIE_ACT_NONE, MIE_ERR_INVALID_ARG,
              "%s: activation %d needs a reservoir", who, act_kind);
  MIE_REQUIRE(addend == nullptr || addend != out_delta, MIE_ERR_INVALID_ARG, "%s: addend must not alias out_delta", who);
  MIE_REQUIRE(x != out_delta && (x2 == nullptr || x2 != out_delta), MIE_ERR_INVALID_ARG,
              "%s: x / x2 must not alias the output", who);
  MIE_REQUIRE(workspace_bytes >= 0 && (workspace != nullptr || workspace_bytes == 0), MIE_ERR_INVALID_ARG,
              "%s: workspace size without a workspace", who);
  MIE_REQUIRE(workspace == nullptr || (workspace != out_delta && workspace != (void*)reservoir && workspace != x && workspace != x2),
              MIE_ERR_INVALID_ARG, "%s: workspace must not alias an operand", who);
  ConvArgsT<T> a;
  a.x = (const T*)x; a.xm = xmask; a.c1 = c1; a.x2 = (const T*)x2; a.x2m = x2mask; a.c2 = c2;
  a.h_in = h_in; a.w_in = w_in; a.filt = filter; a.cin_total = cin_total; a.filt_mc = (const T*)filter_mc;
  a.pad = k / 2; a.cout = cout; a.out = (T*)out_delta; a.res = reservoir; a.act = act_kind; a.slope = slope;
  a.addend = (const T*)addend; a.refresh = refresh ? 1 : 0; a.bias = bias;
  a.hid = 0; a.g_cpd = nullptr; a.g_cpm = nullptr; a.g_cpres = nullptr; a.g_cres = nullptr; a.g_dh = nullptr; a.g_dc = nullptr;
  a.ws = (float*)workspace; a.ws_floats = workspace_bytes / 4; a.ws_plane = 0; a.xcd_fs = 0; a.xcd_m = 0; a.x3 = x3;
  a.ts = mie_dev_tileset(out);
  const TileSetDev pts = mie_dev_tileset(blocks);
  if (lead != nullptr) {
    MIE_REQUIRE(lead_filter != nullptr && mie_aligned(lead, 2 * sizeof(T)) && mie_aligned(lead_filter, 16) && lead != out_delta, MIE_ERR_INVALID_ARG,
                "%s: lead and its filter rows must be given together, aligned, and not alias the output", who);
    a.g_cpd = (const T*)lead; a.g_cpm = lead_mask; a.g_cpres = const_cast<float*>(lead_filter);
  }
  bool ok;
  if constexpr (sizeof(T) == 4) {
    if (x3 == 2) ok = (k == 3) ? launch_tconv<T, 3, 2>(a, pts, (hipStream_t)stream) : launch_tconv<T, 5, 2>(a, pts, (hipStream_t)stream);
    else if (x3) ok = (k == 3) ? launch_tconv<T, 3, 1>(a, pts, (hipStream_t)stream) : launch_tconv<T, 5, 1>(a, pts, (hipStream_t)stream);
    else ok = (k == 3) ? launch_tconv<T, 3>(a, pts, (hipStream_t)stream) : launch_tconv<T, 5>(a, pts, (hipStream_t)stream);
  } else {
    ok = (k == 3) ? launch_tconv<T, 3>(a, pts, (hipStream_t)stream) : launch_tconv<T, 5>(a, pts, (hipStream_t)stream);
  }
  MIE_REQUIRE(ok, MIE_ERR_UNSUPPORTED, "%s: no kernel variant for c1=%d c2=%d cout=%d", who, c1, c2, cout);
  return mie_check_launch(who);
}

}  // namespace

extern "C" int mie_tconv2x_masked(const void* x, const uint8_t* xmask, int c1, const void* x2, const uint8_t* x2mask,
                                  int c2, int h_in, int w_in, const float* filter, const void* filter_mc,
                                  int cin_total, int k, int cout, const mie_tileset* out, const mie_tileset* blocks,
                                  void* out_delta, const void* addend, float* reservoir, int act_kind, float slope,
                                  int dtype, void* workspace, long long workspace_bytes, void* stream) {
  const char* who = "mie_tconv2x_masked";
  mie_clear_error();
  const int x3 = dtype == MIE_DTYPE_F32_BF16X3 ? 1 : dtype == MIE_DTYPE_F32_F16X2 ? 2 : 0;
  if (x3) dtype = MIE_DTYPE_F32;
  MIE_REQUIRE(dtype == MIE_DTYPE_F32 || dtype == MIE_DTYPE_BF16, MIE_ERR_UNSUPPORTED, "%s: unknown delta dtype %d", who, dtype);
  if (dtype == MIE_DTYPE_BF16)
    return tconv2x_impl<mie_bf16>(who, x, xmask, c1, x2, x2mask, c2, h_in, w_in, filter, filter_mc, cin_total, k, cout, out,
                                  blocks, out_delta, addend, reservoir, act_kind, slope, false, nullptr, workspace,
                                  workspace_bytes, stream);
  return tconv2x_impl<float>(who, x, xmask, c1, x2, x2mask, c2, h_in, w_in, filter, filter_mc, cin_total, k, cout, out, blocks,
                             out_delta, addend, reservoir, act_kind, slope, false, nullptr, workspace, workspace_bytes,
                             stream, x3);
}

extern "C" int mie_tconv2x_refresh(const void* x, int c1, const void* x2, int c2, int h_in, int w_in, const float* filter,
                                   const void* filter_mc, int cin_total, int k, int cout, const float* bias,
                                   const mie_tileset* out, const mie_tileset* blocks, void* out_dense, const void* addend,
                                   float* reservoir, int act_kind, float slope, int dtype, void* stream) {
  const char* who = "mie_tconv2x_refresh";
  mie_clear_error();
  const int x3 = dtype == MIE_DTYPE_F32_BF16X3 ? 1 : dtype == MIE_DTYPE_F32_F16X2 ? 2 : 0;
  if (x3) dtype = MIE_DTYPE_F32;
  MIE_REQUIRE(dtype == MIE_DTYPE_F32 || dtype == MIE_DTYPE_BF16, MIE_ERR_UNSUPPORTED, "%s: unknown delta dtype %d", who, dtype);
  if (dtype == MIE_DTYPE_BF16)
    return tconv2x_impl<mie_bf16>(who, x, nullptr, c1, x2, nullptr, c2, h_in, w_in, filter, filter_mc, cin_total, k, cout, out,
                                  blocks, out_dense, addend, reservoir, act_kind, slope, true, bias, nullptr, 0, stream);
  return tconv2x_impl<float>(who, x, nullptr, c1, x2, nullptr, c2, h_in, w_in, filter, filter_mc, cin_total, k, cout, out, blocks,
                             out_dense, addend, reservoir, act_kind, slope, true, bias, nullptr, 0, stream, x3);
}

extern "C" int mie_tconv2x_lead_masked(const void* lead, const uint8_t* lead_mask, const float* lead_filter, const void* x, const uint8_t* xmask,
                                       int c1, const void* x2, const uint8_t* x2mask, int c2, int h_in, int w_in, const float* filter,
                                       const void* filter_mc, int cin_total, int cout, const mie_tileset* out, const mie_tileset* blocks,
                                       void* out_delta, float* reservoir, int act_kind, float slope, int dtype, void* stream) {
  const char* who = "mie_tconv2x_lead_masked";
  mie_clear_error();
  MIE_REQUIRE(lead != nullptr, MIE_ERR_INVALID_ARG, "%s: NULL pointer", who);
  MIE_REQUIRE(dtype == MIE_DTYPE_BF16 || dtype == MIE_DTYPE_F32_BF16X3 || dtype == MIE_DTYPE_F32_F16X2, MIE_ERR_UNSUPPORTED, "%s: bf16 deltas or fp32 ones in terms, not dtype %d", who, dtype);
  if (dtype == MIE_DTYPE_BF16)
    return tconv2x_impl<mie_bf16>(who, x, xmask, c1, x2, x2mask, c2, h_in, w_in, filter, filter_mc, cin_total, 3, cout, out, blocks, out_delta,
                                  nullptr, reservoir, act_kind, slope, false, nullptr, nullptr, 0, stream, 0, lead, lead_mask, lead_filter);
  return tconv2x_impl<float>(who, x, xmask, c1, x2, x2mask, c2, h_in, w_in, filter, filter_mc, cin_total, 3, cout, out, blocks, out_delta, nullptr,
                             reservoir, act_kind, slope, false, nullptr, nullptr, 0, stream, dtype == MIE_DTYPE_F32_F16X2 ? 2 : 1, lead, lead_mask, lead_filter);
}
