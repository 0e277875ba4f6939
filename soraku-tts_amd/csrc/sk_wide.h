// Decode kernels for many rows (more than the GEMV kernels' 4): several
// utterances with CFG decoded together, up to 32 rows (the reference decodes
// one utterance's two CFG rows; fast_generate.py:232-328 batches those).
//
// The projections run as skinny GEMMs on the matrix cores: each
// workgroup owns 16 outputs for all rows and splits K over its waves;
// the per-wave partial tiles are summed through LDS in fixed wave order
// (deterministic).  RMSNorms that feed a projection are folded into it.
#pragma once

#include <hip/hip_runtime.h>

#include <type_traits>

#include "sk_kernels.h"

namespace sk {
namespace {   // internal linkage, as sk_kernels.h: both translation units include these kernels

struct SkinnyArgs {
  const void* w[3]; int seg_rows[3];   // weight segments (q / k / v), rows of each
  const void* w2;                      // SwiGLU: up weights
  const float* x; int ldx;             // [R][K]
  const float* norm_w; float eps;      // optional RMSNorm of x rows (gain [K])
  float* out; int ldo;                 // [R][N]
  const float* res; int ldr;           // residual (may alias out)
  const float* bias;                   // [N]
  int R, N, K;
  int ksplit;                          // K slices per output tile (1, 2 or 4)
  float* partial;                      // [tiles][ksplit][SK_PSZ] slice partials (ksplit > 1)
  unsigned* arrive;                    // [tiles] slice arrival counts, zero between launches
  // BF16 products only:
  const uint16_t* xs;                  // x in split form (xsplit_index), gain applied; null: FP32 x
  const float* ss_in; int n_ss;        // NORM with xs: [32][n_ss] partial sums of x^2 per row
  uint16_t* xs_out;                    // out again in split form for the next GEMM; null: none
  const float* xs_gain;                // gain applied before that split (the next RMSNorm); null: 1
  float* ss_out;                       // [32][N/16] sums of out^2 per row and output tile; null: none
  float* pre_out; int ld_pre;          // SwiGLU: gate and up before the activation, [R][ld_pre]
                                       // (gate at o, up at N + o); null: none
  // Split-K merge by tagged words (null tpart: the arrival-count merge):
  // slices 1.. store their partials as 8-byte words (value, tag) and leave;
  // slice 0 reads them until every tag is this launch's, *fc * 256 + tag_idx
  // + 1 (fc: the frame counter, constant over a frame; tag_idx: the launch's
  // place among the frame's GEMM launches), so a word left by an earlier
  // launch never carries it (the host clears the words wherever the frame
  // counter restarts at 0).  A wait past `spin` ticks sets err bit 1.
  unsigned long long* tpart;           // [tiles][SK_MAX_SPLIT][SK_PSZ]
  const int* fc; int tag_idx;
  unsigned* err; unsigned long long spin;
};

// Floats per slice partial: two epilogue values per thread (SwiGLU) + 32 row
// sums of squares.
constexpr int SK_PSZ = 2 * 512 + 32;
constexpr int SK_MAX_SPLIT = 4;          // largest K split a launch may use

constexpr int SK_ROWS = 32;             // rows covered (two 16-row MFMA tiles)

typedef float sv4f __attribute__((ext_vector_type(4)));

// out[r][o] for 16 outputs o of this workgroup and all rows r < R.  Lane l of
// a wave holds VEC consecutive k at kb + VEC (l / 16) of output o0 + l % 16's
// weights and of rows (l % 16) (+ 16) of x, so every k of a block enters the
// sum exactly once.  Wave w takes blocks w, w + W, ... of the slice.  NORM: x
// is taken through RMSNorm -- the gain is applied per k, the row's sum of
// squares is gathered on the way and 1 / rms scales the sum at the end (out =
// inv_rms * sum_k w_k g_k x_k).  EPI is one of the GEMV epilogues (store, bias,
// residual, SwiGLU).  TR: 16-row tiles of x (1 for R <= 16, which halves the x
// loads and the products).  How the products are formed (MM):
//   MM_SPLIT  BF16 weights, v_mfma_f32_16x16x32_bf16: each x value (times the
//             norm gain) is split into x_hi = bf16(x) and x_lo = bf16(x -
//             x_hi) and both go through the MFMA, so the products are exact in
//             FP32 and x keeps ~16 mantissa bits (relative error <= 2^-16);
//   MM_XS     the same with x already in split form (below);
//   MM_F32    FP32 weights, v_mfma_f32_16x16x4f32: exact FP32 products;
//   MM_WIDE   BF16 weights widened to FP32, the FP32 MFMA (the operator API,
//             whose results are FP32 sums of the exact products).
// MM_F32 and MM_WIDE take K a multiple of 4 and 8 (TAIL: not of the block).
// What bounds it: at 8 to 32 rows the weights (HBM) in principle; in fact the
// latency of a launch's loads, so every load of a slice is issued up front
// where registers allow.  FP32 weights, 8 rows, the O / down projections of
// the 0.6B shape (1024 x 2048 to 3072), mean per launch in the frame: 11.4 us
// with one workgroup per tile over all of K and 32 rows of x, 5.6-6.0 us with K
// over 4 slices and 16 rows; 16 utterances, BF16: unchanged.
//
// Split K (ksplit S > 1, for outputs too few to fill the GPU): the S slices of
// an output tile are workgroups tile % 8 + 8 (S (tile / 8) + s), so all run on
// XCD tile % 8 (workgroups are dispatched to the 8 XCDs round-robin) and share
// its L2.  Each slice stores its partial tile, waits until the stores are
// acknowledged, and counts itself in arrive[tile] (an L2 atomic); the last
// slice to arrive adds the S partials in slice order, applies the epilogue and
// resets the count.  No workgroup waits for another.  The arrival count and
// the partials are workgroup-scope operations: they are coherent only because
// every slice of a tile runs on one XCD.  sk_create checks that mapping with
// xcd_probe_kernel and launches without split K when it does not hold.
//
// Split input (XS): x arrives in split form, written by the kernel that
// produced it with this GEMM's norm gain applied, so a stage is four 16-byte
// fragment loads per lane and no conversion; with NORM the row's sum of
// squares is the sum of the producer's per-tile partials (ss_in).  Outputs
// can be written in split form for the next GEMM (xs_out, with that GEMM's
// gain) together with their per-tile sums of squares (ss_out).
enum { MM_SPLIT = 0, MM_XS = 1, MM_F32 = 2, MM_WIDE = 3 };
typedef __bf16 sbf8 __attribute__((ext_vector_type(8)));
typedef uint32_t su4 __attribute__((ext_vector_type(4)));   // native vectors: copies of HIP's uint4 / float4 structs went through scratch

// XCC_ID hardware register of each workgroup (one 64-thread wave each): the
// XCD it runs on.  Split K needs workgroups whose ids agree modulo 8 to share
// an XCD (and so an L2).
__global__ __launch_bounds__(64) void xcd_probe_kernel(unsigned* ids) {
  const unsigned xcc = __builtin_amdgcn_s_getreg((31 << 11) | 20);   // hwreg(HW_REG_XCC_ID)
  if (threadIdx.x == 0) ids[blockIdx.x] = xcc;
}
constexpr int XCD_PROBE_WGS = 2048;

template <int EPI, int W, bool NORM, int MM, int TR, bool TAIL = false>
__global__ __launch_bounds__(W * 64) void skinny_kernel(SkinnyArgs a) {
  constexpr bool XS = MM == MM_XS, WF = MM == MM_F32, EXACT = MM >= MM_F32;
  static_assert(!XS || W == 8, "split input: one thread per (row, 16th of the partial sums)");
  static_assert(!TAIL || EXACT, "the BF16 products take whole blocks");
  static_assert(W * 64 >= 256 * TR, "one thread per output");
  constexpr int NA = (EPI == EPI_SWIGLU) ? 2 : 1;
  constexpr int VEC = WF ? 4 : 8;       // k per lane and block
  constexpr int BK = 4 * VEC;           // k per block
  constexpr bool XNORM = NORM && !XS;   // gain and sum of squares taken from FP32 x here
  __shared__ float red[W][NA * TR * 4][64];
  __shared__ float ssq[XNORM ? W : 1][TR][64];
  __shared__ float ssr[XS_ROWS];
  __shared__ float sso[TR][4][64];
  __shared__ int last_slice;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int i16 = lane & 15, kq = lane >> 4;
  const int S = a.ksplit;
  const bool tagged = S > 1 && a.tpart != nullptr;
  const int fcv = tagged ? *a.fc : 0;
  int tile = blockIdx.x, slice = 0;
  if (S > 1) {
    const int xcd = blockIdx.x & 7, q = blockIdx.x >> 3;
    slice = q % S;
    tile = (q / S) * 8 + xcd;
  }
  const int kbeg = slice * (a.K / S), kend = kbeg + a.K / S;
  const int o0 = tile * 16;
  const int o = min(o0 + i16, a.N - 1);
  const void* wb;
  int wr;
  if (o < a.seg_rows[0]) { wb = a.w[0]; wr = o; }
  else if (o < a.seg_rows[0] + a.seg_rows[1]) { wb = a.w[1]; wr = o - a.seg_rows[0]; }
  else { wb = a.w[2]; wr = o - a.seg_rows[0] - a.seg_rows[1]; }
  constexpr int WES = WF ? 4 : 2;       // bytes of a weight
  const char* wp = static_cast<const char*>(wb) + ((size_t)wr * a.K + VEC * kq) * WES;
  const char* w2p = NA == 2 ? static_cast<const char*>(a.w2) + ((size_t)o * a.K + VEC * kq) * WES : nullptr;
  const float* xr[TR];
#pragma unroll
  for (int t = 0; t < TR; ++t) xr[t] = a.x + (size_t)min(16 * t + i16, a.R - 1) * a.ldx + VEC * kq;
  const float* gp = XNORM ? a.norm_w + VEC * kq : nullptr;
  const su4* xsp = XS ? reinterpret_cast<const su4*>(a.xs) + lane : nullptr;
  constexpr int NX = VEC / 4;           // float4 of x per lane, block and row tile
  struct StageF { su4 w[NA]; sv4f x[TR][NX], g[XNORM ? NX : 1]; };
  struct StageS { su4 w[NA]; su4 xs[2 * TR]; };   // hi/lo of each row tile
  using Stage = typename std::conditional<XS, StageS, StageF>::type;
  auto load = [&](int kb, Stage& st) __attribute__((always_inline)) {
    int off = kb;                       // TAIL: lanes past K re-read K's last elements, zeroed below
    bool in = true;
    if constexpr (TAIL) {
      in = kb + VEC * kq < a.K;
      off = min(kb, a.K - VEC - VEC * kq);
    }
    st.w[0] = *reinterpret_cast<const su4*>(wp + (ptrdiff_t)off * WES);
    if constexpr (NA == 2) st.w[NA - 1] = *reinterpret_cast<const su4*>(w2p + (ptrdiff_t)off * WES);
    if constexpr (XS) {
#pragma unroll
      for (int j = 0; j < 2 * TR; ++j) st.xs[j] = xsp[((size_t)(kb >> 5) * 4 + j) * 64];
    } else {
#pragma unroll
      for (int h = 0; h < NX; ++h) {
#pragma unroll
        for (int t = 0; t < TR; ++t) {
          st.x[t][h] = *reinterpret_cast<const sv4f*>(xr[t] + off + 4 * h);
          if constexpr (TAIL) {
#pragma unroll
            for (int i = 0; i < 4; ++i) st.x[t][h][i] = in ? st.x[t][h][i] : 0.f;
          }
        }
        if constexpr (XNORM) st.g[h] = *reinterpret_cast<const sv4f*>(gp + off + 4 * h);
      }
    }
    if constexpr (TAIL) {
#pragma unroll
      for (int n = 0; n < NA; ++n)
#pragma unroll
        for (int i = 0; i < 4; ++i) st.w[n][i] = in ? st.w[n][i] : 0u;
    }
  };
  // Exact products: four sums, of k = 0, 1, 2, 3 mod 4, flushed into a total
  // every 4 stages: chains of at most 32 (FP32: 16) products keep the sums'
  // rounding below the GEMV kernels' (one chain over a wave's K: twice theirs).
  constexpr int NACC = EXACT ? 4 : 1;
  sv4f accs[NACC][NA][TR], tot[EXACT ? NA : 1][EXACT ? TR : 1];
#pragma unroll
  for (int n = 0; n < NA; ++n)
#pragma unroll
    for (int t = 0; t < TR; ++t) {
#pragma unroll
      for (int c = 0; c < NACC; ++c) accs[c][n][t] = sv4f{0.f, 0.f, 0.f, 0.f};
      if constexpr (EXACT) tot[n][t] = sv4f{0.f, 0.f, 0.f, 0.f};
    }
  auto flush = [&]() __attribute__((always_inline)) {
    if constexpr (EXACT) {
#pragma unroll
      for (int n = 0; n < NA; ++n)
#pragma unroll
        for (int t = 0; t < TR; ++t) {
          tot[n][t] += (accs[0][n][t] + accs[1 % NACC][n][t]) + (accs[2 % NACC][n][t] + accs[3 % NACC][n][t]);
#pragma unroll
          for (int c = 0; c < NACC; ++c) accs[c][n][t] = sv4f{0.f, 0.f, 0.f, 0.f};
        }
    }
  };
  float ssx[TR] = {};
  // this lane's x of row tile t, gain applied (XNORM: its squares gathered first)
  auto xval = [&](const auto& st, int t, float (&v)[VEC]) __attribute__((always_inline)) {
#pragma unroll
    for (int h = 0; h < NX; ++h) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        v[4 * h + i] = st.x[t][h][i];
        if constexpr (XNORM) {
          ssx[t] = fmaf(v[4 * h + i], v[4 * h + i], ssx[t]);
          v[4 * h + i] *= st.g[h][i];
        }
      }
    }
  };
  auto comp = [&](const Stage& st) __attribute__((always_inline)) {
    if constexpr (EXACT) {
      float v[TR][VEC];
#pragma unroll
      for (int t = 0; t < TR; ++t) xval(st, t, v[t]);
#pragma unroll
      for (int j = 0; j < VEC; ++j)
#pragma unroll
        for (int n = 0; n < NA; ++n) {
          const uint32_t ww = st.w[n][WF ? j % 4 : j / 2];
          const float wv = __uint_as_float(WF ? ww : j & 1 ? ww & 0xffff0000u : ww << 16);
#pragma unroll
          for (int t = 0; t < TR; ++t)
            accs[j % NACC][n][t] = __builtin_amdgcn_mfma_f32_16x16x4f32(wv, v[t][j], accs[j % NACC][n][t], 0, 0, 0);
        }
    } else {
      sbf8 hi[TR], lo[TR];
#pragma unroll
      for (int t = 0; t < TR; ++t) {
        if constexpr (XS) {
          hi[t] = __builtin_bit_cast(sbf8, st.xs[2 * t]);
          lo[t] = __builtin_bit_cast(sbf8, st.xs[2 * t + 1]);
        } else {
          float v[VEC];
          xval(st, t, v);
#pragma unroll
          for (int j = 0; j < VEC; ++j) {
            const __bf16 h = (__bf16)v[j];
            hi[t][j] = h;
            lo[t][j] = (__bf16)(v[j] - (float)h);
          }
        }
      }
#pragma unroll
      for (int n = 0; n < NA; ++n) {
        const sbf8 wa = __builtin_bit_cast(sbf8, st.w[n]);
#pragma unroll
        for (int t = 0; t < TR; ++t) {
          accs[0][n][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wa, hi[t], accs[0][n][t], 0, 0, 0);
          accs[0][n][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wa, lo[t], accs[0][n][t], 0, 0, 0);
        }
      }
    }
  };
  // Split input with NORM: the producer's partial sums of squares of row
  // tid / 16, 16 threads per row, loaded ahead of the first stage.
  constexpr int SSP = 16;               // partials per thread: n_ss <= 256
  float ssp[(XS && NORM) ? SSP : 1];
  if constexpr (XS && NORM) {
    // index clamped in bounds, value masked: no branch between the loads
    const float* sp = a.ss_in + (size_t)(tid >> 4) * a.n_ss;
#pragma unroll
    for (int i = 0; i < SSP; ++i) {
      const int j = (tid & 15) + 16 * i;
      const float v = sp[min(j, a.n_ss - 1)];
      ssp[i] = j < a.n_ss ? v : 0.f;
    }
  }
  // Epilogue operands of this thread's output (row r, column oo), loaded at
  // entry: they do not depend on the sums.
  const bool et = tid < 256 * TR;       // these threads own one (row tile, v, lane) each
  const int t = TR == 2 ? (tid >> 8) & 1 : 0, v = (tid >> 6) & 3, l = tid & 63;
  const int oo = o0 + 4 * (l >> 4) + v, r = 16 * t + (l & 15);
  const bool ok = et && oo < a.N && r < a.R;
  float epi_in = 0.f;
  if constexpr (EPI == EPI_BIAS) epi_in = ok ? a.bias[oo] : 0.f;
  if constexpr (EPI == EPI_RESID) epi_in = ok ? a.res[(size_t)r * a.ldr + oo] : 0.f;
  // the split-form output's gain too (index clamped: no branch around the load)
  const float gain_in = a.xs_gain ? a.xs_gain[min(oo, a.N - 1)] : 1.f;
  constexpr int STEP = W * BK;
  // This wave's stages: k = kw0 + i * STEP for i < nst.  Up to UP stages (8, or 4
  // where a stage is wide; nearly every slice of the 0.6B shapes) the wave
  // issues all of its loads up front, in straight-line code for its exact
  // stage count, then multiplies the stages in order: each multiply waits for
  // its own stage only.  (In a loop with conditional loads the compiler cannot
  // count the loads in flight and waited for all of them.)  Longer slices go
  // in chunks of UP / 2 stages, the next chunk's loads in flight under this one's
  // products, then the remainder up front.
  const int kw0 = kbeg + wave * BK;
  const int nst = kw0 < kend ? (kend - kw0 + STEP - 1) / STEP : 0;
  constexpr int SREG = XS ? 4 * NA + 8 * TR : (NA + (TR + (XNORM ? 1 : 0)) * NX) * 4;   // registers of a stage
  // Registers of 8 stages, the sums and the operands in work: past 224 of the
  // 256 that a lane of 8 waves has, the compiler spills.  4 stages instead of 8
  // with spills: FP32 gate/up, 18 / 20 / 32 rows, 0.6B frame 1,852 / 1,901 /
  // 2,091 us -> 1,832 / 1,882 / 2,071 (6 stages 1,885 / 1,935 / 2,107); BF16
  // operators of 20 rows, 1024 x 3080 14.8 -> 12.2 us, 2048 x 6136 25.0 -> 20.8.
  constexpr int REGS8 = 8 * SREG + (EXACT ? (NACC + 1) * NA * TR * 4 + TR * VEC + (TAIL ? 2 * VEC : 0) : 0);
  constexpr int UP = SREG > 20 || (MM <= MM_XS && TR == 2) ? 4 : REGS8 > 224 ? 4 : 8, CH = UP / 2;
  auto upfront = [&](int k0, auto nc) __attribute__((always_inline)) {
    constexpr int NC = decltype(nc)::value;
    Stage st[NC];
#pragma unroll
    for (int i = 0; i < NC; ++i) load(k0 + i * STEP, st[i]);
    asm volatile("" ::: "memory");   // not sunk towards the multiplies
#pragma unroll
    for (int i = 0; i < NC; ++i) {
      comp(st[i]);
      if (i % 4 == 3 || i == NC - 1) flush();
    }
  };
  auto rest = [&](int k0, int n) __attribute__((always_inline)) {
    if (n == 1) upfront(k0, std::integral_constant<int, 1>{});
    else if (n == 2) upfront(k0, std::integral_constant<int, 2>{});
    else if (n == 3) upfront(k0, std::integral_constant<int, 3>{});
    else if (n == 4) upfront(k0, std::integral_constant<int, 4>{});
    if constexpr (UP == 8) {
      if (n == 5) upfront(k0, std::integral_constant<int, 5>{});
      else if (n == 6) upfront(k0, std::integral_constant<int, 6>{});
      else if (n == 7) upfront(k0, std::integral_constant<int, 7>{});
      else if (n == 8) upfront(k0, std::integral_constant<int, 8>{});
    }
  };
  int done = 0;                         // stages already multiplied
  if (nst > UP) {
    Stage sa[CH], sb[CH];
    auto load4 = [&](int c, Stage (&st)[CH]) __attribute__((always_inline)) {
#pragma unroll
      for (int i = 0; i < CH; ++i) load(kw0 + (c * CH + i) * STEP, st[i]);
      asm volatile("" ::: "memory");
    };
    auto comp4 = [&](const Stage (&st)[CH]) __attribute__((always_inline)) {
#pragma unroll
      for (int i = 0; i < CH; ++i) comp(st[i]);
      flush();
    };
    const int nch = nst / CH;
    load4(0, sa);
    for (int c = 0;; c += 2) {
      if (c + 1 >= nch) { comp4(sa); break; }
      load4(c + 1, sb);
      comp4(sa);
      if (c + 2 >= nch) { comp4(sb); break; }
      load4(c + 2, sa);
      comp4(sb);
    }
    done = nch * CH;
  }
  rest(kw0 + done * STEP, nst - done);
  // The row's sum of squares is needed only by the epilogue: summed after the
  // stream, so waiting for the partials never holds back a stage's loads.
  if constexpr (XS && NORM) {
    float t = 0.f;
#pragma unroll
    for (int i = 0; i < SSP; ++i) t += ssp[i];
    t += __shfl_xor(t, 8, 64);          // the row's 16 threads; each pair adds in both orders alike
    t += __shfl_xor(t, 4, 64);
    t += __shfl_xor(t, 2, 64);
    t += __shfl_xor(t, 1, 64);
    if ((tid & 15) == 0) ssr[tid >> 4] = t;
  }
#pragma unroll
  for (int n = 0; n < NA; ++n)
#pragma unroll
    for (int t = 0; t < TR; ++t)
#pragma unroll
      for (int v = 0; v < 4; ++v)
        red[wave][(n * TR + t) * 4 + v][lane] = EXACT ? tot[EXACT ? n : 0][EXACT ? t : 0][v] : accs[0][n][t][v];
  if constexpr (XNORM) {
#pragma unroll
    for (int t = 0; t < TR; ++t) ssq[wave][t][lane] = ssx[t];
  }
  __syncthreads();
  // Waves past the output threads only take part in the barriers.
  float c[NA];
#pragma unroll
  for (int n = 0; n < NA; ++n) {
    float sacc = 0.f;
    if constexpr (EXACT && W % 4 == 0) {   // in groups of 4 waves, for the sums' rounding
#pragma unroll
      for (int w = 0; w < W; w += 4) {
        const int i = (n * TR + t) * 4 + v;
        sacc += (red[w][i][l] + red[w + 1][i][l]) + (red[w + 2][i][l] + red[w + 3][i][l]);
      }
    } else {
#pragma unroll
      for (int w = 0; w < W; ++w) sacc += red[w][(n * TR + t) * 4 + v][l];
    }
    c[n] = sacc;
  }
  float ss = 0.f;
  if constexpr (XNORM) {
#pragma unroll
    for (int w = 0; w < W; ++w)
#pragma unroll
      for (int k4 = 0; k4 < 4; ++k4) ss += ssq[w][t][k4 * 16 + (l & 15)];
  }
  if constexpr (XS && NORM) ss = ssr[r];
  if (tagged) {
    const unsigned long long tag = (unsigned long long)((unsigned)fcv * 256u + (unsigned)a.tag_idx + 1u) << 32;
    unsigned long long* tp = a.tpart + (size_t)tile * SK_MAX_SPLIT * SK_PSZ;
    auto put = [&](unsigned long long* p, float x) {
      __hip_atomic_store(p, tag | __float_as_uint(x), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    };
    if (slice != 0) {
      if (et) {
#pragma unroll
        for (int n = 0; n < NA; ++n) put(tp + (size_t)slice * SK_PSZ + n * 512 + tid, c[n]);
        if (XNORM && v == 0 && (l >> 4) == 0) put(tp + (size_t)slice * SK_PSZ + 2 * 512 + r, ss);
      }
      return;
    }
    if (et) {
      // slices 1 .. S-1 (unrolled to SK_MAX_SPLIT, slice index clamped):
      // word (q - 1) * NA + n, then the row sums of squares
      constexpr int NW = (NA + (XNORM ? 1 : 0)) * (SK_MAX_SPLIT - 1);
      auto addr = [&](int i) {
        const int q = i < NA * (SK_MAX_SPLIT - 1) ? i / NA + 1 : i - NA * (SK_MAX_SPLIT - 1) + 1;
        const size_t qo = (size_t)min(q, S - 1) * SK_PSZ;
        return i < NA * (SK_MAX_SPLIT - 1) ? tp + qo + (i % NA) * 512 + tid : tp + qo + 2 * 512 + r;
      };
      unsigned long long w[NW];
#pragma unroll
      for (int i = 0; i < NW; ++i) w[i] = *addr(i);
      const unsigned long long deadline = __builtin_amdgcn_s_memrealtime() + a.spin;
      for (;;) {
        bool miss = false;
#pragma unroll
        for (int i = 0; i < NW; ++i) miss |= (w[i] & 0xffffffff00000000ull) != tag;
        if (!miss) break;
        if (__builtin_amdgcn_s_memrealtime() > deadline) {
          __hip_atomic_fetch_or(a.err, 2u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
          break;
        }
#pragma unroll
        for (int i = 0; i < NW; ++i)
          if ((w[i] & 0xffffffff00000000ull) != tag)
            w[i] = __hip_atomic_load(addr(i), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
      // in slice order, as the arrival-count merge adds them
#pragma unroll
      for (int n = 0; n < NA; ++n)
#pragma unroll
        for (int q = 1; q < SK_MAX_SPLIT; ++q)
          if (q < S) c[n] += __uint_as_float((unsigned)w[(q - 1) * NA + n]);
      if constexpr (XNORM) {
#pragma unroll
        for (int q = 1; q < SK_MAX_SPLIT; ++q)
          if (q < S) ss += __uint_as_float((unsigned)w[NA * (SK_MAX_SPLIT - 1) + q - 1]);
      }
    }
  } else if (S > 1) {
    float* mine = a.partial + ((size_t)tile * S + slice) * SK_PSZ;
    if (et) {
#pragma unroll
      for (int n = 0; n < NA; ++n) mine[n * 512 + tid] = c[n];
      if (XNORM && v == 0 && (l >> 4) == 0) mine[2 * 512 + r] = ss;
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // this thread's partials are in L2
    __syncthreads();
    if (tid == 0)
      last_slice = __hip_atomic_fetch_add(a.arrive + tile, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) + 1u ==
                   (unsigned)S;
    __syncthreads();
    if (!last_slice) return;
    if (tid == 0) __hip_atomic_store(a.arrive + tile, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    if (et) {
      // All slices' partials loaded together (slice index clamped, unrolled
      // to SK_MAX_SPLIT), then summed in slice order: a loop over the runtime
      // S waited for each load before issuing the next.
      const float* all = a.partial + (size_t)tile * S * SK_PSZ;
      float pv[NA][SK_MAX_SPLIT], sv[XNORM ? SK_MAX_SPLIT : 1];
#pragma unroll
      for (int q = 0; q < SK_MAX_SPLIT; ++q) {
        const size_t qo = (size_t)min(q, S - 1) * SK_PSZ;
#pragma unroll
        for (int n = 0; n < NA; ++n) pv[n][q] = all[qo + n * 512 + tid];
        if constexpr (XNORM) sv[q] = all[qo + 2 * 512 + r];
      }
#pragma unroll
      for (int n = 0; n < NA; ++n) {
        float sacc = 0.f;
#pragma unroll
        for (int q = 0; q < SK_MAX_SPLIT; ++q)
          if (q < S) sacc += pv[n][q];
        c[n] = sacc;
      }
      if constexpr (XNORM) {
        ss = 0.f;
#pragma unroll
        for (int q = 0; q < SK_MAX_SPLIT; ++q)
          if (q < S) ss += sv[q];
      }
    }
  }
  if constexpr (NORM) {
    const float inv = 1.0f / sqrtf(ss / (float)a.K + a.eps);
#pragma unroll
    for (int n = 0; n < NA; ++n) c[n] *= inv;
  }
  float y = 0.f;
  if (ok) {
    y = c[0];
    if constexpr (EPI == EPI_BIAS) y = y + epi_in;
    if constexpr (EPI == EPI_RESID) y = epi_in + y;
    if constexpr (EPI == EPI_SWIGLU) {
      if (a.pre_out) {
        a.pre_out[(size_t)r * a.ld_pre + oo] = y;
        a.pre_out[(size_t)r * a.ld_pre + a.N + oo] = c[NA - 1];
      }
      y = y / (1.0f + expf(-y)) * c[NA - 1];
    }
    a.out[(size_t)r * a.ldo + oo] = y;
    if (a.xs_out) xsplit_store(a.xs_out, r, oo, a.xs_gain ? y * gain_in : y);
  }
  if (a.ss_out) {                       // uniform over the workgroup
    if (et) sso[t][v][l] = y * y;
    __syncthreads();
    if (et && v == 0 && (l >> 4) == 0 && r < a.R) {
      float sq = 0.f;
#pragma unroll
      for (int v2 = 0; v2 < 4; ++v2)
#pragma unroll
        for (int q = 0; q < 4; ++q) sq += sso[t][v2][q * 16 + (l & 15)];
      a.ss_out[(size_t)r * (a.N / 16) + tile] = sq;
    }
  }
}


// K over 4 or 2 workgroups per output tile when the tiles alone would fill
// fewer than 256 CUs (tiles a multiple of 8, slices whole blocks).
template <int EPI, bool NORM, int MM, int TR>
inline hipError_t launch_skinny_t(SkinnyArgs a, bool allow_split, hipStream_t st) {
  const int tiles = (a.N + 15) / 16;
  constexpr int BK = MM == MM_F32 ? 16 : 32;
  a.ksplit = 1;
  if (allow_split && tiles % 8 == 0) {
    if (tiles <= 64 && a.K % (4 * BK) == 0) a.ksplit = 4;
    else if (tiles <= 128 && a.K % (2 * BK) == 0) a.ksplit = 2;
  }
  static_assert(SK_MAX_SPLIT >= 4, "the kernel's split-K merge covers the splits chosen here");
  hipLaunchKernelGGL((skinny_kernel<EPI, 8, NORM, MM, TR>), dim3(tiles * a.ksplit), dim3(8 * 64), 0, st, a);
  return hipGetLastError();
}
// A GEMM of at most 32 rows in the engine's forms: split products with BF16
// weights (x in split form when a.xs is given), exact FP32 ones otherwise.
template <int EPI, bool NORM>
inline hipError_t launch_skinny_w(bool bf16, const SkinnyArgs& a, bool allow_split, hipStream_t st) {
  const bool one = a.R <= 16;
  if (!bf16) return one ? launch_skinny_t<EPI, NORM, MM_F32, 1>(a, allow_split, st)
                        : launch_skinny_t<EPI, NORM, MM_F32, 2>(a, allow_split, st);
  if (a.xs) return one ? launch_skinny_t<EPI, NORM, MM_XS, 1>(a, allow_split, st)
                       : launch_skinny_t<EPI, NORM, MM_XS, 2>(a, allow_split, st);
  return one ? launch_skinny_t<EPI, NORM, MM_SPLIT, 1>(a, allow_split, st)
             : launch_skinny_t<EPI, NORM, MM_SPLIT, 2>(a, allow_split, st);
}

// The operator API's projections of at most 32 rows: exact products, any N, K
// a multiple of 8, in workgroups of 8 waves.  SwiGLU of up to 16 rows takes 4
// waves where that was faster: more than 256 output tiles, so that a CU holds
// two workgroups (232 registers; one where K has a tail) and one loads while the
// other multiplies, and wide FP32 rows.  us of a launch, 7 rows, gate and up,
// 4 waves / 8: BF16 2048 x 1024 7.0 / 5.7, 2688 x 1344 8.9 / 7.0, 4096 x 2048
// 12.0 / 11.2, 4608 x 1536 13.9 / 14.8, 6144 x 2048 16.4 / 20.7; FP32 2000 x 1000
// 7.2 / 6.5, 3072 x 1024 7.4 / 7.1, 2688 x 1344 9.3 / 9.5, 4096 x 2048 13.7 /
// 14.3, 6144 x 2048 22.2 / 24.1; 5, 11 and 16 rows the same way round.  (The
// others, BF16 2048 x 6144: 8 waves 15.2, 4 waves 19.6, 16 waves 22.5.)
template <int EPI, int MM, int TR, bool TAIL>
inline hipError_t launch_rows_t(const SkinnyArgs& a, hipStream_t st) {
  const int tiles = (a.N + 15) / 16;
  if constexpr (EPI == EPI_SWIGLU && TR == 1) {
    if (tiles > 256 || (MM == MM_F32 && a.K > 1024)) {
      hipLaunchKernelGGL((skinny_kernel<EPI, 4, false, MM, TR, TAIL>), dim3(tiles), dim3(4 * 64), 0, st, a);
      return hipGetLastError();
    }
  }
  hipLaunchKernelGGL((skinny_kernel<EPI, 8, false, MM, TR, TAIL>), dim3(tiles), dim3(8 * 64), 0, st, a);
  return hipGetLastError();
}
template <int EPI, int MM>
inline hipError_t launch_rows_m(const SkinnyArgs& a, hipStream_t st) {
  const bool tail = a.K % (MM == MM_F32 ? 16 : 32) != 0;
  if (a.R <= 16) return tail ? launch_rows_t<EPI, MM, 1, true>(a, st) : launch_rows_t<EPI, MM, 1, false>(a, st);
  return tail ? launch_rows_t<EPI, MM, 2, true>(a, st) : launch_rows_t<EPI, MM, 2, false>(a, st);
}
template <int EPI>
inline hipError_t launch_rows(bool bf16, SkinnyArgs a, hipStream_t st) {
  a.ksplit = 1;
  return bf16 ? launch_rows_m<EPI, MM_WIDE>(a, st) : launch_rows_m<EPI, MM_F32>(a, st);
}
inline SkinnyArgs skinny_args(const void* w, int N, int K, const float* x, int ldx, float* out, int ldo, int R) {
  SkinnyArgs a{};
  a.w[0] = w;
  a.seg_rows[0] = N;
  a.x = x; a.ldx = ldx; a.out = out; a.ldo = ldo;
  a.R = R; a.N = N; a.K = K;
  return a;
}

}  // namespace
}  // namespace sk
