// GEMMs of the batched prefill on the matrix cores: C[M][N] = A[M][K] . B[N][K]^T
// for every prefix token of a call at once (M = 1 .. thousands).
//
// FP32 weights run on the FP32 matrix cores (v_mfma_f32_16x16x4f32, exact FP32
// products).  BF16 weights run on the BF16 ones (v_mfma_f32_16x16x32_bf16):
// the activations arrive as two BF16 planes x_hi = bf16(x), x_lo = bf16(x -
// x_hi), written by the kernel that produced them, and each product takes two
// MFMAs, exact in FP32, so x keeps ~16 mantissa bits.
//
// What bounds it: getting the tiles into LDS in time (the loop without its
// loads runs 1.5x faster, without its MFMAs no faster; the matrix cores are
// busy 23-41% of the time with BF16 weights, 4,754 tokens at 0.6B and 1,314 at
// 1.7B, and 47-58% with FP32, 387 tokens).  So the loads go straight to LDS (no
// registers, no conversion: both operands are already in their final form), S - 1
// stages ahead of the multiplies in a ring, with one barrier per stage; a wave's
// part of a stage lies in LDS as whole MFMA fragments (16 rows x 64 bytes = 1 KB, a
// lane's 16 bytes at 16 * lane), so every fragment is one conflict-free 16-byte
// read per lane.  Stages of 64 bytes per row and a deeper ring beat 128 bytes
// (4700 x 4096 x 1024, BF16, 128 x 256 tiles: 105 us against 118 us).
// Measured against the kernels before it (two barriers per 32 k, operands
// through registers; us, MI355X): BF16 4700 x (2 x 3072) x 1024 SwiGLU 168 ->
// 115, 58 x 1024 x 3072 54 -> 5.3; FP32 387 x (2 x 3072) x 1024 84 -> 54,
// 387 x 1024 x 3072 66 -> 30.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>

#include "sk_kernels.h"

namespace sk {

enum { GEPI_STORE = 0, GEPI_SWIGLU = 1 };

typedef float v4f __attribute__((ext_vector_type(4)));
typedef __bf16 pbf8 __attribute__((ext_vector_type(8)));

// FP32 -> (hi, lo) BF16 pair of 4 values, packed 4 x 16 bits each.
__device__ __forceinline__ void split4(const float4 v, uint2& hi, uint2& lo) {
  const float x[4] = {v.x, v.y, v.z, v.w};
  uint16_t h[4], l[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const __bf16 b = (__bf16)x[i];
    h[i] = __builtin_bit_cast(uint16_t, b);
    l[i] = __builtin_bit_cast(uint16_t, (__bf16)(x[i] - (float)b));
  }
  hi = make_uint2((uint32_t)h[0] | ((uint32_t)h[1] << 16), (uint32_t)h[2] | ((uint32_t)h[3] << 16));
  lo = make_uint2((uint32_t)l[0] | ((uint32_t)l[1] << 16), (uint32_t)l[2] | ((uint32_t)l[3] << 16));
}

struct GemmArgs {
  const void* A; size_t a_lo;          // activations [M][K]: FP32, or BF16 hi plane and, a_lo elements on, lo plane
  const void* B[3]; int seg_rows[3];   // weight segments (q / k / v), rows of each
  const void* B2;                      // SwiGLU: up weights
  float* out; int ldo; size_t slice;   // FP32 output; K slice s writes at out + s * slice
  const float* res;                    // added to C if not null (out's layout, may be out)
  uint16_t* xs; size_t xs_lo;          // SwiGLU with BF16 weights: output as hi and lo planes [M][N]
  int M, N, K;
  int mt, nt, ksplit;                  // tiles along M and N, K slices
  int gm;                              // tiles along M per group (order of the tiles)
};

// 16 bytes per lane from g straight into LDS at l + 16 * lane (l wave-uniform).
// Written as assembly because with the builtin the compiler waits for every
// load in flight (vmcnt(0)) before the next LDS read, whichever part of the
// ring it reads; the loop below does the waiting itself (stage_sync).  M0 holds
// the LDS address and is declared overwritten: a value that the compiler keeps
// there is set again afterwards (it does so, although it warns that M0 is a
// reserved register).  The statement has no outputs: nothing is
// written but LDS.
__device__ __forceinline__ void lds_load16(const char* base, unsigned voff, const char* l) {
  const unsigned a = __builtin_amdgcn_readfirstlane((unsigned)(uintptr_t)(const __attribute__((address_space(3))) void*)l);
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(voff), "s"(base), "s"(a)
               : "memory", "m0");
}

// This wave's stage loads but the last N are in and its LDS reads are done;
// then the workgroup meets.
template <int N>
__device__ __forceinline__ void stage_sync() {
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(N) : "memory");
}

// WL: WF32 or WBF16.  Workgroup tile BM x BN (weights: BN columns; SwiGLU:
// BN / 2 gate and the same BN / 2 up columns), WM x WN waves, S stages of the
// ring, H x 64 bytes of every row per stage.  The MFMAs take the weights as
// their row operand, so a lane ends up with 4 consecutive columns of one row
// of C: 16-byte stores.  Rows past M or N are clamped on load and not stored.
// Epilogues: store (with a residual added, or K slice s at out + s * slice:
// whoever reads it adds the slices in order), SwiGLU silu(A Bg^T) * (A Bu^T) in the form the next GEMM
// takes.  K a multiple of 32, N of 16.
template <int EPI, typename WL, int BM, int BN, int WM, int WN, int S, int H>
__global__ __launch_bounds__(WM * WN * 64) void gemm_kernel(GemmArgs a) {
  constexpr bool BF = sizeof(typename WL::elem) == 2;
  constexpr int ES = BF ? 2 : 4;                 // bytes of an operand element
  constexpr int PA = BF ? 2 : 1;                 // A planes (hi, lo)
  constexpr int W = WM * WN;
  constexpr int KS = 64 * H / ES;                // k per stage: H x 64 bytes of every row
  constexpr int CA = PA * (BM / 16), CB = BN / 16;   // 16-row groups of a stage
  constexpr int C = CA + CB, CPW = (C + W - 1) / W;   // groups, groups per wave (the last may be loaded twice)
  constexpr int TM = BM / WM / 16, TN = BN / WN / 16;
  static_assert(EPI != GEPI_SWIGLU || TN % 2 == 0, "SwiGLU: every wave holds gate and up of its columns");
  constexpr int STAGE = C * H * 1024;                // bytes
  __shared__ __attribute__((aligned(1024))) char lds[S * STAGE];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int i16 = lane & 15, q4 = lane >> 4;

  // tile of this workgroup
  const int T = a.mt * a.nt * a.ksplit, per = (T + 7) / 8;
  const int t = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
  if ((blockIdx.x >> 3) >= per || t >= T) return;
  const int ks = t % a.ksplit, tt = t / a.ksplit;
  // tiles in groups of a.gm along M, M fastest within a group: the 32 tiles
  // that an XCD works on at a time share gm row panels and 32 / gm column
  // panels, which its L2 holds for the step of K that all of them are in
  const int gsz = a.gm * a.nt, gi = tt / gsz, gr = tt - gi * gsz;
  const int gm = min(a.gm, a.mt - gi * a.gm);
  const int m0 = (gi * a.gm + gr % gm) * BM;
  const int ti = gr / gm;
  constexpr int NC = EPI == GEPI_SWIGLU ? BN / 2 : BN;   // output columns of the tile
  const int n0 = ti * NC;
  // stages in K; K is a multiple of 32, so with BF16 the last stage may hold
  // one 32-k half: its second half is loaded from the first's address (in
  // bounds) and not multiplied
  const int st_all = (a.K + KS - 1) / KS;
  const bool odd = a.K % KS != 0;
  const int s0 = st_all * ks / a.ksplit, nst = st_all * (ks + 1) / a.ksplit - s0;

  // loader: group g of the stage = 16 rows x H pieces of 64 bytes (1 KB each);
  // scalar base per group (its first row), the lane's row and 16 bytes in voff
  const char* gb[CPW];
  unsigned voff[CPW];
  const int K = a.K;
#pragma unroll
  for (int c = 0; c < CPW; ++c) {
    const int g = min(wave * CPW + c, C - 1);
    const char* base;
    int row, last;
    if (g < CA) {
      const int plane = g / (BM / 16), rg = g % (BM / 16);
      base = static_cast<const char*>(a.A) + (plane ? a.a_lo * ES : 0);
      row = m0 + rg * 16;
      last = a.M - 1;
    } else {
      const int cg = g - CA;
      if constexpr (EPI == GEPI_SWIGLU) {
        const int half = BN / 32;                // 16-column groups of gate (then of up)
        base = static_cast<const char*>(cg < half ? a.B[0] : a.B2);
        row = n0 + (cg % half) * 16;
        last = a.N - 1;
      } else {                                   // segments are multiples of 16 rows when there are several
        row = n0 + cg * 16;
        base = static_cast<const char*>(a.B[0]);
        last = a.seg_rows[0] - 1;
        if (row > last && a.seg_rows[1]) {
          row -= a.seg_rows[0];
          base = static_cast<const char*>(a.B[1]);
          last = a.seg_rows[1] - 1;
          if (row > last) { row -= a.seg_rows[1]; base = static_cast<const char*>(a.B[2]); last = a.seg_rows[2] - 1; }
        }
      }
    }
    const int r0 = min(row, last);
    gb[c] = base + (size_t)r0 * K * ES;
    voff[c] = (unsigned)((min(row + i16, last) - r0) * K * ES + q4 * 16);
  }
  auto issue = [&](int s) {
    const int sk = s0 + s;
    const char* l = lds + (s % S) * STAGE;
#pragma unroll
    for (int c = 0; c < CPW; ++c) {
      const char* b = gb[c] + (size_t)sk * (64 * H);
      const int g = min(wave * CPW + c, C - 1);
      lds_load16(b, voff[c], l + g * H * 1024);
      if constexpr (H == 2) lds_load16(b + (odd && sk == st_all - 1 ? 0 : 64), voff[c], l + g * 2048 + 1024);
    }
  };
  const int wm = wave / WN, wn = wave % WN;
  v4f acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] = v4f{0.f, 0.f, 0.f, 0.f};
  // column group j of this wave (SwiGLU: first half gate, second half up)
  auto cgrp = [&](int j) {
    if constexpr (EPI == GEPI_SWIGLU) return j < TN / 2 ? wn * (TN / 2) + j : CB / 2 + wn * (TN / 2) + j - TN / 2;
    else return wn * TN + j;
  };
#pragma unroll
  for (int s = 0; s < S - 1; ++s)
    if (s < nst) issue(s);
  constexpr int L = CPW * H;                     // loads per wave and stage
  for (int s = 0; s < nst; ++s) {
    const int ahead = nst - 1 - s;
    if (ahead >= S - 2) stage_sync<L * (S - 2)>();
    else if (S > 4 && ahead == 2) stage_sync<(S > 4 ? 2 * L : 0)>();
    else if (S > 3 && ahead == 1) stage_sync<(S > 3 ? L : 0)>();
    else stage_sync<0>();
    if (s + S - 1 < nst) issue(s + S - 1);
    const char* l = lds + (s % S) * STAGE + lane * 16;
#pragma unroll
    for (int kb = 0; kb < H; ++kb) {
      if (kb == 1 && odd && s0 + s == st_all - 1) break;
      uint4 af[PA][TM], bf[TN];
#pragma unroll
      for (int p = 0; p < PA; ++p)
#pragma unroll
        for (int i = 0; i < TM; ++i)
          af[p][i] = *reinterpret_cast<const uint4*>(l + (p * (BM / 16) + wm * TM + i) * (H * 1024) + kb * 1024);
#pragma unroll
      for (int j = 0; j < TN; ++j) bf[j] = *reinterpret_cast<const uint4*>(l + (CA + cgrp(j)) * (H * 1024) + kb * 1024);
      if constexpr (BF) {
#pragma unroll
        for (int p = 0; p < PA; ++p)
#pragma unroll
          for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int i = 0; i < TM; ++i)
              acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(pbf8, bf[j]),
                                                                  __builtin_bit_cast(pbf8, af[p][i]), acc[i][j], 0, 0, 0);
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
          for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int i = 0; i < TM; ++i) {
              const v4f bv = __builtin_bit_cast(v4f, bf[j]), av = __builtin_bit_cast(v4f, af[0][i]);
              acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(bv[e], av[e], acc[i][j], 0, 0, 0);
            }
      }
    }
  }
  // lane: row m = lane % 16, columns 4 (lane / 16) .. + 3 of each 16 x 16 tile
#pragma unroll
  for (int i = 0; i < TM; ++i) {
    const int m = m0 + (wm * TM + i) * 16 + i16;
    if (m >= a.M) continue;
    if constexpr (EPI == GEPI_SWIGLU) {
#pragma unroll
      for (int j = 0; j < TN / 2; ++j) {
        const int n = n0 + (wn * (TN / 2) + j) * 16 + q4 * 4;
        if (n >= a.N) continue;
        float y[4];
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const float g = acc[i][j][v];
          y[v] = g / (1.0f + expf(-g)) * acc[i][j + TN / 2][v];
        }
        if constexpr (BF) {
          uint2 hi, lo;
          split4(make_float4(y[0], y[1], y[2], y[3]), hi, lo);
          uint16_t* o = a.xs + (size_t)m * a.N + n;
          *reinterpret_cast<uint2*>(o) = hi;
          *reinterpret_cast<uint2*>(o + a.xs_lo) = lo;
        } else {
          *reinterpret_cast<float4*>(a.out + (size_t)m * a.ldo + n) = make_float4(y[0], y[1], y[2], y[3]);
        }
      }
    } else {
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        const int n = n0 + (wn * TN + j) * 16 + q4 * 4;
        if (n >= a.N) continue;
        const size_t at = (size_t)m * a.ldo + n;
        float4 c = make_float4(acc[i][j][0], acc[i][j][1], acc[i][j][2], acc[i][j][3]);
        if (a.res) {
          const float4 r = *reinterpret_cast<const float4*>(a.res + at);
          c = make_float4(r.x + c.x, r.y + c.y, r.z + c.z, r.w + c.w);
        }
        *reinterpret_cast<float4*>(a.out + (size_t)ks * a.slice + at) = c;
      }
    }
  }
}

// ------------------------------------------------------------ choice of tile
// Estimated us of a launch in which every CU runs r = ceil(tiles * ks / 256)
// workgroups over u 64-byte units of K each: fix + r * round + u * (lat +
// (r - 1) * thr) (lat: a unit alone on a CU, thr: one more beside it).  The
// constants are fitted to measured times (M = 7 .. 4700 over the GEMM shapes
// of both trunks, K in 1 to 16 slices, rms error 3-15%); the tile with the
// smallest estimate is within 6% of the fastest one on nearly all of them.
// The extra traffic of K slices goes to whoever adds them up (~6 TB/s, and
// ~0.1 us per slice for its loads).  E.g. BF16 4700 x 4096 x 1024: 192 x 256
// tiles 94 us, 128 x 256 112 us (25 x 16 tiles are two rounds of the 256 CUs,
// 37 x 16 three); 58 x 1024 x 3072: 64 x 64 tiles in 16
// slices 5.3 us, in one 38 us.
struct GemmTile { int bm, bn; float fix, round, lat, thr; bool swiglu; };
constexpr GemmTile GEMM_BF16[] = {
    {256, 256, 2.9f, 11.9f, 1.333f, 1.528f, true}, {192, 256, 3.6f, 10.2f, 1.058f, 1.224f, true},
    {160, 256, 4.2f, 6.9f, 1.086f, 1.171f, true},  {128, 256, 2.1f, 8.3f, .856f, .922f, true},
    {96, 256, 3.7f, 6.4f, .847f, .848f, true},     {128, 128, 0.f, 4.4f, .584f, .715f, true},
    {64, 128, 1.4f, 2.2f, .399f, .451f, true},     {32, 128, 1.7f, 1.2f, .315f, .321f, true},
    {64, 64, 2.1f, .7f, .300f, .341f, true},       {32, 64, 1.9f, .6f, .206f, .217f, true}};
constexpr GemmTile GEMM_F32[] = {{64, 64, 2.f, 1.1f, .398f, .199f, true},
                                 {48, 64, 2.3f, .6f, .312f, .180f, false},   // one column tile per wave
                                 {64, 32, 2.6f, 0.f, .243f, .209f, true},
                                 {32, 64, 2.5f, .3f, .250f, .208f, true},
                                 {32, 32, 3.f, 0.f, .246f, .088f, true}};
constexpr int GEMM_MAX_SPLIT = 16;

struct GemmPlan { int tile, ksplit; };
inline GemmPlan plan_gemm(bool bf16, bool swiglu, int M, int N, int K, int max_split) {
  GemmPlan best{0, 1};
  float bt = 1e30f;
  const int nt = bf16 ? (int)(sizeof(GEMM_BF16) / sizeof(GemmTile)) : (int)(sizeof(GEMM_F32) / sizeof(GemmTile));
  const int units = (K * (bf16 ? 2 : 4) + 63) / 64;
  for (int t = 0; t < nt; ++t) {
    const GemmTile g = bf16 ? GEMM_BF16[t] : GEMM_F32[t];
    if (swiglu && !g.swiglu) continue;
    const int nc = swiglu ? g.bn / 2 : g.bn;
    const long tiles = (long)((M + g.bm - 1) / g.bm) * ((N + nc - 1) / nc);
    for (int ks : {1, 2, 3, 4, 6, 8, 12, 16}) {
      if (ks > 1 && (ks > max_split || units < 4 * ks)) break;   // (short K: one slice, of the tile that fits M and N)
      const long rounds = (tiles * ks + 255) / 256;
      const float us = g.fix + rounds * g.round + ((units + ks - 1) / ks) * (g.lat + (rounds - 1) * g.thr) +
                       (ks - 1) * ((float)M * N * 8e-6f / 6.f + .1f);
      if (us < bt) { bt = us; best = GemmPlan{t, ks}; }
    }
  }
  return best;
}

template <int EPI, typename WL, int BM, int BN, int WM, int WN, int S, int H>
static hipError_t launch_gemm_t(GemmArgs a, hipStream_t st) {
  constexpr int NC = EPI == GEPI_SWIGLU ? BN / 2 : BN;
  a.mt = (a.M + BM - 1) / BM;
  a.nt = (a.N + NC - 1) / NC;
  a.gm = 8;
  const int tiles = a.mt * a.nt * a.ksplit;
  hipLaunchKernelGGL((gemm_kernel<EPI, WL, BM, BN, WM, WN, S, H>), dim3((tiles + 7) / 8 * 8), dim3(WM * WN * 64), 0,
                     st, a);
  return hipGetLastError();
}
template <int EPI>
static hipError_t launch_gemm(bool bf16, int tile, const GemmArgs& a, hipStream_t st) {
  if (!bf16) {
    switch (tile) {
      case 0: return launch_gemm_t<EPI, WF32, 64, 64, 2, 2, 3, 1>(a, st);
      case 1:
        if constexpr (EPI == GEPI_STORE) return launch_gemm_t<EPI, WF32, 48, 64, 1, 4, 3, 1>(a, st);
        else return hipErrorInvalidConfiguration;   // not planned
      case 2: return launch_gemm_t<EPI, WF32, 64, 32, 4, 1, 4, 1>(a, st);
      case 3: return launch_gemm_t<EPI, WF32, 32, 64, 2, 2, 4, 1>(a, st);
      default: return launch_gemm_t<EPI, WF32, 32, 32, 2, 1, 6, 1>(a, st);
    }
  }
  switch (tile) {
    case 0: return launch_gemm_t<EPI, WBF16, 256, 256, 4, 2, 3, 1>(a, st);
    case 1: return launch_gemm_t<EPI, WBF16, 192, 256, 2, 4, 3, 1>(a, st);
    case 2: return launch_gemm_t<EPI, WBF16, 160, 256, 2, 4, 3, 1>(a, st);
    case 3: return launch_gemm_t<EPI, WBF16, 128, 256, 2, 4, 4, 1>(a, st);
    case 4: return launch_gemm_t<EPI, WBF16, 96, 256, 2, 4, 4, 1>(a, st);
    case 5: return launch_gemm_t<EPI, WBF16, 128, 128, 2, 2, 3, 1>(a, st);
    case 6: return launch_gemm_t<EPI, WBF16, 64, 128, 2, 2, 4, 1>(a, st);
    case 7: return launch_gemm_t<EPI, WBF16, 32, 128, 2, 2, 5, 1>(a, st);
    case 8: return launch_gemm_t<EPI, WBF16, 64, 64, 2, 2, 4, 1>(a, st);
    default: return launch_gemm_t<EPI, WBF16, 32, 64, 2, 2, 4, 2>(a, st);
  }
}

}  // namespace sk
