// Batched prefill kernels: every prefix token of every row goes through the
// trunk at once (model.py:623-656 over Qwen3Model.forward,
// modeling_qwen3.py:367-427).  Tokens are packed row after row: token m is
// row tok_row[m] at position tok_pos[m]; row r's tokens start at row_start[r].
//
//   X = prefix embeddings -> per layer: Xn = RMSNorm(X); QKV = Xn Wqkv^T (MFMA GEMM,
//   sk_gemm.h); QK-norm + RoPE, K/V written into the decode cache; causal
//   attention per row; P = Att Wo^T; X += P, Xn = RMSNorm(X); Act = silu(Xn
//   Wg^T) * (Xn Wu^T); P = Act Wd^T, added to X by the next norm -> hidden =
//   RMSNorm_final(X[last token of each row]).  P and QKV may come in K slices,
//   summed by their reader in slice order.
//
// GEMM tiles and K slices and the attention's key split are chosen by the tokens
// of the whole call, so a row's results depend on the rows beside it in their
// last bits (order of sums), and in nothing else.
#pragma once

#include <hip/hip_runtime.h>

#include <type_traits>

#include "sk_gemm.h"
#include "sk_kernels.h"

namespace sk {

// ------------------------------------------------------------ prefix embeddings
// X[m] for every packed token: src[m] >= 0 a text id (language rows replaced,
// model.py:326-338), else frame -1 - src[m] of codes [frames][Q]: scale *
// sum_q table[q, code q], in q order (model.py:105-114).  One launch for all
// rows, 8 table rows in flight per thread; each row used to be embedded by a
// launch of its own (20-60 us: its 16 table rows one after another), copied in
// and waited for when it was staged.
template <typename TL>
__global__ __launch_bounds__(NT) void pf_embed_kernel(const int* src, const int* codes, const void* embed,
                                                      const float* lang_table, int n_lang, int l0, int l1, int l2,
                                                      int l3, const void* table, int Q, int V, int D, float scale,
                                                      float* X) {
  const int m = blockIdx.x, id = src[m];
  for (int k = threadIdx.x * 4; k < D; k += NT * 4) {
    float e[4];
    if (id >= 0) {
      const int lj = n_lang == 0 ? -1 : id == l0 ? 0 : id == l1 ? 1 : id == l2 ? 2 : id == l3 ? 3 : -1;
      if (lj >= 0) {
        const float4 t = *reinterpret_cast<const float4*>(lang_table + (size_t)lj * D + k);
        e[0] = t.x; e[1] = t.y; e[2] = t.z; e[3] = t.w;
      } else {
        RowPiece<TL, 4> t;
        t.load(embed, (size_t)id * D + k);
#pragma unroll
        for (int i = 0; i < 4; ++i) e[i] = t.get(i);
      }
    } else {
      const int* c = codes + (size_t)(-1 - id) * Q;
#pragma unroll
      for (int i = 0; i < 4; ++i) e[i] = 0.f;
      for (int j0 = 0; j0 < Q; j0 += 8) {
        RowPiece<TL, 4> t[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          const int q = min(j0 + j, Q - 1);
          t[j].load(table, ((size_t)q * V + c[q]) * D + k);
        }
#pragma unroll
        for (int j = 0; j < 8; ++j)
          if (j0 + j < Q) {
#pragma unroll
            for (int i = 0; i < 4; ++i) e[i] = j0 + j == 0 ? t[j].get(i) : __fadd_rn(e[i], t[j].get(i));
          }
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) e[i] = __fmul_rn(e[i], scale);
    }
    *reinterpret_cast<float4*>(X + (size_t)m * D + k) = make_float4(e[0], e[1], e[2], e[3]);
  }
}

// ------------------------------------------------------------ residual + norm
// Token m: x = residual X[m] + the ns K slices of the GEMM before it (P, in
// slice order; ns = 0: that GEMM added to X itself), written back to X; Xn =
// RMSNorm(x) in the form the next GEMM takes (FP32, or BF16 hi / lo planes).
// The slices' sum lives here because this kernel reads x anyway: a GEMM cut
// into slices costs no launch of its own.  NCH: float4 of the row per thread,
// kept in registers (0: any D, the row is read back for the norm).
template <bool BF, int NCH>
__global__ __launch_bounds__(NT) void pf_norm_kernel(const float* P, int ns, size_t slice, const float* w, float eps,
                                                     int D, float* X, float* Xn, uint16_t* xs, size_t xs_lo) {
  __shared__ float red[WAVES];
  const int m = blockIdx.x, tid = threadIdx.x, D4 = D / 4;
  const float4* pp = reinterpret_cast<const float4*>(P) + (size_t)m * D4;
  float4* xo = reinterpret_cast<float4*>(X) + (size_t)m * D4;
  auto load = [&](int k) {
    float4 x = xo[k];
    float4 p[4];
    for (int s0 = 0; s0 < ns; s0 += 4) {
#pragma unroll
      for (int j = 0; j < 4; ++j) p[j] = pp[(size_t)min(s0 + j, ns - 1) * (slice / 4) + k];
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if (s0 + j < ns) { x.x += p[j].x; x.y += p[j].y; x.z += p[j].z; x.w += p[j].w; }
    }
    return x;
  };
  auto put = [&](int k, const float4 x, float inv) {
    const float4 g = reinterpret_cast<const float4*>(w)[k];
    const float4 y = make_float4(g.x * (x.x * inv), g.y * (x.y * inv), g.z * (x.z * inv), g.w * (x.w * inv));
    if constexpr (BF) {
      uint2 hi, lo;
      split4(y, hi, lo);
      uint16_t* o = xs + (size_t)m * D + 4 * k;
      *reinterpret_cast<uint2*>(o) = hi;
      *reinterpret_cast<uint2*>(o + xs_lo) = lo;
    } else {
      reinterpret_cast<float4*>(Xn)[(size_t)m * D4 + k] = y;
    }
  };
  float s = 0.f;
  if constexpr (NCH > 0) {
    float4 x[NCH];
#pragma unroll
    for (int c = 0; c < NCH; ++c) {
      const int k = tid + c * NT;
      x[c] = load(min(k, D4 - 1));
      if (k < D4) {
        if (ns) xo[k] = x[c];
        s += x[c].x * x[c].x + x[c].y * x[c].y + x[c].z * x[c].z + x[c].w * x[c].w;
      }
    }
    const float inv = 1.0f / sqrtf(block_sum(s, red) / (float)D + eps);
#pragma unroll
    for (int c = 0; c < NCH; ++c)
      if (tid + c * NT < D4) put(tid + c * NT, x[c], inv);
  } else {
    for (int k = tid; k < D4; k += NT) {
      const float4 x = load(k);
      if (ns) xo[k] = x;
      s += x.x * x.x + x.y * x.y + x.z * x.z + x.w * x.w;
    }
    const float inv = 1.0f / sqrtf(block_sum(s, red) / (float)D + eps);
    for (int k = tid; k < D4; k += NT) put(k, xo[k], inv);   // this thread's own stores
  }
}

// ------------------------------------------------------------ per-token kernels
// (cos, sin) of positions 0..n-1 (rope_cs), one block per position.
__global__ __launch_bounds__(NT) void pf_rope_table_kernel(const float* inv_freq, int half, float2* tab) {
  const int p = blockIdx.x;
  for (int t = threadIdx.x; t < half; t += NT) tab[(size_t)p * half + t] = rope_cs(p, inv_freq[t]);
}

// Token m: q, k, v = the sum of the projection's ns K slices; per-head RMSNorm
// of q and k (gains qn_w / kn_w), rotate-half RoPE at the token's position,
// q -> Q[m][Hq][hd]; k, v -> this layer's cache at (row, kv head, position),
// rounded to BF16 when KT is.  A wave takes every 4th head, 8 at a time with
// their loads issued together; lane i holds dims i and i + hd / 2, so the
// rotation is lane-local.  Bound by its bytes (4700 tokens: 39 us when each
// head waited for its own loads, 26 us now).
template <typename KT>
__global__ __launch_bounds__(NT) void pf_qkv_kernel(const float* qkv, int ldqkv, int ns, size_t slice,
                                                    const int* tok_row, const int* tok_pos, const float* qn_w,
                                                    const float* kn_w, float eps, const float2* rope_tab, int Hq,
                                                    int Hkv, int hd, int max_ctx, float* Q, KT* kc, KT* vc) {
  const int m = blockIdx.x;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int half = hd / 2, H = Hq + 2 * Hkv, i = min(lane, half - 1);
  const bool live = lane < half;
  const int r = tok_row[m], p = tok_pos[m];
  const float* row = qkv + (size_t)m * ldqkv + i;
  const float2 cs = rope_tab[(size_t)p * half + i];
  const float wq1 = qn_w[i], wq2 = qn_w[i + half], wk1 = kn_w[i], wk2 = kn_w[i + half];
  constexpr int U = 8;
  for (int h0 = wave; h0 < H; h0 += U * WAVES) {
    float a[U], b[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const float* src = row + (size_t)min(h0 + u * WAVES, H - 1) * hd;
      a[u] = src[0];
      b[u] = src[half];
    }
    for (int s = 1; s < ns; ++s) {
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const float* src = row + s * slice + (size_t)min(h0 + u * WAVES, H - 1) * hd;
        a[u] += src[0];
        b[u] += src[half];
      }
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int h = h0 + u * WAVES;
      if (h >= H) break;
      float y1 = a[u], y2 = b[u];
      if (h < Hq + Hkv) {
        const bool isq = h < Hq;
        const float ss = wave_sum_dpp(live ? y1 * y1 + y2 * y2 : 0.f);
        const float inv = 1.0f / sqrtf(ss / (float)hd + eps);
        const float x1 = (isq ? wq1 : wk1) * (y1 * inv), x2 = (isq ? wq2 : wk2) * (y2 * inv);
        y1 = x1 * cs.x - x2 * cs.y;
        y2 = x2 * cs.x + x1 * cs.y;
      }
      if (!live) continue;
      if (h < Hq) {
        float* dq = Q + ((size_t)m * Hq + h) * hd;
        dq[i] = y1;
        dq[i + half] = y2;
      } else {
        const int kh = h < Hq + Hkv ? h - Hq : h - Hq - Hkv;
        KT* dst = (h < Hq + Hkv ? kc : vc) + (((size_t)r * Hkv + kh) * max_ctx + p) * hd;
        if constexpr (sizeof(KT) == 2) { dst[i] = (KT)bf16_bits(y1); dst[i + half] = (KT)bf16_bits(y2); }
        else { dst[i] = y1; dst[i + half] = y2; }
      }
    }
  }
}

// ------------------------------------------------------------ causal attention
// The workgroup holds PF_NQ = 32 query vectors (two MFMA tiles of 16): the G
// heads of kv head h for 32 / G consecutive positions of row r.  Its WK waves
// share the keys up to the last query position, 16 at a time (wave w takes
// tiles w, w + WK, ...), each with its own online softmax; the partial
// outputs meet in LDS at the end.  No barrier and no LDS inside the loop:
//   S^T = K Q^T on the FP32 matrix cores (v_mfma_f32_16x16x4f32): lane l holds
//     the scores of query l % 16 for keys 4 (l / 16) + v, v < 4;
//   the softmax of a query is 4 values per lane and two exchanges between
//     lanes 16 and 32 apart;
//   O^T += V^T P^T takes those four values as they are: step v multiplies the
//     keys 4 q + v, q = 0 .. 3, of P (this lane's) and V (row 4 q + v).
// K and V come straight from the cache just written (BF16 widened), 16 bytes
// per lane, V of a tile in flight under S, the next K under the softmax and
// PV.  A K load gives dims KW q + e of key l % 16 to lane l (q = l / 16), a V
// load dims VW i + e of keys 4 q + v to lane i + 16 q; Q is loaded in K's
// order, and O's rows come out in V's.
//
// What bounds it: FP32 MFMA time (50% of the kernel at 1,314 tokens of one row,
// 30% at 32 rows of 60-240, 11% at 241 + 146) with the
// softmax, rescaling and merge arithmetic beside it; workgroups with the
// longest walk start first.  Tried: K of the next tile loaded under a branch or
// past the end of the keys (PV then waits for it, 29 -> 40 us on the pair
// below).  us per layer before (32 queries per workgroup through LDS, four
// barriers per 32 keys) -> now: 1314 tokens, 1.7B 224 -> 92; 241 + 146 tokens
// 34 -> 17.5; 32 rows of 60-240 tokens, BF16 cache 133 -> 73.
constexpr int PF_NQ = 32;

template <typename KT, int HD>
struct PfAttDims {
  static constexpr int KW = (16 / (int)sizeof(KT)) < HD / 4 ? 16 / (int)sizeof(KT) : HD / 4;   // dims per K load
  static constexpr int NK = HD / (4 * KW);                                                     // K loads per tile
  static constexpr int NDT = HD / 16;                                                          // 16-dim output tiles
  static constexpr int VW = (16 / (int)sizeof(KT)) < NDT ? 16 / (int)sizeof(KT) : NDT;         // dims per V load
  static constexpr int NV = NDT / VW;                                                          // V loads per key row
  static constexpr int LDO = HD + 4;                                                           // merge row stride
};
template <typename KT, int HD>
constexpr size_t pf_attn_smem(int wk) {   // bytes: partial outputs, then (max, sum) per wave and query
  return ((size_t)wk * PF_NQ * PfAttDims<KT, HD>::LDO + 2 * (size_t)wk * PF_NQ) * sizeof(float);
}

// N consecutive cache elements as loaded; get<i>() widens one to FP32 (kept
// packed until used: half the registers with BF16).
template <typename KT, int N>
struct KvPiece {
  uint32_t w[(N * sizeof(KT) + 3) / 4];
  __device__ __forceinline__ void load(const KT* base, unsigned off) {   // off in bytes
    const char* p = reinterpret_cast<const char*>(base) + off;
    if constexpr (N * sizeof(KT) == 16) {
      const uint4 v = *reinterpret_cast<const uint4*>(p);
      w[0] = v.x; w[1] = v.y; w[2] = v.z; w[3] = v.w;
    } else if constexpr (N * sizeof(KT) == 8) {
      const uint2 v = *reinterpret_cast<const uint2*>(p);
      w[0] = v.x; w[1] = v.y;
    } else if constexpr (N * sizeof(KT) == 4) {
      w[0] = *reinterpret_cast<const uint32_t*>(p);
    } else {
      w[0] = *reinterpret_cast<const uint16_t*>(p);
    }
  }
  __device__ __forceinline__ float get(int i) const {
    if constexpr (sizeof(KT) == 4) return __uint_as_float(w[i]);
    else return __uint_as_float(i & 1 ? w[i / 2] & 0xffff0000u : w[i / 2] << 16);
  }
};

template <typename KT, int HD, int WK, bool BF>
__global__ __launch_bounds__(WK * 64) __attribute__((amdgpu_waves_per_eu(2, 2))) void pf_attention_kernel(
    const float* Q, const KT* kc, const KT* vc, const int* row_start, const int* len, int Hq, int Hkv, int max_ctx,
    float scale, float* out, int ldo, uint16_t* xs, size_t xs_lo) {
  using D = PfAttDims<KT, HD>;
  constexpr int KW = D::KW, NK = D::NK, NDT = D::NDT, VW = D::VW, NV = D::NV, LDO = D::LDO;
  extern __shared__ __attribute__((aligned(16))) float psm[];
  const int G = Hq / Hkv, QB = PF_NQ / G;
  const int h = blockIdx.x % Hkv, r = blockIdx.x / Hkv;
  const int n = len[r], p0 = (int)(gridDim.y - 1 - blockIdx.y) * QB;
  if (p0 >= n) return;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int i16 = lane & 15, q4 = lane >> 4;
  const int m0 = row_start[r], last_p = min(p0 + QB, n) - 1;
  const KT* kb = kc + ((size_t)r * Hkv + h) * max_ctx * HD;
  const KT* vb = vc + ((size_t)r * Hkv + h) * max_ctx * HD;
  // query vector qv = g * QB + t: head h * G + g at position p0 + t
  int qp[2];
  float qf[2][NK * KW];
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int qv = j * 16 + i16, g = qv / QB;
    qp[j] = p0 + qv - g * QB;
    const float* qr = Q + ((size_t)(m0 + min(qp[j], n - 1)) * Hq + h * G + g) * HD;
#pragma unroll
    for (int t = 0; t < NK; ++t)
#pragma unroll
      for (int e = 0; e < KW; e += 4) {
        const float4 v = *reinterpret_cast<const float4*>(qr + t * 4 * KW + KW * q4 + e);
        qf[j][t * KW + e] = v.x; qf[j][t * KW + e + 1] = v.y; qf[j][t * KW + e + 2] = v.z; qf[j][t * KW + e + 3] = v.w;
      }
  }
  KvPiece<KT, KW> kf[NK];
  KvPiece<KT, VW> vf[4][NV];
  auto load_k = [&](int k0) {
    const unsigned p = (unsigned)(min(k0 + i16, n - 1) * HD + KW * q4) * sizeof(KT);
#pragma unroll
    for (int t = 0; t < NK; ++t) kf[t].load(kb, p + t * 4 * KW * sizeof(KT));
  };
  auto load_v = [&](int k0) {
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const unsigned p = (unsigned)(min(k0 + 4 * q4 + v, n - 1) * HD + VW * i16) * sizeof(KT);
#pragma unroll
      for (int t = 0; t < NV; ++t) vf[v][t].load(vb, p + t * 16 * VW * sizeof(KT));
    }
  };
  v4f o[2][NDT];
#pragma unroll
  for (int j = 0; j < 2; ++j)
#pragma unroll
    for (int t = 0; t < NDT; ++t) o[j][t] = v4f{0.f, 0.f, 0.f, 0.f};
  float mr[2] = {-INFINITY, -INFINITY}, lr[2] = {0.f, 0.f};
  const int k_first = wave * 16;
  // one tile; `next`: the K of the wave's next tile is loaded on the way (a
  // template argument: with a branch the compiler would make PV wait for those
  // loads too)
  auto tile = [&](int k0, auto next) {
    load_v(k0);
    v4f s[2] = {v4f{0.f, 0.f, 0.f, 0.f}, v4f{0.f, 0.f, 0.f, 0.f}};
#pragma unroll
    for (int t = 0; t < NK; ++t)
#pragma unroll
      for (int e = 0; e < KW; ++e) {
        const float k = kf[t].get(e);
#pragma unroll
        for (int j = 0; j < 2; ++j) s[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(k, qf[j][t * KW + e], s[j], 0, 0, 0);
      }
    if constexpr (decltype(next)::value) load_k(k0 + WK * 16);
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      float mx = -INFINITY;
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int key = k0 + 4 * q4 + v;
        s[j][v] = key <= qp[j] && key < n ? s[j][v] * scale : -INFINITY;
        mx = fmaxf(mx, s[j][v]);
      }
      mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
      mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
      const float mn = fmaxf(mr[j], mx);
      const bool none = mn == -INFINITY;         // every key so far is masked for this query
      const float sc = none ? 1.f : expf(mr[j] - mn);
      float sum = 0.f;
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        s[j][v] = none ? 0.f : expf(s[j][v] - mn);
        sum += s[j][v];
      }
      lr[j] = lr[j] * sc + sum;                  // this lane's keys; the four lanes of a query add up at the end
      mr[j] = mn;
      if (__any(sc != 1.f)) {                    // some query's maximum moved
#pragma unroll
        for (int t = 0; t < NDT; ++t) o[j][t] *= sc;
      }
    }
#pragma unroll
    for (int v = 0; v < 4; ++v)
#pragma unroll
      for (int t = 0; t < NV; ++t)
#pragma unroll
        for (int e = 0; e < VW; ++e) {
          const float x = vf[v][t].get(e);
#pragma unroll
          for (int j = 0; j < 2; ++j)
            o[j][t * VW + e] = __builtin_amdgcn_mfma_f32_16x16x4f32(x, s[j][v], o[j][t * VW + e], 0, 0, 0);
        }
  };
  if (k_first <= last_p) {
    load_k(k_first);
    int k0 = k_first;
    for (; k0 + WK * 16 <= last_p; k0 += WK * 16) tile(k0, std::true_type{});
    tile(k0, std::false_type{});
  }
  // merge: every wave's partial output rows and (max, sum) per query
  float* po = psm;                               // [WK][NQ][LDO]
  float* pm = psm + WK * PF_NQ * LDO;            // [WK][NQ] max, then [WK][NQ] sum
  float* pl = pm + WK * PF_NQ;
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    float l = lr[j];
    l += __shfl_xor(l, 16, 64);
    l += __shfl_xor(l, 32, 64);
    if (q4 == 0) { pm[wave * PF_NQ + j * 16 + i16] = mr[j]; pl[wave * PF_NQ + j * 16 + i16] = l; }
    float* row = po + (size_t)(wave * PF_NQ + j * 16 + i16) * LDO;
#pragma unroll
    for (int t = 0; t < NV; ++t)
#pragma unroll
      for (int v = 0; v < 4; ++v) {              // rows 4 q + v of tile (t, e): dim 16 VW t + VW (4 q + v) + e
        float* d = row + 16 * VW * t + VW * (4 * q4 + v);
        if constexpr (VW % 4 == 0) {
#pragma unroll
          for (int e = 0; e < VW; e += 4)
            *reinterpret_cast<float4*>(d + e) = make_float4(o[j][t * VW + e][v], o[j][t * VW + e + 1][v],
                                                            o[j][t * VW + e + 2][v], o[j][t * VW + e + 3][v]);
        } else {
#pragma unroll
          for (int e = 0; e < VW; ++e) d[e] = o[j][t * VW + e][v];
        }
      }
  }
  __syncthreads();
  if (tid < PF_NQ) {                             // each wave's factor for query tid, in place of its max
    float mx = -INFINITY, l = 0.f, f[WK];
#pragma unroll
    for (int w = 0; w < WK; ++w) mx = fmaxf(mx, pm[w * PF_NQ + tid]);   // finite: key 0 is wave 0's
#pragma unroll
    for (int w = 0; w < WK; ++w) {
      f[w] = expf(pm[w * PF_NQ + tid] - mx);
      l = fmaf(f[w], pl[w * PF_NQ + tid], l);
    }
#pragma unroll
    for (int w = 0; w < WK; ++w) pm[w * PF_NQ + tid] = f[w] / l;
  }
  __syncthreads();
  constexpr int NF = HD / 4;                     // float4 per output row
  for (int it = tid; it < PF_NQ * NF; it += WK * 64) {
    const int qv = it / NF, d = (it - qv * NF) * 4, g = qv / QB, pos = p0 + qv - g * QB;
    if (pos >= n) continue;
    float4 y = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
    for (int w = 0; w < WK; ++w) {
      const float wt = pm[w * PF_NQ + qv];
      const float4 x = *reinterpret_cast<const float4*>(po + (size_t)(w * PF_NQ + qv) * LDO + d);
      y.x = fmaf(wt, x.x, y.x); y.y = fmaf(wt, x.y, y.y); y.z = fmaf(wt, x.z, y.z); y.w = fmaf(wt, x.w, y.w);
    }
    const size_t at = (size_t)(m0 + pos) * ldo + (size_t)(h * G + g) * HD + d;
    if constexpr (BF) {                          // the O projection's input: BF16 hi and lo planes
      uint2 hi, lo;
      split4(y, hi, lo);
      *reinterpret_cast<uint2*>(xs + at) = hi;
      *reinterpret_cast<uint2*>(xs + at + xs_lo) = lo;
    } else {
      *reinterpret_cast<float4*>(out + at) = y;
    }
  }
}

// Row r after its prefix: hidden = RMSNorm_final(X[last token] + the last down
// projection's K slices); kv_len and
// position = prefix length, RoPE (cos, sin) at that position, row active; the
// first depth step's input abuf = RMSNorm_in(hidden) (and its split form).
// Rows with no tokens in this prefill keep their state.
__global__ __launch_bounds__(NT) void pf_finish_kernel(float* X, const float* P, int ns, size_t slice,
                                                       const int* row_start, const int* len,
                                                       const float* w, float eps, int D, float* hidden,
                                                       int* kv_len, int* pos, int* active, const float* inv_freq,
                                                       int half, float2* rope, const float* w_in, float eps_in,
                                                       float* abuf, uint16_t* xs_abuf) {
  __shared__ float red[WAVES];
  const int r = blockIdx.x;
  const int n = len[r];
  if (n == 0) return;                    // not in this prefill: the row keeps its state
  float* xr = X + (size_t)(row_start[r] + n - 1) * D;
  const float* pr = P + (size_t)(row_start[r] + n - 1) * D;
  const size_t ro = (size_t)r * D;
  float s = 0.f;
  for (int k = threadIdx.x; k < D; k += NT) {
    float x = xr[k];
    for (int q = 0; q < ns; ++q) x += pr[q * slice + k];
    if (ns) xr[k] = x;                   // read back by this thread below
    s += x * x;
  }
  const float inv = 1.0f / sqrtf(block_sum(s, red) / (float)D + eps);
  float s2 = 0.f;
  for (int k = threadIdx.x; k < D; k += NT) {
    const float h = w[k] * (xr[k] * inv);
    hidden[ro + k] = h;
    s2 = fmaf(h, h, s2);
  }
  // The first frame's depth step 0 input, RMSNorm_in(hidden) (zero prefix).
  const float inv2 = 1.0f / sqrtf(block_sum(s2, red) / (float)D + eps_in);
  for (int k = threadIdx.x; k < D; k += NT) {
    const float y = w_in[k] * (hidden[ro + k] * inv2);
    abuf[ro + k] = y;
    if (xs_abuf) xsplit_store(xs_abuf, r, k, y);
  }
  for (int t = threadIdx.x; t < half; t += NT) rope[(size_t)r * half + t] = rope_cs(n, inv_freq[t]);
  if (threadIdx.x == 0) { kv_len[r] = n; pos[r] = n; active[r] = 1; }
}

}  // namespace sk
