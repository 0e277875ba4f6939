// Batched prefill kernels: every prefix token of every row goes through the
// trunk at once (model.py:623-656 over Qwen3Model.forward,
// modeling_qwen3.py:367-427).  Tokens are packed row after row: token m is
// row tok_row[m] at position tok_pos[m]; row r's tokens start at row_start[r].
//
//   X = embeds -> per layer: Xn = RMSNorm(X); QKV = Xn Wqkv^T (MFMA GEMM,
//   sk_gemm.h); QK-norm + RoPE, K/V written into the decode cache; causal
//   attention per row; P = Att Wo^T; X += P, Xn = RMSNorm(X); Act = silu(Xn
//   Wg^T) * (Xn Wu^T); P = Act Wd^T, added to X by the next norm -> hidden =
//   RMSNorm_final(X[last token of each row]).  P and QKV may come in K slices,
//   summed by their reader in slice order.
#pragma once

#include <hip/hip_runtime.h>

#include "sk_gemm.h"
#include "sk_kernels.h"

namespace sk {

// ------------------------------------------------------------ residual + norm
// Token m: x = residual + the ns K slices of the GEMM before it (P, in slice
// order; ns = 0: that GEMM added to X itself), written back to X; Xn =
// RMSNorm(x) in the form the next GEMM takes (FP32, or BF16 hi / lo planes).
// The slices' sum lives here because this kernel reads x anyway: a GEMM cut
// into slices costs no launch of its own.  The residual is X[m], or for the
// first layer (embeds != null) the prefix embedding of the token.  NCH: float4
// of the row per thread, kept in registers (0: any D, the row is read back for
// the norm).
template <bool BF, int NCH>
__global__ __launch_bounds__(NT) void pf_norm_kernel(const float* embeds, int max_ctx, const int* tok_row,
                                                     const int* tok_pos, const float* P, int ns, size_t slice,
                                                     const float* w, float eps, int D, float* X, float* Xn,
                                                     uint16_t* xs, size_t xs_lo) {
  __shared__ float red[WAVES];
  const int m = blockIdx.x, tid = threadIdx.x, D4 = D / 4;
  const float4* src = reinterpret_cast<const float4*>(
      embeds ? embeds + ((size_t)tok_row[m] * max_ctx + tok_pos[m]) * D : X + (size_t)m * D);
  const float4* pp = reinterpret_cast<const float4*>(P) + (size_t)m * D4;
  float4* xo = reinterpret_cast<float4*>(X) + (size_t)m * D4;
  const bool keep = ns > 0 || embeds;        // x differs from X[m]
  auto load = [&](int k) {
    float4 x = src[k];
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
        if (keep) xo[k] = x[c];
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
      if (keep) xo[k] = x;
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
// head waited for its own loads).
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
// Grid (query blocks, Hkv, rows); the workgroup holds PF_NQ = 32 query
// vectors: the G heads of kv head h for QB = 32 / G consecutive positions of
// the row, and walks the row's keys 0 .. (last query position) in chunks of
// 32 with an online softmax (scale hd^-1/2, keys after the query masked).
// Per chunk: S = Q K^T on the matrix cores (one 16 x 16 tile per wave, Q
// fragments kept in registers), softmax over each query's 32 scores by 8
// threads (DPP all-reduce), O += P V on the matrix cores.  K / V come from
// the cache just written (BF16 widened), so attention sees exactly what
// decode steps will see.
constexpr int PF_NQ = 32, PF_KC = 32;

__host__ __device__ constexpr int pf_ldk(int hd) { return hd + 2; }    // lanes 0-15: 16 rows, 2 banks apart
__host__ __device__ constexpr int pf_ldv(int hd) { return hd + 16; }   // lanes 16-31: next row, 16 banks on
constexpr int PF_LDS = PF_KC + 1;
__host__ __device__ constexpr size_t pf_attn_smem_floats(int hd) {
  return (size_t)PF_KC * pf_ldk(hd) + (size_t)PF_KC * pf_ldv(hd) + (size_t)PF_NQ * PF_LDS + 2 * (size_t)PF_NQ;
}

// all-reduce over each aligned group of 8 lanes
__device__ __forceinline__ float grp8_max(float v) {
  v = fmaxf(v, dpp_keep<0xb1, 0xf>(v));    // quad_perm [1,0,3,2]
  v = fmaxf(v, dpp_keep<0x4e, 0xf>(v));    // quad_perm [2,3,0,1]
  return fmaxf(v, dpp_keep<0x141, 0xf>(v));  // row_half_mirror: lane i <-> 7 - i
}
__device__ __forceinline__ float grp8_sum(float v) {
  v += dpp_keep<0xb1, 0xf>(v);
  v += dpp_keep<0x4e, 0xf>(v);
  return v + dpp_keep<0x141, 0xf>(v);
}

template <typename KT, bool BF>
__global__ __launch_bounds__(NT) void pf_attention_kernel(const float* Q, const KT* kc, const KT* vc,
                                                          const int* row_start, const int* len, int Hq, int Hkv,
                                                          int hd, int max_ctx, float scale, float* out, int ldo,
                                                          uint16_t* xs, size_t xs_lo) {
  extern __shared__ __attribute__((aligned(16))) float psm[];
  const int G = Hq / Hkv, QB = PF_NQ / G;
  const int qb = blockIdx.x, h = blockIdx.y, r = blockIdx.z;
  const int n = len[r];
  const int p0 = qb * QB;
  if (p0 >= n) return;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int ldk = pf_ldk(hd), ldv = pf_ldv(hd);
  float* Ks = psm;                              // [KC][ldk]
  float* Vs = Ks + PF_KC * ldk;                 // [KC][ldv]
  float* P = Vs + PF_KC * ldv;                  // [NQ][PF_LDS] scores, then probabilities
  float* Msc = P + PF_NQ * PF_LDS;              // [NQ] rescale of this chunk
  float* Ml = Msc + PF_NQ;                      // [NQ] final sums
  const size_t head_base = ((size_t)r * Hkv + h) * max_ctx;
  const int m0 = row_start[r];
  // query vector qv = g * QB + tq: head h * G + g at position p0 + tq
  auto qpos = [&](int qv) { return p0 + (qv - (qv / QB) * QB); };
  auto qhead = [&](int qv) { return h * G + qv / QB; };
  const int i16 = lane & 15, k4 = lane >> 4;
  // S tile of this wave: queries [16 qi, +16), keys [16 ki, +16)
  const int qi = wave >> 1, ki = wave & 1;
  float qf[32];                                 // A fragments over hd / 4 k-steps
  {
    const int qv = qi * 16 + i16;
    const int p = min(qpos(qv), n - 1);
    const float* qrow = Q + ((size_t)(m0 + p) * Hq + qhead(qv)) * hd;
#pragma unroll
    for (int ks = 0; ks < 32; ++ks) qf[ks] = (ks * 4 < hd) ? qrow[ks * 4 + k4] : 0.f;
  }
  // softmax role: query tid / 8, keys (tid % 8) * 4 .. + 4
  const int sq = tid >> 3, sk0 = (tid & 7) * 4;
  const int sp = qpos(sq);
  float m_run = -INFINITY, l_run = 0.f;
  // PV tiles of this wave: (query tile, d tile) pairs t = wave, wave + 4, ...
  const int ndt = hd / 16, ntile = 2 * ndt;
  v4f o[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) o[i] = v4f{0.f, 0.f, 0.f, 0.f};
  const int last_p = min(p0 + QB, n) - 1;
  // K / V chunk staging: groups of 4 dims, up to 4 per thread (hd <= 128),
  // loaded one chunk ahead into registers.
  const int q4 = hd / 4, n4 = PF_KC * q4;
  float4 kr[4], vr[4];
  auto fetch = [&](int k0) {
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int i = min(tid + u * NT, n4 - 1);
      const int j = i / q4, d = (i - j * q4) * 4;
      const size_t off = (head_base + min(k0 + j, n - 1)) * hd + d;
      if constexpr (sizeof(KT) == 2) {
        const uint2 kb = *reinterpret_cast<const uint2*>(kc + off);
        const uint2 vb = *reinterpret_cast<const uint2*>(vc + off);
        kr[u] = make_float4(__uint_as_float(kb.x << 16), __uint_as_float(kb.x & 0xffff0000u),
                            __uint_as_float(kb.y << 16), __uint_as_float(kb.y & 0xffff0000u));
        vr[u] = make_float4(__uint_as_float(vb.x << 16), __uint_as_float(vb.x & 0xffff0000u),
                            __uint_as_float(vb.y << 16), __uint_as_float(vb.y & 0xffff0000u));
      } else {   // built element-wise like the BF16 form, which keeps kr / vr in registers
        const float4 kb = *reinterpret_cast<const float4*>(kc + off);
        const float4 vb = *reinterpret_cast<const float4*>(vc + off);
        kr[u] = make_float4(kb.x, kb.y, kb.z, kb.w);
        vr[u] = make_float4(vb.x, vb.y, vb.z, vb.w);
      }
    }
  };
  fetch(0);
  for (int k0 = 0; k0 <= last_p; k0 += PF_KC) {
    __syncthreads();
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int i = tid + u * NT;
      if (i < n4) {
        const int j = i / q4, d = (i - j * q4) * 4;
        float2* kd = reinterpret_cast<float2*>(Ks + j * ldk + d);
        kd[0] = make_float2(kr[u].x, kr[u].y);
        kd[1] = make_float2(kr[u].z, kr[u].w);
        *reinterpret_cast<float4*>(Vs + j * ldv + d) = vr[u];
      }
    }
    __syncthreads();
    if (k0 + PF_KC <= last_p) fetch(k0 + PF_KC);
    // S tile = Q K^T
    {
      v4f sacc = v4f{0.f, 0.f, 0.f, 0.f};
      const float* kp = Ks + (ki * 16 + i16) * ldk + k4;
#pragma unroll
      for (int ks = 0; ks < 32; ++ks)
        if (ks * 4 < hd) sacc = __builtin_amdgcn_mfma_f32_16x16x4f32(qf[ks], kp[ks * 4], sacc, 0, 0, 0);
      const int key = k0 + ki * 16 + i16;
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int qv = qi * 16 + 4 * k4 + v;
        const int pq = qpos(qv);
        const bool ok = key <= pq && pq < n;
        P[qv * PF_LDS + ki * 16 + i16] = ok ? sacc[v] * scale : -INFINITY;
      }
    }
    __syncthreads();
    // online softmax of query sq over its 32 scores (8 threads, 4 each)
    {
      float sv[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) sv[j] = P[sq * PF_LDS + sk0 + j];
      const float mx = grp8_max(fmaxf(fmaxf(sv[0], sv[1]), fmaxf(sv[2], sv[3])));
      const float mn = fmaxf(m_run, mx);
      const bool none = (mn == -INFINITY);
      const float sc = none ? 1.f : expf(m_run - mn);
      float part = 0.f;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float e = none ? 0.f : expf(sv[j] - mn);
        P[sq * PF_LDS + sk0 + j] = e;
        part += e;
      }
      l_run = l_run * sc + grp8_sum(part);
      m_run = mn;
      if ((tid & 7) == 0) Msc[sq] = sc;
    }
    __syncthreads();
    // O = O * rescale + P V
#pragma unroll
    for (int t4 = 0; t4 < 4; ++t4) {
      const int t = wave + 4 * t4;
      if (t < ntile) {
        const int tq = t / ndt, td = t - tq * ndt;
#pragma unroll
        for (int v = 0; v < 4; ++v) o[t4][v] *= Msc[tq * 16 + 4 * k4 + v];
        const float* pp = P + (tq * 16 + i16) * PF_LDS + k4;
        const float* vp = Vs + k4 * ldv + td * 16 + i16;
#pragma unroll
        for (int ks = 0; ks < PF_KC / 4; ++ks)
          o[t4] = __builtin_amdgcn_mfma_f32_16x16x4f32(pp[ks * 4], vp[ks * 4 * ldv], o[t4], 0, 0, 0);
      }
    }
  }
  if ((tid & 7) == 0) Ml[sq] = l_run;
  __syncthreads();
#pragma unroll
  for (int t4 = 0; t4 < 4; ++t4) {
    const int t = wave + 4 * t4;
    if (t < ntile) {
      const int tq = t / ndt, td = t - tq * ndt;
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int qv = tq * 16 + 4 * k4 + v;
        const int pq = qpos(qv);
        if (pq < n) {
          const float y = o[t4][v] / Ml[qv];
          const size_t at = (size_t)(m0 + pq) * ldo + (size_t)qhead(qv) * hd + td * 16 + i16;
          if constexpr (BF) {   // the O projection's input: BF16 hi and lo planes
            const __bf16 hi = (__bf16)y;
            xs[at] = __builtin_bit_cast(uint16_t, hi);
            xs[at + xs_lo] = __builtin_bit_cast(uint16_t, (__bf16)(y - (float)hi));
          } else {
            out[at] = y;
          }
        }
      }
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
