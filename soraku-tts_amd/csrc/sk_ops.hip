// Operator API: the fused decode kernels one at a time, on a caller stream.
// Counterparts of the TileLang factories in
// soraku_inference/acceleration/tilelang_kernels.py (same operands and
// meaning; masking uses -inf as the native path does, model.py:582-584,
// instead of the -1e30 of tilelang_kernels.py:31).
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "sk_error.h"
#include "sk_kernels.h"
#include "sk_launch.h"
#include "sk_wide.h"
#include "soraku_mi355x.h"

using namespace sk;

namespace {

int check_wdtype(int32_t wdtype) {
  SK_CHECK(wdtype == SK_F32 || wdtype == SK_BF16, SK_EINVAL, "wdtype must be SK_F32 or SK_BF16");
  return SK_OK;
}

bool aligned16(const void* p) { return ((uintptr_t)p & 15) == 0; }

// A projection of B activation rows.  Up to 4 rows: the GEMV kernels.  More:
// 32 rows per launch on the FP32 matrix cores (skinny_kernel), where one pass
// over the weights serves them all (in chunks of 4 rows through the GEMV the
// weights are read B / 4 times).  us per launch, GEMV chunks / one pass: 4 rows,
// FP32 2051 x 1024 4.1 / 4.9; 7 rows BF16 2 x 6144 x 2048 34 / 16.4, 2048 x 6144
// 36 / 15; 20 rows FP32 2051 x 1024 20 / 7.4.
//
// 5 to 8 rows of few but long weight rows (K to 6,144, where measured) keep the
// two GEMV launches: they spread the rows over the GPU one or two per wave,
// where the one pass has a workgroup per 16 of them and takes as long as a CU
// needs to load those and x in 64-byte pieces (16 waves instead of 8 changed
// nothing).  From 8 KB per output on for 5 and 6 rows (7 and 8: 12 KB FP32, 16
// KB BF16), up to 1,536 outputs (1,024 of one matrix with K past 3,072) and 24
// MB of weights, which the second launch finds in cache; not BF16 with a bias,
// where one pass is faster.  FP32 1024 x 2048, 5 rows 6.5 / 7.6, 1024 x 3072 5
// rows 7.9 / 10.1, 8 rows 10.9 / 11.1, 512 x 4096 5 rows 8.9 / 12.5, 2 x 1024 x
// 2048 5 rows 7.9 / 11.8, 8 rows 10.9 / 12.4; BF16 2 x 1024 x 2048 5 rows 8.3 /
// 9.1, 1024 x 6144 5 rows 11.2 / 13.1.  Past those lines: FP32 2048 x 2048 5
// rows 10.6 / 8.1, 1024 x 1024 5.5 / 5.0, 2 x 1536 x 3072 8 rows 21.1 / 17.3,
// BF16 1024 x 2048 8 rows 9 / 5.7.
constexpr int ROWS_GEMV = 4;
template <int EPI>
bool rows_in_chunks(bool bf16, int B, int N, int K) {
  if (B <= ROWS_GEMV) return true;
  if (B > 2 * ROWS_GEMV || K > 6144 || (bf16 && EPI == EPI_BIAS)) return false;
  const size_t row = (size_t)K * (bf16 ? 2 : 4) * (EPI == EPI_SWIGLU ? 2 : 1);
  const int most = EPI != EPI_SWIGLU && K > 3072 ? 1024 : 1536;
  return row >= (B <= 6 ? 8192u : bf16 ? 16384u : 12288u) && N <= most && row * N <= (24u << 20);
}
template <int EPI>
int project_rows(hipStream_t st, int wdtype, int B, const GemvArgs& a) {
  if (rows_in_chunks<EPI>(wdtype == SK_BF16, B, a.N, a.K)) {
    for (int b0 = 0; b0 < B; b0 += ROWS_GEMV) {
      GemvArgs c = a;
      c.x = a.x + (size_t)b0 * a.ldx;
      c.out = a.out + (size_t)b0 * a.ldo;
      if (a.res) c.res = a.res + (size_t)b0 * a.ldr;
      SK_HIP((launch_gemv<PRO_NONE, EPI>(wdtype, B - b0 < ROWS_GEMV ? B - b0 : ROWS_GEMV, c, st)));
    }
    return SK_OK;
  }
  for (int b0 = 0; b0 < B; b0 += SK_ROWS) {
    SkinnyArgs k = skinny_args(a.w[0], a.N, a.K, a.x + (size_t)b0 * a.ldx, a.ldx, a.out + (size_t)b0 * a.ldo, a.ldo,
                               B - b0 < SK_ROWS ? B - b0 : SK_ROWS);
    k.w2 = a.w[1];
    k.bias = a.bias;
    if (a.res) { k.res = a.res + (size_t)b0 * a.ldr; k.ldr = a.ldr; }
    SK_HIP((launch_rows<EPI>(wdtype == SK_BF16, k, st)));
  }
  return SK_OK;
}

}  // namespace

extern "C" {

int sk_op_add_rmsnorm(void* stream, int32_t B, int32_t D, float eps, const float* hidden,
                      const float* prefix, const float* weight, float* out) {
  SK_CHECK(B > 0 && D > 0, SK_EINVAL, "B and D must be positive");
  SK_CHECK(hidden && prefix && weight && out, SK_EINVAL, "NULL operand");
  hipLaunchKernelGGL(rmsnorm_rows_kernel, dim3(B), dim3(NT), 0, (hipStream_t)stream, hidden, prefix,
                     weight, eps, D, out, nullptr);
  SK_HIP(hipGetLastError());
  return SK_OK;
}

int sk_op_rmsnorm(void* stream, int32_t B, int32_t D, float eps, const float* x, const float* weight,
                  float* out) {
  SK_CHECK(B > 0 && D > 0, SK_EINVAL, "B and D must be positive");
  SK_CHECK(x && weight && out, SK_EINVAL, "NULL operand");
  hipLaunchKernelGGL(rmsnorm_rows_kernel, dim3(B), dim3(NT), 0, (hipStream_t)stream, x, nullptr,
                     weight, eps, D, out, nullptr);
  SK_HIP(hipGetLastError());
  return SK_OK;
}

int sk_op_swiglu_gemv(void* stream, int32_t B, int32_t I, int32_t D, int32_t wdtype, const float* x,
                      const void* wg, const void* wu, float* out) {
  int rc = check_wdtype(wdtype);
  if (rc) return rc;
  SK_CHECK(B > 0 && I > 0 && D > 0 && D % 8 == 0, SK_EINVAL, "B, I > 0 and D a positive multiple of 8");
  SK_CHECK(x && wg && wu && out, SK_EINVAL, "NULL operand");
  SK_CHECK(aligned16(x) && aligned16(wg) && aligned16(wu), SK_EINVAL, "operands must be 16-byte aligned");
  GemvArgs a = gemv_args(wg, I, D, x, D, out, I);
  a.w[1] = wu;
  return project_rows<EPI_SWIGLU>((hipStream_t)stream, wdtype, B, a);
}

int sk_op_down_residual_gemv(void* stream, int32_t B, int32_t D, int32_t I, int32_t wdtype,
                             const float* act, const void* wd, const float* residual, float* out) {
  int rc = check_wdtype(wdtype);
  if (rc) return rc;
  SK_CHECK(B > 0 && D > 0 && I > 0 && I % 8 == 0, SK_EINVAL, "B, D > 0 and I a positive multiple of 8");
  SK_CHECK(act && wd && residual && out, SK_EINVAL, "NULL operand");
  SK_CHECK(aligned16(act) && aligned16(wd), SK_EINVAL, "operands must be 16-byte aligned");
  GemvArgs a = gemv_args(wd, D, I, act, I, out, D);
  a.res = residual; a.ldr = D;
  return project_rows<EPI_RESID>((hipStream_t)stream, wdtype, B, a);
}

int sk_op_classifier_gemv(void* stream, int32_t B, int32_t V, int32_t D, int32_t wdtype,
                          const float* body, const void* wq, const float* bias, float* out) {
  int rc = check_wdtype(wdtype);
  if (rc) return rc;
  SK_CHECK(B > 0 && V > 0 && D > 0 && D % 8 == 0, SK_EINVAL, "B, V > 0 and D a positive multiple of 8");
  SK_CHECK(body && wq && bias && out, SK_EINVAL, "NULL operand");
  SK_CHECK(aligned16(body) && aligned16(wq), SK_EINVAL, "operands must be 16-byte aligned");
  GemvArgs a = gemv_args(wq, V, D, body, D, out, V);
  a.bias = bias;
  return project_rows<EPI_BIAS>((hipStream_t)stream, wdtype, B, a);
}

int sk_op_frame_embed(void* stream, int32_t R, int32_t Q, int32_t V, int32_t D, float scale,
                      const int64_t* codes, const float* table, float* out) {
  SK_CHECK(R > 0 && Q > 0 && V > 0 && D > 0, SK_EINVAL, "R, Q, V, D must be positive");
  SK_CHECK(codes && table && out, SK_EINVAL, "NULL operand");
  hipLaunchKernelGGL(frame_embed_op_kernel, dim3(R), dim3(NT), 0, (hipStream_t)stream, codes, table, Q, V,
                     D, scale, out);
  SK_HIP(hipGetLastError());
  return SK_OK;
}

int sk_op_prefix_add(void* stream, int32_t B, int32_t V, int32_t D, float scale, const float* prefix,
                     const float* table_q, const int64_t* code, float* out) {
  SK_CHECK(B > 0 && V > 0 && D > 0, SK_EINVAL, "B, V, D must be positive");
  SK_CHECK(prefix && table_q && code && out, SK_EINVAL, "NULL operand");
  hipLaunchKernelGGL(prefix_add_op_kernel, dim3(B), dim3(NT), 0, (hipStream_t)stream, prefix, table_q,
                     code, V, D, scale, out);
  SK_HIP(hipGetLastError());
  return SK_OK;
}

int sk_op_sampling_prep(void* stream, int32_t V, int32_t bos_id, int32_t pad_id, int32_t eos_id,
                        const float* logits, const float* temperature, const int32_t* mask_eos,
                        float* out) {
  SK_CHECK(V > 0, SK_EINVAL, "V must be positive");
  SK_CHECK(logits && temperature && mask_eos && out, SK_EINVAL, "NULL operand");
  hipLaunchKernelGGL(sampling_prep_op_kernel, dim3((V + NT - 1) / NT), dim3(NT), 0, (hipStream_t)stream,
                     logits, temperature, mask_eos, V, bos_id, pad_id, eos_id, out);
  SK_HIP(hipGetLastError());
  return SK_OK;
}

int sk_op_sample(void* stream, int32_t rows, int32_t V, const float* logits, float cfg_scale, int32_t q,
                 int32_t mask_eos_q0, int32_t bos_id, int32_t eos_id, int32_t pad_id, float temperature,
                 int32_t top_k, float top_p, double u, int64_t* code_out) {
  SK_CHECK(rows == 1 || rows == 2, SK_EINVAL, "rows must be 1 or 2");
  SK_CHECK(V > 3 && V <= MAX_V, SK_EINVAL, "V must be in [4, %d]", MAX_V);
  SK_CHECK(logits && code_out, SK_EINVAL, "NULL operand");
  SK_CHECK(u >= 0.0 && u < 1.0, SK_EINVAL, "u must lie in [0, 1)");
  SK_CHECK(q >= 0, SK_EINVAL, "q must be non-negative");
  SK_HIP(prepare_sampler());
  SK_HIP(with_vpt(V, [&](auto vpt) {
    hipLaunchKernelGGL((sample_op_kernel<decltype(vpt)::value>), dim3(1), dim3(SNT), SAMPLE_SMEM,
                       (hipStream_t)stream, logits, rows, V, cfg_scale, q, mask_eos_q0, bos_id, eos_id, pad_id,
                       temperature, top_k, top_p, u, code_out);
    return hipGetLastError();
  }));
  return SK_OK;
}

}  // extern "C"
