// C ABI of the BF16 MLP primitives (include/pyscfad_amd_mlp.h).
#include <hip/hip_runtime.h>
#include <stdint.h>
#include "../../include/pyscfad_amd_ccsdt.h"
#include <cmath>
#include <cstring>
#include "../../include/pyscfad_amd_mlp.h"
#include "mlp_fused.h"

namespace pamd {
hipError_t launch_gemm_bf16_tn(int M, int N, int K, const uint16_t *A, int lda, const uint16_t *B,
                               int ldb, const float *bias, float *C, int ldc, int accumulate,
                               hipStream_t s);
hipError_t launch_act_out(int M, int N, const float *Z, int act, uint16_t *Y, uint16_t *Yt,
                          hipStream_t s);
hipError_t launch_act_back(int M, int N, const float *Z, const float *dY, int act, uint16_t *dZ,
                           uint16_t *dZt, float *db, hipStream_t s);
hipError_t launch_adam(int R, int Ccols, float *w, const float *g, float *m1, float *m2, uint16_t *wb,
                       uint16_t *wt, float lr, float b1, float b2, float eps, float wd, int step,
                       hipStream_t s);
hipError_t launch_mse(int n, const float *pred, const float *y, float *dpred, float *loss,
                      hipStream_t s);
hipError_t launch_f32_to_bf16(size_t n, const float *x, uint16_t *y, int M, int N, uint16_t *yt,
                              hipStream_t s);
}  // namespace pamd

using namespace pamd;

static int status(hipError_t e) { return e == hipSuccess ? PAMD_OK : PAMD_ERR_HIP; }
static bool aligned16(const void *p) { return ((uintptr_t)p & 15u) == 0; }

extern "C" {

int pamd_bf16_gemm_tn(int M, int N, int K, const uint16_t *A, int lda, const uint16_t *B, int ldb,
                      const float *bias, float *C, int ldc, int accumulate, void *stream) {
  if (M < 1 || N < 1 || K < 1 || !A || !B || !C) return PAMD_ERR_ARG;
  if (K % 8 || lda % 8 || ldb % 8 || lda < K || ldb < K || ldc < N) return PAMD_ERR_ARG;
  if (!aligned16(A) || !aligned16(B)) return PAMD_ERR_ARG;
  return status(launch_gemm_bf16_tn(M, N, K, A, lda, B, ldb, bias, C, ldc, accumulate,
                                    (hipStream_t)stream));
}

int pamd_bf16_act_fwd(int M, int N, const float *Z, int act, uint16_t *Y, uint16_t *Yt,
                      void *stream) {
  if (M < 1 || N < 1 || !Z || (act != 0 && act != 1)) return PAMD_ERR_ARG;
  return status(launch_act_out(M, N, Z, act, Y, Yt, (hipStream_t)stream));
}

int pamd_bf16_act_bwd(int M, int N, const float *Z, const float *dY, int act, uint16_t *dZ,
                      uint16_t *dZt, float *db, void *stream) {
  if (M < 1 || N < 1 || !Z || !dY || !dZ || !dZt || !db || (act != 0 && act != 1))
    return PAMD_ERR_ARG;
  return status(launch_act_back(M, N, Z, dY, act, dZ, dZt, db, (hipStream_t)stream));
}

int pamd_adam_step(int R, int C, float *w, const float *g, float *m1, float *m2, uint16_t *wb,
                   uint16_t *wt, float lr, float beta1, float beta2, float eps, float wd, int step,
                   void *stream) {
  if (R < 1 || C < 1 || !w || !g || !m1 || !m2 || step < 1) return PAMD_ERR_ARG;
  return status(launch_adam(R, C, w, g, m1, m2, wb, wt, lr, beta1, beta2, eps, wd, step,
                            (hipStream_t)stream));
}

int pamd_mse(int n, const float *pred, const float *y, float *dpred, float *loss, void *stream) {
  if (n < 1 || !pred || !y) return PAMD_ERR_ARG;
  return status(launch_mse(n, pred, y, dpred, loss, (hipStream_t)stream));
}

int pamd_f32_to_bf16(size_t n, const float *x, uint16_t *y, int M, int N, uint16_t *yt,
                     void *stream) {
  if (!x || !y || n != (size_t)M * N) return PAMD_ERR_ARG;
  return status(launch_f32_to_bf16(n, x, y, M, N, yt, (hipStream_t)stream));
}

// widths that the whole-network kernels take: multiples of 8, activations within LDS
static bool mlp_sizes_ok(int nlayers, const int *sizes, bool train) {
  if (nlayers < 1 || nlayers > kMlpMaxLayers) return false;
  for (int l = 0; l <= nlayers; ++l)
    if (sizes[l] < 8 || sizes[l] % 8 || sizes[l] > 4096) return false;
  return mlp_lds_bytes(nlayers, sizes, train) <= kMlpMaxLds;
}

int pamd_mlp_train_scratch(int nlayers, const int *sizes, int rows, size_t *bytes) {
  if (nlayers < 1 || !sizes || rows < 1 || !bytes) return PAMD_ERR_ARG;
  if (rows % 8 || !mlp_sizes_ok(nlayers, sizes, true)) return PAMD_ERR_UNSUPPORTED;
  size_t n = 0;
  for (int l = 1; l <= nlayers; ++l) n += (size_t)sizes[l] * rows * (l < nlayers ? 2 : 1);
  *bytes = n * sizeof(uint16_t) + sizeof(float) * (size_t)((rows + 15) / 16);
  return PAMD_OK;
}

int pamd_mlp_train_step(int nlayers, const int *sizes, int rows, void *const *ptrs, const uint16_t *x,
                        const uint16_t *xt, const float *y, float lr, float beta1, float beta2, float eps,
                        float wd, int step, void *scratch, size_t scratch_bytes, float *loss, void *stream) {
  if (nlayers < 1 || !sizes || rows < 1 || !ptrs || !x || !xt || !y || !scratch || !loss || step < 1)
    return PAMD_ERR_ARG;
  size_t need = 0;
  const int st = pamd_mlp_train_scratch(nlayers, sizes, rows, &need);
  if (st != PAMD_OK) return st;
  if (scratch_bytes < need) return PAMD_ERR_WORKSPACE;
  MlpNet a;
  MlpRows r;
  memset(&a, 0, sizeof(a));
  memset(&r, 0, sizeof(r));
  a.nl = nlayers;
  memcpy(a.size, sizes, sizeof(int) * (size_t)(nlayers + 1));
  r.rows = rows;
  r.x = x;
  r.xt = xt;
  r.y = y;
  r.loss = loss;
  if (!aligned16(x) || !aligned16(xt) || !aligned16(scratch)) return PAMD_ERR_UNSUPPORTED;
  uint16_t *at = (uint16_t *)scratch;
  for (int l = 0; l < nlayers; ++l) {
    void *const *p = ptrs + 8 * l;
    for (int q = 0; q < 8; ++q)
      if (!p[q]) return PAMD_ERR_ARG;
    r.w[l] = (float *)p[0];
    r.bias[l] = (float *)p[1];
    r.m_w[l] = (float *)p[2];
    r.v_w[l] = (float *)p[3];
    r.m_b[l] = (float *)p[4];
    r.v_b[l] = (float *)p[5];
    r.wb[l] = (uint16_t *)p[6];
    r.wt[l] = (uint16_t *)p[7];
    if (!aligned16(p[6]) || !aligned16(p[7])) return PAMD_ERR_UNSUPPORTED;
    a.wb[0][l] = r.wb[l];
    a.b[0][l] = r.bias[l];
    r.dzt[l] = at;
    at += (size_t)sizes[l + 1] * rows;
    if (l + 1 < nlayers) {
      r.yt[l] = at;
      at += (size_t)sizes[l + 1] * rows;
    }
  }
  r.part = (float *)at;
  MlpAdam o = {lr, beta1, beta2, eps, wd, 1.f - powf(beta1, (float)step), 1.f - powf(beta2, (float)step)};
  return status(launch_mlp_train(a, r, o, (hipStream_t)stream));
}

int pamd_mlp_forward(int members, int nlayers, const int *sizes, int rows, void *const *ptrs, const uint16_t *x,
                     float *out, void *stream) {
  if (members < 1 || nlayers < 1 || !sizes || rows < 1 || !ptrs || !x || !out) return PAMD_ERR_ARG;
  if (members > kMlpMaxMembers || !mlp_sizes_ok(nlayers, sizes, false) || !aligned16(x))
    return PAMD_ERR_UNSUPPORTED;
  MlpNet a;
  MlpRows r;
  memset(&a, 0, sizeof(a));
  memset(&r, 0, sizeof(r));
  a.nl = nlayers;
  memcpy(a.size, sizes, sizeof(int) * (size_t)(nlayers + 1));
  for (int m = 0; m < members; ++m)
    for (int l = 0; l < nlayers; ++l) {
      void *const *p = ptrs + 2 * (m * nlayers + l);
      if (!p[0] || !p[1]) return PAMD_ERR_ARG;
      if (!aligned16(p[0])) return PAMD_ERR_UNSUPPORTED;
      a.wb[m][l] = (const uint16_t *)p[0];
      a.b[m][l] = (const float *)p[1];
    }
  r.rows = rows;
  r.x = x;
  r.out = out;
  return status(launch_mlp_forward(a, r, members, (hipStream_t)stream));
}

int pamd_standardise_bf16(int rows, int n, int ld, const double *x, const double *mean, const double *stddev,
                          uint16_t *out, void *stream) {
  if (rows < 1 || n < 1 || ld < n || !x || !mean || !stddev || !out) return PAMD_ERR_ARG;
  return status(launch_standardise(rows, n, ld, x, mean, stddev, out, (hipStream_t)stream));
}

}  // extern "C"
