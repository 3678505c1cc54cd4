// Whole-network MLP launches (mlp_fused.hip), used by mlp_capi.cpp.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace pamd {

constexpr int kMlpMaxLayers = 4, kMlpMaxMembers = 8;
constexpr int kMlpMaxLds = 64 * 1024;

// layer widths and the read-only side of every member
struct MlpNet {
  int nl;
  int size[kMlpMaxLayers + 1];
  const uint16_t *wb[kMlpMaxMembers][kMlpMaxLayers];
  const float *b[kMlpMaxMembers][kMlpMaxLayers];
};

// one batch; the fields below `out` are those of a training step of one member
struct MlpRows {
  int rows;
  const uint16_t *x;  // [rows][size[0]]
  float *out;         // forward: [members][rows][size[nl]]
  const uint16_t *xt;  // [size[0]][rows]
  const float *y;
  float *loss, *part;  // part: (rows + 15) / 16 partial losses
  uint16_t *yt[kMlpMaxLayers], *dzt[kMlpMaxLayers];  // transposed activations and dZ, [N][rows]
  float *w[kMlpMaxLayers], *m_w[kMlpMaxLayers], *v_w[kMlpMaxLayers];
  float *bias[kMlpMaxLayers], *m_b[kMlpMaxLayers], *v_b[kMlpMaxLayers];
  uint16_t *wb[kMlpMaxLayers], *wt[kMlpMaxLayers];
};

struct MlpAdam {
  float lr, b1, b2, eps, wd, c1, c2;
};

int mlp_lds_bytes(int nl, const int *size, bool train);
hipError_t launch_mlp_forward(const MlpNet &a, const MlpRows &r, int members, hipStream_t s);
hipError_t launch_mlp_train(const MlpNet &a, const MlpRows &r, const MlpAdam &o, hipStream_t s);
hipError_t launch_standardise(int rows, int n, int ld, const double *x, const double *mean, const double *std_,
                              uint16_t *out, hipStream_t s);

}  // namespace pamd
