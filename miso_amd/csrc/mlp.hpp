// What the surrogate's kernels (mlp.hip) and its C ABI (mlp_capi.cpp) share.
#pragma once

#include "../../include/misohip.h"
#include "launch.hpp"

namespace misohip {

// One layer, in device memory.  Packed arrays: blocks of 16 rows x 32 k, see
// mlp.hip.
struct MlpLayer {
  int in, out;
  int tile0;  // its first 32 x 32 tile of the weight gradients' and the update's launch
  float *w, *b, *gw, *gb, *mw, *vw, *mb, *vb;  // w, gw, mw, vw: [out][in]
  uint16_t *wp, *wtp;  // packed: outputs x inputs, inputs x outputs
  float *pre;          // hidden layers: pre-activations, by the lanes of the chain
  uint16_t *aT, *dT;   // packed with the columns as k: input, pre-activation gradient
};

struct MlpLoss {
  const float *T;  // targets [M][out]
  float scale;     // 1 / (M out)
};

struct MlpAdam {
  float lr, b1, b2, eps, c1, c2, wd;
};

// Q_rad field from the network output: qrad = y * sd[kz] + mu[kz] (+ corr,
// the column correction the last plain solve left); columns with flag != 0
// take q_rt.  qrad null: the output alone.
struct MlpField {
  const float *mu, *sd;
  const int *flag;
  const double *q_rt, *corr;
  double *qrad;
  Shape sh;
  int col0;  // the interior column (i fastest) of the first one
};

// two activation buffers of 16 columns and widths up to maxw exceed the LDS
bool mlp_is_wide(int n_in, int maxw);
hipError_t launch_mlp_forward(hipStream_t, const MlpLayer *, int nl, int n_in, int n_hidden,
                              bool wide, int maxw, const uint16_t *X, int M, float *Y,
                              const MlpField &, uint16_t *g0, uint16_t *g1);
// tiles: of 32 x 32 weights of all layers, bias_tiles of 32 biases; Y may be null
hipError_t launch_mlp_grad(hipStream_t, const MlpLayer *, int nl, int n_in, bool wide, int maxw,
                           int tiles, int bias_tiles, const uint16_t *X, int M, const MlpLoss &,
                           float *Y, uint16_t *g0, uint16_t *g1);
// sums of squares of Y - T into part[0 .. *parts - 1]
hipError_t launch_mlp_loss(hipStream_t, const float *Y, const float *T, float *part, long n,
                           int *parts);
hipError_t launch_mlp_adam(hipStream_t, const MlpLayer *, int nl, int tiles, const MlpAdam &);
// the packed copies of one layer's weights
hipError_t launch_mlp_pack(hipStream_t, const MlpLayer *, int nl, int layer, int tiles);
hipError_t launch_column_features(hipStream_t, const Fld<const double> &, const Shape &, double,
                                  const float *, const float *, uint16_t *, float *, int);
constexpr int MLP_SHARES = MISOHIP_MOMENT_SHARES;
hipError_t launch_moments(hipStream_t, const void *x, bool f64, const long long *rows, long n,
                          int W, double *mean, double *sd, double *mean_abs, double *work);
hipError_t launch_normalize(hipStream_t, const void *x, bool f64, long n, int W,
                            const double *mean, const double *sd, void *out, bool bf16);
hipError_t launch_column_residual(hipStream_t, const float *, const Shape &, const float *,
                                  const float *, const double *, int *, float, double *);

}  // namespace misohip
