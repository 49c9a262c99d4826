// What the surrogate's kernels (mlp.hip) and its C ABI (mlp_capi.cpp) share.
#pragma once

#include "../../include/misohip.h"
#include "launch.hpp"

namespace misohip {

// The network's device arrays, the layers of each behind one another: a kernel
// finds a layer's part by arithmetic on its arguments (a table of layers in
// memory cost every layer of every workgroup a chain of cold scalar loads).
// Packed arrays: blocks of 16 rows x 32 k, see mlp.hip.
struct MlpNet {
  int n_in, n_hidden, n_out, nl;
  long rows;                                   // columns that pre, aT and dT hold
  float *w, *b, *gw, *gb, *mw, *vw, *mb, *vb;  // w, gw, mw, vw: [out][in]
  uint16_t *wp, *wtp;  // packed: outputs x inputs, inputs x outputs
  float *pre;          // hidden layers: pre-activations, by the lanes of the chain
  uint16_t *aT, *dT;   // packed with the columns as k: input, pre-activation gradient
  __host__ __device__ int in(int l) const { return l ? n_hidden : n_in; }
  __host__ __device__ int out(int l) const { return l == nl - 1 ? n_out : n_hidden; }
  __host__ __device__ long w_at(int l) const {
    return l ? (long)n_hidden * (n_in + (l - 1L) * n_hidden) : 0;
  }
  __host__ __device__ long b_at(int l) const { return (long)l * n_hidden; }
  __host__ __device__ long d_at(int l) const { return rows * n_hidden * l; }  // pre, dT
  __host__ __device__ long a_at(int l) const {
    return l ? rows * (n_in + (l - 1L) * n_hidden) : 0;
  }
  // 32 x 32 tiles of weights, 32 biases: layer l's first, and all
  __host__ __device__ int tile_at(int l) const { return (int)(w_at(l) / 1024); }
  __host__ __device__ int tiles() const { return tile_at(nl - 1) + n_hidden / 32 * (n_out / 32); }
  __host__ __device__ int bias_tiles() const { return (n_hidden * (nl - 1) + n_out) / 32; }
  __host__ __device__ int layer_of(int tile) const {  // nl is at least 2
    const int t = tile - tile_at(1), per = n_hidden / 32 * (n_hidden / 32);
    return t < 0 ? 0 : t / per < nl - 2 ? 1 + t / per : nl - 1;
  }
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

// two activation buffers of 16 columns and widths up to `width` exceed the LDS
bool mlp_is_wide(int n_in, int width);
// inference goes layer by layer, by way of g0 and g1
bool mlp_by_layers(int n_in, int n_hidden);
// g0, g1: rows of maxw + 8 for M columns, rounded up to whole 64s
hipError_t launch_mlp_forward(hipStream_t, const MlpNet &, int maxw, const uint16_t *X, int M,
                              float *Y, const MlpField &, uint16_t *g0, uint16_t *g1);
// Y may be null
hipError_t launch_mlp_grad(hipStream_t, const MlpNet &, bool wide, int maxw, const uint16_t *X,
                           int M, const MlpLoss &, float *Y, uint16_t *g0, uint16_t *g1);
// sums of squares of Y - T into part[0 .. *parts - 1]
hipError_t launch_mlp_loss(hipStream_t, const float *Y, const float *T, float *part, long n,
                           int *parts);
hipError_t launch_mlp_adam(hipStream_t, const MlpNet &, const MlpAdam &);
// the packed copies of one layer's weights
hipError_t launch_mlp_pack(hipStream_t, const MlpNet &, int layer);
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
