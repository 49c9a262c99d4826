// C ABI of the per-column MLP surrogate (include/misohip.h, misohip_mlp_*).
// The library owns the network state; the network, its gradients and its
// update are kernels of mlp.hip.
#include <cmath>
#include <cstring>
#include <new>
#include <vector>

#include "ctx_internal.hpp"
#include "mlp.hpp"

using namespace misohip;

struct misohip_mlp {
  int n_in, n_hidden, n_out, n_layers;  // n_layers = hidden layers + output layer
  int max_batch;
  int maxw;    // the widest activation
  bool wide;   // training: activations in g0, g1 instead of LDS
  bool by_layers;  // inference: the same
  long t;  // Adam step
  MlpNet net;
  uint16_t *g0 = nullptr, *g1 = nullptr;
  float *y = nullptr;            // the network's output where the loss is asked for
  float *loss_part = nullptr;
  float *h_loss = nullptr;       // pinned
  float *mu_in = nullptr, *sd_in = nullptr, *mu_out = nullptr, *sd_out = nullptr;
  std::vector<void *> allocs;
};

namespace {

template <typename T> hipError_t alloc(misohip_mlp *m, T **p, size_t n) {
  void *q = nullptr;
  hipError_t e = hipMalloc(&q, sizeof(T) * (n ? n : 1));
  if (e != hipSuccess) return e;
  e = hipMemset(q, 0, sizeof(T) * (n ? n : 1));
  m->allocs.push_back(q);
  *p = static_cast<T *>(q);
  return e;
}

int forward(misohip_ctx *ctx, misohip_mlp *m, const uint16_t *X, int batch, float *Y,
            const MlpField &field) {
  MISOHIP_TRY(launch_mlp_forward(ctx->stream, m->net, m->maxw, X, batch, Y, field, m->g0, m->g1));
  return MISOHIP_OK;
}

int check_batch(misohip_mlp *m, int batch) {
  if (batch < 1 || batch > m->max_batch) return MISOHIP_E_RANGE;
  return MISOHIP_OK;
}

Shape shape_of(const misohip_grid *g) {
  Shape s;
  s.It = g->i_total; s.Jt = g->j_total; s.Kt = g->k_total;
  s.mi = g->i_margin; s.mj = g->j_margin; s.mk = g->k_margin;
  s.is = g->is; s.js = g->js; s.ks = g->ks;
  return s;
}

}  // namespace

extern "C" {

int misohip_mlp_create(misohip_ctx *ctx, int n_in, int n_hidden, int n_hidden_layers, int n_out,
                       int max_batch, misohip_mlp **out) {
  if (!ctx || !out || n_in <= 0 || n_hidden <= 0 || n_out <= 0 || n_hidden_layers < 1)
    return MISOHIP_E_ARG;
  if (n_in % 32 || n_hidden % 32 || n_out % 32 || max_batch < 32 || max_batch % 32)
    return MISOHIP_E_ARG;  // GEMM K dimensions and the split-K batch
  *out = nullptr;
  MISOHIP_TRY(hipSetDevice(ctx->device));
  misohip_mlp *m = new (std::nothrow) misohip_mlp;
  if (!m) return MISOHIP_E_NOMEM;
  m->n_in = n_in;
  m->n_hidden = n_hidden;
  m->n_out = n_out;
  m->n_layers = n_hidden_layers + 1;
  m->max_batch = max_batch;
  m->t = 0;
  m->maxw = n_hidden > n_out ? n_hidden : n_out;
  m->wide = mlp_is_wide(n_in, m->maxw);
  m->by_layers = mlp_by_layers(n_in, n_hidden);
  hipError_t e = hipSuccess;
  MlpNet &net = m->net;
  net.n_in = n_in;
  net.n_hidden = n_hidden;
  net.n_out = n_out;
  net.nl = m->n_layers;
  net.rows = max_batch;
  const size_t nw = (size_t)net.w_at(m->n_layers - 1) + (size_t)n_hidden * n_out;
  const size_t nb = (size_t)net.b_at(m->n_layers - 1) + n_out;
  for (float **p : {&net.w, &net.gw, &net.mw, &net.vw})
    if (e == hipSuccess) e = alloc(m, p, nw);
  for (float **p : {&net.b, &net.gb, &net.mb, &net.vb})
    if (e == hipSuccess) e = alloc(m, p, nb);
  for (uint16_t **p : {&net.wp, &net.wtp})
    if (e == hipSuccess) e = alloc(m, p, nw);
  if (e == hipSuccess) e = alloc(m, &net.pre, (size_t)net.d_at(m->n_layers - 1));
  if (e == hipSuccess) e = alloc(m, &net.aT, (size_t)net.a_at(m->n_layers));
  if (e == hipSuccess)
    e = alloc(m, &net.dT, (size_t)net.d_at(m->n_layers - 1) + (size_t)max_batch * n_out);
  if (m->wide || m->by_layers) {
    const size_t rows = (size_t)(max_batch + 63) / 64 * 64;  // whole tiles of columns
    if (e == hipSuccess) e = alloc(m, &m->g0, rows * (m->maxw + 8));
    if (e == hipSuccess) e = alloc(m, &m->g1, rows * (m->maxw + 8));
  }
  if (e == hipSuccess) e = alloc(m, &m->loss_part, (size_t)max_batch * n_out / 256 + 1);
  if (e == hipSuccess) e = alloc(m, &m->y, (size_t)max_batch * n_out);
  if (e == hipSuccess) e = alloc(m, &m->mu_in, n_in);
  if (e == hipSuccess) e = alloc(m, &m->sd_in, n_in);
  if (e == hipSuccess) e = alloc(m, &m->mu_out, n_out);
  if (e == hipSuccess) e = alloc(m, &m->sd_out, n_out);
  if (e == hipSuccess)
    e = hipHostMalloc(&m->h_loss, sizeof(float) * ((size_t)max_batch * n_out / 256 + 1), hipHostMallocDefault);
  if (e != hipSuccess) {
    for (void *q : m->allocs) (void)hipFree(q);
    delete m;
    return hip_fail(e);
  }
  *out = m;
  return MISOHIP_OK;
}

int misohip_mlp_destroy(misohip_mlp *m) {
  if (!m) return MISOHIP_E_ARG;
  (void)hipDeviceSynchronize();
  for (void *q : m->allocs) (void)hipFree(q);
  if (m->h_loss) (void)hipHostFree(m->h_loss);
  delete m;
  return MISOHIP_OK;
}

int misohip_mlp_set_layer(misohip_ctx *ctx, misohip_mlp *m, int layer, const float *w_host,
                          const float *b_host) {
  if (!ctx || !m || layer < 0 || layer >= m->n_layers || !w_host || !b_host) return MISOHIP_E_ARG;
  MISOHIP_TRY(hipSetDevice(ctx->device));
  const MlpNet &y = m->net;
  const long w0 = y.w_at(layer), b0 = y.b_at(layer);
  const size_t nw = sizeof(float) * y.out(layer) * y.in(layer), nb = sizeof(float) * y.out(layer);
  MISOHIP_TRY(hipMemcpy(y.w + w0, w_host, nw, hipMemcpyHostToDevice));
  MISOHIP_TRY(hipMemcpy(y.b + b0, b_host, nb, hipMemcpyHostToDevice));
  MISOHIP_TRY(launch_mlp_pack(ctx->stream, y, layer));
  MISOHIP_TRY(hipMemsetAsync(y.mw + w0, 0, nw, ctx->stream));
  MISOHIP_TRY(hipMemsetAsync(y.vw + w0, 0, nw, ctx->stream));
  MISOHIP_TRY(hipMemsetAsync(y.mb + b0, 0, nb, ctx->stream));
  MISOHIP_TRY(hipMemsetAsync(y.vb + b0, 0, nb, ctx->stream));
  MISOHIP_TRY(hipStreamSynchronize(ctx->stream));
  m->t = 0;
  return MISOHIP_OK;
}

// which: 0 = fp32 master weights, 1 = biases, 2 = weight gradients, 3 = bias gradients
int misohip_mlp_get_layer(misohip_ctx *ctx, misohip_mlp *m, int layer, int which, float *host) {
  if (!ctx || !m || layer < 0 || layer >= m->n_layers || !host || which < 0 || which > 3)
    return MISOHIP_E_ARG;
  MISOHIP_TRY(hipSetDevice(ctx->device));
  MISOHIP_TRY(hipStreamSynchronize(ctx->stream));
  const MlpNet &y = m->net;
  const bool bias = which == 1 || which == 3;
  const float *src = (which == 0 ? y.w : which == 1 ? y.b : which == 2 ? y.gw : y.gb) +
                     (bias ? y.b_at(layer) : y.w_at(layer));
  const size_t n = bias ? (size_t)y.out(layer) : (size_t)y.out(layer) * y.in(layer);
  MISOHIP_TRY(hipMemcpy(host, src, sizeof(float) * n, hipMemcpyDeviceToHost));
  return MISOHIP_OK;
}

int misohip_mlp_set_norm(misohip_ctx *ctx, misohip_mlp *m, const float *mu_in, const float *sd_in,
                         const float *mu_out, const float *sd_out) {
  if (!ctx || !m || !mu_in || !sd_in || !mu_out || !sd_out) return MISOHIP_E_ARG;
  MISOHIP_TRY(hipSetDevice(ctx->device));
  MISOHIP_TRY(hipMemcpy(m->mu_in, mu_in, sizeof(float) * m->n_in, hipMemcpyHostToDevice));
  MISOHIP_TRY(hipMemcpy(m->sd_in, sd_in, sizeof(float) * m->n_in, hipMemcpyHostToDevice));
  MISOHIP_TRY(hipMemcpy(m->mu_out, mu_out, sizeof(float) * m->n_out, hipMemcpyHostToDevice));
  MISOHIP_TRY(hipMemcpy(m->sd_out, sd_out, sizeof(float) * m->n_out, hipMemcpyHostToDevice));
  return MISOHIP_OK;
}

int misohip_mlp_forward(misohip_ctx *ctx, misohip_mlp *m, const void *X, int batch, float *Y) {
  if (!ctx || !m || !X || !Y) return MISOHIP_E_ARG;
  if (int rc = check_batch(m, batch)) return rc;
  MISOHIP_TRY(hipSetDevice(ctx->device));
  Timed t_(ctx, MISOHIP_KIND_MLP);
  return forward(ctx, m, static_cast<const uint16_t *>(X), batch, Y, MlpField{});
}

// loss and gradients (MSE on the batch); *loss receives the mean squared error
int misohip_mlp_grad(misohip_ctx *ctx, misohip_mlp *m, const void *X, const float *T, int batch,
                     double *loss) {
  if (!ctx || !m || !X || !T) return MISOHIP_E_ARG;
  if (int rc = check_batch(m, batch)) return rc;
  if (batch % 32) return MISOHIP_E_ARG;  // the batch is the weight-gradient GEMM's K
  MISOHIP_TRY(hipSetDevice(ctx->device));
  {
    Timed t_(ctx, MISOHIP_KIND_MLP);
    const long n = (long)batch * m->n_out;
    MlpLoss ls;
    ls.T = T;
    ls.scale = 1.f / (float)n;
    MISOHIP_TRY(launch_mlp_grad(ctx->stream, m->net, m->wide, m->maxw,
                                static_cast<const uint16_t *>(X), batch, ls,
                                loss ? m->y : nullptr, m->g0, m->g1));
    int nb = 0;
    if (loss) MISOHIP_TRY(launch_mlp_loss(ctx->stream, m->y, T, m->loss_part, n, &nb));
    if (loss) {
      MISOHIP_TRY(hipMemcpyAsync(m->h_loss, m->loss_part, sizeof(float) * nb,
                                 hipMemcpyDeviceToHost, ctx->stream));
      MISOHIP_TRY(hipStreamSynchronize(ctx->stream));
      double s = 0.0;
      for (int i = 0; i < nb; ++i) s += m->h_loss[i];
      *loss = s / (double)n;
    }
  }
  return MISOHIP_OK;
}

// Adam update of every layer from the current gradients
int misohip_mlp_adam(misohip_ctx *ctx, misohip_mlp *m, float lr, float beta1, float beta2,
                     float eps, float weight_decay) {
  if (!ctx || !m || !(lr > 0.f)) return MISOHIP_E_ARG;
  MISOHIP_TRY(hipSetDevice(ctx->device));
  Timed t_(ctx, MISOHIP_KIND_MLP);
  m->t += 1;
  const float c1 = 1.f - std::pow(beta1, (float)m->t), c2 = 1.f - std::pow(beta2, (float)m->t);
  const MlpAdam p = {lr, beta1, beta2, eps, c1, c2, weight_decay};
  MISOHIP_TRY(launch_mlp_adam(ctx->stream, m->net, p));
  return MISOHIP_OK;
}

int misohip_mlp_features(misohip_ctx *ctx, misohip_mlp *m, const misohip_grid *g,
                         const misohip_fields *qq, double gm, void *X, float *Xf) {
  if (!ctx || !m || !g || !qq || !X) return MISOHIP_E_ARG;
  const int nz = g->k_total - 2 * g->k_margin;
  const int nfeat = nz > 0 && m->n_in % nz == 0 ? m->n_in / nz : 0;
  if (nfeat != 3 && nfeat != 4) return MISOHIP_E_ARG;
  if (nfeat == 4 && (g->i_size < 2 || g->j_size < 2)) return MISOHIP_E_ARG;
  MISOHIP_TRY(hipSetDevice(ctx->device));
  Fld<const double> q;
  for (int f = 0; f < 9; ++f) q.q[f] = static_cast<const double *>(qq->q[f]);
  Timed t_(ctx, MISOHIP_KIND_MLP);
  MISOHIP_TRY(launch_column_features(ctx->stream, q, shape_of(g), gm, m->mu_in, m->sd_in,
                                     static_cast<uint16_t *>(X), Xf, nfeat));
  return MISOHIP_OK;
}

// Q_rad of every interior cell from the network (columns along z), plus the
// correction field corr when given; columns with flag != 0 take q_rt
// instead.  Y is scratch of (columns x n_out).
int misohip_mlp_qrad(misohip_ctx *ctx, misohip_mlp *m, const misohip_grid *g, const void *X,
                     float *Y, const int *flags, const void *q_rt, const void *corr,
                     void *qrad) {
  if (!ctx || !m || !g || !X || !Y || !qrad) return MISOHIP_E_ARG;
  const int ncol = (g->i_total - 2 * g->i_margin) * (g->j_total - 2 * g->j_margin);
  if (g->k_total - 2 * g->k_margin != m->n_out) return MISOHIP_E_ARG;
  if (flags && !q_rt) return MISOHIP_E_ARG;
  MISOHIP_TRY(hipSetDevice(ctx->device));
  Timed t_(ctx, MISOHIP_KIND_MLP);
  MlpField f;
  f.mu = m->mu_out;
  f.sd = m->sd_out;
  f.flag = flags;
  f.q_rt = static_cast<const double *>(q_rt);
  f.corr = static_cast<const double *>(corr);
  f.qrad = static_cast<double *>(qrad);
  f.sh = shape_of(g);
  // activations in LDS: any number of columns; else as many as g0, g1 hold
  const int step = m->by_layers ? m->max_batch : ncol;
  for (int c0 = 0; c0 < ncol; c0 += step) {
    const int nb = ncol - c0 < step ? ncol - c0 : step;
    f.col0 = c0;
    if (int rc = forward(ctx, m, static_cast<const uint16_t *>(X) + (long)c0 * m->n_in, nb,
                         Y + (long)c0 * m->n_out, f))
      return rc;
  }
  return MISOHIP_OK;
}

int misohip_column_moments(misohip_dtype dt, const void *x, const long long *rows, long n,
                           int width, double *mean, double *sd, double *mean_abs, double *work,
                           void *stream) {
  if (n < 0 || width < 1 || (n > 0 && (!x || !rows)) || !mean || !sd || !mean_abs || !work)
    return MISOHIP_E_ARG;
  if (dt != MISOHIP_F64 && dt != MISOHIP_F32) return MISOHIP_E_DTYPE;
  MISOHIP_TRY(launch_moments(static_cast<hipStream_t>(stream), x, dt == MISOHIP_F64, rows, n,
                             width, mean, sd, mean_abs, work));
  return MISOHIP_OK;
}

int misohip_column_normalize(misohip_dtype dt, const void *x, long n, int width,
                             const double *mean, const double *sd, int bf16, void *out,
                             void *stream) {
  if (n < 0 || width < 4 || width % 4 || (n > 0 && (!x || !out)) || !mean || !sd)
    return MISOHIP_E_ARG;
  if (dt != MISOHIP_F64 && dt != MISOHIP_F32) return MISOHIP_E_DTYPE;
  if ((double)n * width / 1024.0 >= 4294967295.0) return MISOHIP_E_RANGE;
  if (n == 0) return MISOHIP_OK;
  MISOHIP_TRY(launch_normalize(static_cast<hipStream_t>(stream), x, dt == MISOHIP_F64, n, width,
                               mean, sd, out, bf16 != 0));
  return MISOHIP_OK;
}

// residual indicator: flag columns whose network Q_rad (from Y) differs from
// the plain-RT q_rt by more than tol in relative L2 over the column; corr
// (optional) receives q_rt - network on every interior cell
int misohip_mlp_residual(misohip_ctx *ctx, misohip_mlp *m, const misohip_grid *g, const float *Y,
                         const void *q_rt, int *flags, double tol, void *corr) {
  if (!ctx || !m || !g || !Y || !q_rt || !flags) return MISOHIP_E_ARG;
  MISOHIP_TRY(hipSetDevice(ctx->device));
  Timed t_(ctx, MISOHIP_KIND_MLP);
  MISOHIP_TRY(launch_column_residual(ctx->stream, Y, shape_of(g), m->mu_out, m->sd_out,
                                     static_cast<const double *>(q_rt), flags, (float)tol,
                                     static_cast<double *>(corr)));
  return MISOHIP_OK;
}

}  // extern "C"
