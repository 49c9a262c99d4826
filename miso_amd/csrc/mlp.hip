// Per-column MLP surrogate of the radiative heating: BF16 operands on the
// CDNA4 matrix cores (v_mfma_f32_16x16x32_bf16), FP32 accumulation, FP32
// master weights.  No counterpart in the reference (it has no MHD-RT
// coupling at all).
//
// Network: x (3*nz or 4*nz features of one column) -> hidden -> ... -> nz,
// SiLU on the hidden layers; every width a multiple of 32.
//
// MFMA 16x16x32 lane layout: lane l holds A[l%16][8*(l/16) .. +7],
// B[8*(l/16) .. +7][l%16], and accumulator v holds D[4*(l/16) + v][l%16].
// Every operand that a kernel takes from global memory is kept in blocks of
// 16 rows x 32 k (1 KiB), the lane's 8 values next to each other ("packed"),
// so that a wave loads a fragment as 1 KiB of consecutive bytes.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>
#include <type_traits>

#include "mlp.hpp"

namespace misohip {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
// the caller's fp32 arrays: four floats at any multiple of four bytes
typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));

__device__ __forceinline__ uint16_t f2bf(float f) {  // round to nearest even
  uint32_t u = __float_as_uint(f);
  if ((u & 0x7fffffffu) > 0x7f800000u) return (uint16_t)((u >> 16) | 0x40u);  // NaN stays NaN
  u += 0x7fffu + ((u >> 16) & 1u);
  return (uint16_t)(u >> 16);
}
__device__ __forceinline__ uint2 f2bf4(f32x4 x) {
  return make_uint2((uint32_t)f2bf(x[0]) | (uint32_t)f2bf(x[1]) << 16,
                    (uint32_t)f2bf(x[2]) | (uint32_t)f2bf(x[3]) << 16);
}
__device__ __forceinline__ f32x4 mfma(bf16x8 a, bf16x8 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

// The waves of a workgroup exchange activations through LDS (147456 columns of
// inference 635 -> 622 us with loads and stores in flight across it); WIDE:
// through global memory.
template <bool WIDE> __device__ __forceinline__ void chain_barrier() {
  if (WIDE)
    __syncthreads();
  else
    lds_barrier();
}

// features of X that a workgroup of 64 columns takes at a time
constexpr int MLP_X_TALL = 128;

// The network from its input columns to its output (TRAIN: and back from the
// gradient of the mean squared error to every layer's pre-activation gradient;
// Y, where given, receives the output) in one launch: a workgroup
// takes NS = 16 NT columns through all layers.  A layer is D = W a: the
// weights are the A operand, from their packed copies (L2 holds all of them),
// the activations the B operand, rows of one column in one of two buffers in
// LDS (WIDE: in the columns' part of g0, g1, where two of them do not fit);
// lanes are columns in D, so that a lane holds four consecutive outputs of
// one column.  X passes through LDS in chunks of xw features (all but the last
// a multiple of 32 PD: the k-steps in flight keep their places).
//   WIDE: `phase` alone, a layer forward or (nl, nl + 1, ..) back, its input by
// way of LDS as X, its outputs spread over the launch's rows of workgroups: with
// all layers in a workgroup, which fetched its fragments from g0, g1 as it came
// to them, a batch of 32 through 1536-2048-2048-2048-384 took 521 us, this 54
// (128 x 128 tiles of a launch per layer 190; 16384 columns 2269, 668, 1053; a
// training step's gradients at a batch of 32 972, 114, 490).
//   A wave takes cnt <= RT row tiles of 16 outputs at a time and keeps PD
// k-steps of their weights in flight; the first PD of the next layer are
// loaded before the barrier that ends a layer.
//   TRAIN keeps what the weight gradients read, packed with the columns as k:
// X and the activations (aT), the pre-activation gradients (dT); and the
// hidden layers' pre-activations in FP32, which the lane that wrote them
// reads again.
// NT = 1 (16 waves) spreads a batch of 1024 over 64 CUs; NT = 4 (eight waves,
// two workgroups a CU) reads the weights a quarter as often, for large
// batches of inference (NT = 2: 736 us for 635 at 147456 columns; four waves
// of twice the row tiles 680; three row tiles a wave spill: 994; features of
// X by 256, one workgroup a CU: 850).
// A training step's chain at a batch of 1024 and 1536-256-256-256-384 is bound
// by latency: seven layers of 4 to 5 us (first weights, code that runs a few
// times, the barrier; waves wait in 55 % of their cycles), with 117 MB from L2
// in 34 us a third of what the 64 CUs could take, and VALU issue at 8 %.  A
// launch per layer, product and elementwise step (128 x 128 tiles: 16
// workgroups) took 232.  147456 columns of inference, their Q_rad field
// included, are bound by HBM: 2.2 GB in 622 us, 957 before (without its 1.1 GB
// of Y, corrections and Q_rad it would take 363).  Sums go in the order of k, 32
// to an instruction; the 32 x 32 x 16 products before, 16 to an instruction,
// gave the same bits at every size compared (outputs, gradients and weights of
// hidden widths 32 to 4096 at batches of 1 to 16384).
template <int NT, int WAVES, int RT, int PD, bool TRAIN, bool WIDE>
__global__ __launch_bounds__(64 * WAVES, 4) void mlp_chain_kernel(
    MlpNet net, const uint16_t *__restrict__ X, int M,
    float *__restrict__ Y, MlpLoss ls, MlpField fo, uint16_t *g0, uint16_t *g1, int bw, int xoff,
    int xw, int phase) {
  constexpr int NS = 16 * NT, NTHR = 64 * WAVES;
  static_assert(RT <= 3, "product()");
  static_assert(NT > 1 || RT == 1, "one row tile a wave");
  static_assert(NT == 1 || !TRAIN, "the packed columns of a training tile are 16");
  extern __shared__ __attribute__((aligned(16))) uint16_t lds[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int col = lane & 15, kq = lane >> 4;
  const int s0 = blockIdx.x * NS;
  const int pitch = bw + 8, xpitch = xw + 8;  // odd multiples of 16 bytes: no bank conflicts
  // the input layer writes the first buffer (X may be staged in the second)
  uint16_t *nxt = WIDE ? (phase & 1 ? g1 : g0) + (long)s0 * pitch : lds;
  uint16_t *cur = WIDE ? (phase & 1 ? g0 : g1) + (long)s0 * pitch : lds + NS * pitch;
  uint16_t *xbuf = lds + xoff;
  const int nl = net.nl;
  // what passes through xbuf, by columns: X, in a layer of its own its input
  const uint16_t *src = WIDE && phase ? cur : X + (long)s0 * net.n_in;
  const int ld = WIDE && phase ? pitch : net.n_in;

  bf16x8 a[PD][RT];
  f32x4 acc[RT][NT];
  auto frag = [&](const uint16_t *wp, int KT, int tile, int kt) {
    return *reinterpret_cast<const bf16x8 *>(wp + ((long)tile * KT + kt) * 512 + lane * 8);
  };
  // row tiles per wave in a pass over a layer of OT row tiles, evened out
  auto tiles_of = [&](int OT) {
    const int np = (OT + WAVES * RT - 1) / (WAVES * RT);
    return (OT + np * WAVES - 1) / (np * WAVES);
  };
  // first k-steps of the weights (tiles past the last one load the last)
  auto preload = [&](const uint16_t *wp, int KT, int OT, int base, int cnt) {
#pragma unroll
    for (int p = 0; p < PD; ++p)
#pragma unroll
      for (int r = 0; r < RT; ++r)
        if (r < cnt)
          a[p][r] = frag(wp, KT, min(base + wave * cnt + r, OT - 1), min(p, KT - 1));
  };
  // 8 consecutive columns of feature f per lane, in blocks of 16 f x 32 columns
  auto pack = [&](const uint16_t *src, int sp, int nf, uint16_t *dst, int f0) {
    for (int t = tid; t < 2 * nf; t += NTHR) {
      const int f = t & 15, o = (t >> 4) & 1, ft = t >> 5;
      uint32_t v[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const uint16_t *q = src + (8 * o + 2 * e) * sp + ft * 16 + f;
        v[e] = (uint32_t)q[0] | (uint32_t)q[sp] << 16;
      }
      const long blk = (long)(f0 / 16 + ft) * (M >> 5) + (s0 >> 5);
      *reinterpret_cast<uint4 *>(dst + blk * 512 + (f + 16 * (o + ((s0 >> 3) & 2))) * 8) =
          make_uint4(v[0], v[1], v[2], v[3]);
    }
  };
  // features [f0, f0 + cw) of K of the workgroup's columns into xbuf
  auto stage = [&](int K, int f0) {
    const int cw = min(xw, K - f0), per = cw >> 3, n = NS * per;
    chain_barrier<WIDE>();
    for (int t = tid; t < n; t += 4 * NTHR) {
      uint4 v[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int q = t + e * NTHR, r = q / per, c = q - r * per;
        v[e] = make_uint4(0, 0, 0, 0);
        if (q < n && s0 + r < M)
          v[e] = *reinterpret_cast<const uint4 *>(src + (long)r * ld + f0 + 8 * c);
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int q = t + e * NTHR, r = q / per, c = q - r * per;
        if (q < n) *reinterpret_cast<uint4 *>(xbuf + r * xpitch + 8 * c) = v[e];
      }
    }
    chain_barrier<WIDE>();
    return cw;
  };
  // NT > 1: the thread's part of XW features of the workgroup's columns, in
  // flight while the chunk before is multiplied
  constexpr int XW = MLP_X_TALL, XE = NT > 1 ? NS * XW / 8 / NTHR : 1;
  uint4 xr[XE];
  auto fetch = [&](int K, int f0) {
#pragma unroll
    for (int e = 0; e < XE; ++e) {
      const int q = tid + e * NTHR, r = q / (XW / 8), f = f0 + 8 * (q % (XW / 8));
      xr[e] = make_uint4(0, 0, 0, 0);
      if (s0 + r < M && f < K) xr[e] = *reinterpret_cast<const uint4 *>(src + (long)r * ld + f);
    }
  };
  auto put = [&](uint16_t *xb) {
#pragma unroll
    for (int e = 0; e < XE; ++e) {
      const int q = tid + e * NTHR;
      *reinterpret_cast<uint4 *>(xb + q / (XW / 8) * xpitch + 8 * (q % (XW / 8))) = xr[e];
    }
  };
  // acc = W b over all k for `cnt` row tiles; input: b by way of xbuf, chunk by
  // chunk; keep: b is X, for the weight gradients
  auto gemm = [&](auto cnt_, const uint16_t *wp, int KT, int OT, int base, const uint16_t *b,
                  bool input, bool keep) {
    constexpr int cnt = decltype(cnt_)::value;
    int tile[cnt];
#pragma unroll
    for (int r = 0; r < cnt; ++r) tile[r] = min(base + wave * cnt + r, OT - 1);
#pragma unroll
    for (int r = 0; r < cnt; ++r)
#pragma unroll
      for (int n = 0; n < NT; ++n) acc[r][n] = (f32x4){0.f, 0.f, 0.f, 0.f};
    // K-steps k0 .. k0 + ke - 1, their B operand from `row` on.  Whole rounds
    // of the PD k-steps in flight have no branch inside: past one the compiler
    // would wait for all loads in flight at the start of every round (38 us a
    // training step's chain for 34; with 8 in flight 35, with 2 37.5).
    auto steps = [&](const uint16_t *row, int rp, int k0, int ke) {
      auto one = [&](int p, int k) {
        bf16x8 bv[NT];
#pragma unroll
        for (int n = 0; n < NT; ++n)
          bv[n] = *reinterpret_cast<const bf16x8 *>(row + n * rp + k * 32);
#pragma unroll
        for (int r = 0; r < cnt; ++r)
#pragma unroll
          for (int n = 0; n < NT; ++n) acc[r][n] = mfma(a[p][r], bv[n], acc[r][n]);
      };
      int k = 0;
      for (; k + PD <= ke && k0 + k + PD < KT; k += PD) {
#pragma unroll
        for (int p = 0; p < PD; ++p) {
          one(p, k + p);
#pragma unroll
          for (int r = 0; r < cnt; ++r)
            a[p][r] = frag(wp, KT, tile[r], min(k0 + k + p + PD, KT - 1));
        }
      }
#pragma unroll
      for (int p = 0; p < PD; ++p) {  // the last PD k-steps at most
        if (k + p >= ke) break;
        one(p, k + p);
      }
    };
    if (!input) {
      steps(b + col * pitch + kq * 8, 16 * pitch, 0, KT);
    } else if constexpr (NT > 1) {
      fetch(32 * KT, 0);
      if (base) chain_barrier<WIDE>();
      put(xbuf);
      for (int k0 = 0, h = 0; k0 < KT; k0 += XW / 32, h ^= 1) {
        chain_barrier<WIDE>();
        if (k0 + XW / 32 < KT) fetch(32 * KT, k0 * 32 + XW);
        steps(xbuf + (h * NS + col) * xpitch + kq * 8, 16 * xpitch, k0, min(XW / 32, KT - k0));
        if (k0 + XW / 32 < KT) put(xbuf + (h ^ 1) * NS * xpitch);
      }
    } else {
      for (int k0 = 0; k0 < KT; k0 += xw >> 5) {
        const int cw = stage(32 * KT, k0 * 32);
        if (TRAIN && keep) pack(xbuf, xpitch, cw, net.aT, k0 * 32);
        steps(xbuf + col * xpitch + kq * 8, 16 * xpitch, k0, cw >> 5);
      }
    }
  };
  auto product = [&](int cnt, const uint16_t *wp, int KT, int OT, int base, const uint16_t *b,
                     bool input, bool keep) {
    if (RT > 2 && cnt == 3)
      gemm(std::integral_constant<int, (RT > 2 ? 3 : 1)>{}, wp, KT, OT, base, b, input, keep);
    else if (RT > 1 && cnt == 2)
      gemm(std::integral_constant<int, (RT > 1 ? 2 : 1)>{}, wp, KT, OT, base, b, input, keep);
    else
      gemm(std::integral_constant<int, 1>{}, wp, KT, OT, base, b, input, keep);
  };

  // the output of row tile r, from output o on: Y, and the Q_rad field, 32
  // columns at a time; loads go before the stores, which the compiler takes
  // for possible aliases
  auto store_output = [&](int r, int o, f32x4 bias) {
    constexpr int H = NT < 2 ? NT : 2;
    const int no = net.n_out, st = fo.sh.It * fo.sh.Jt;
    f32x4 mu, sd;
    if (fo.qrad) {
      mu = *reinterpret_cast<const f32x4 *>(fo.mu + o);
      sd = *reinterpret_cast<const f32x4 *>(fo.sd + o);
    }
#pragma unroll
    for (int n0 = 0; n0 < NT; n0 += H) {
      double other[H][4];
      int c0[H], fall[H];
      if (fo.qrad) {
#pragma unroll
        for (int n = 0; n < H; ++n) {
          const int cs = fo.col0 + min(s0 + 16 * (n0 + n) + col, M - 1);
          const int ni = fo.sh.It - 2 * fo.sh.mi, j = cs / ni, i = cs - j * ni;
          c0[n] = fo.sh.idx(fo.sh.mi + i, fo.sh.mj + j, fo.sh.mk + o);
          fall[n] = fo.flag ? fo.flag[cs] : 0;
        }
#pragma unroll
        for (int n = 0; n < H; ++n) {
          const double *q = fall[n] ? fo.q_rt : fo.corr;
#pragma unroll
          for (int v = 0; v < 4; ++v) other[n][v] = q ? q[c0[n] + v * st] : 0.0;
        }
      }
#pragma unroll
      for (int n = 0; n < H; ++n) {
        const int s = s0 + 16 * (n0 + n) + col;
        if (s >= M) continue;
        const f32x4 x = acc[r][n0 + n] + bias;
        *reinterpret_cast<f32x4u *>(Y + (long)s * no + o) = x;
        if (fo.qrad) {
#pragma unroll
          for (int v = 0; v < 4; ++v) {
            const double net = (double)(x[v] * sd[v] + mu[v]);
            fo.qrad[c0[n] + v * st] =
                fall[n] ? other[n][v] : fo.corr ? net + other[n][v] : net;
          }
        }
      }
    }
  };

  // the outputs of this workgroup among O, packed
  auto pack_rows = [&](int O, uint16_t *dst) {
    if (!WIDE) return pack(nxt, pitch, O, dst, 0);
    for (int f = blockIdx.y * WAVES * 16; f < O; f += gridDim.y * WAVES * 16)
      pack(nxt + f, pitch, min(WAVES * 16, O - f), dst, f);
  };

  auto load4 = [](const float *q) { return *reinterpret_cast<const f32x4u *>(q); };
  // WIDE: a row of workgroups per pass over the layer's outputs
  const int row = WIDE ? blockIdx.y : 0, rows = WIDE ? gridDim.y : 1;
  // ---- forward
  if (!WIDE) preload(net.wp, net.n_in / 32, net.out(0) / 16, 0, tiles_of(net.out(0) / 16));
  for (int l = WIDE ? phase : 0; l < (WIDE ? min(phase + 1, nl) : nl); ++l) {
    const bool last = l == nl - 1;
    const int KT = net.in(l) / 32, O = net.out(l), OT = O / 16, cnt = tiles_of(OT);
    const uint16_t *wp = net.wp + net.w_at(l);
    const float *b = net.b + net.b_at(l);
    for (int base = row * WAVES * cnt; base < OT; base += rows * WAVES * cnt) {
      if (WIDE || base) preload(wp, KT, OT, base, cnt);
      product(cnt, wp, KT, OT, base, cur, WIDE || l == 0, l == 0 && base == 0);
#pragma unroll
      for (int r = 0; r < RT; ++r) {
        const int tile = base + wave * cnt + r;
        if (r >= cnt || tile >= OT) break;
        const int o = tile * 16 + 4 * kq;
        const f32x4 bias = load4(b + o);
        if (!TRAIN && last) {
          store_output(r, o, bias);
          continue;
        }
#pragma unroll
        for (int n = 0; n < NT; ++n) {
          const int sl = 16 * n + col;
          const f32x4 x = acc[r][n] + bias;
          f32x4 h;
          if (!last) {
            if (TRAIN)
              *reinterpret_cast<f32x4 *>(net.pre + net.d_at(l) +
                                         ((long)blockIdx.x * OT + tile) * 256 + lane * 4) = x;
#pragma unroll
            for (int v = 0; v < 4; ++v) h[v] = x[v] / (1.f + expf(-x[v]));
          } else {
            const f32x4 t = load4(ls.T + (long)(s0 + sl) * O + o);
#pragma unroll
            for (int v = 0; v < 4; ++v) {
              const float d = x[v] - t[v];
              h[v] = 2.f * d * ls.scale;
            }
            if (Y) *reinterpret_cast<f32x4u *>(Y + (long)(s0 + sl) * O + o) = x;
          }
          *reinterpret_cast<uint2 *>(nxt + sl * pitch + o) = f2bf4(h);
        }
      }
    }
    if (!WIDE && !last)
      preload(net.wp + net.w_at(l + 1), O / 32, net.out(l + 1) / 16, 0,
              tiles_of(net.out(l + 1) / 16));
    else if (!WIDE && TRAIN)
      preload(net.wtp + net.w_at(l), O / 32, net.in(l) / 16, 0, tiles_of(net.in(l) / 16));
    if (TRAIN || (!WIDE && !last)) {
      chain_barrier<WIDE>();
      if (TRAIN) pack_rows(O, last ? net.dT + net.d_at(l) : net.aT + net.a_at(l + 1));
      uint16_t *swap = cur;
      cur = nxt;
      nxt = swap;
    }
  }
  if constexpr (TRAIN) {
    // ---- back: the gradient of layer l's input, times silu' of layer l - 1
    const int from = !WIDE ? nl - 1 : phase < nl ? 0 : 2 * nl - 1 - phase;
    for (int l = from; l > (WIDE ? max(from - 1, 0) : 0); --l) {
      const int KT = net.out(l) / 32, I = net.in(l), OT = I / 16, cnt = tiles_of(OT);
      const uint16_t *wp = net.wtp + net.w_at(l);
      for (int base = row * WAVES * cnt; base < OT; base += rows * WAVES * cnt) {
        if (WIDE || base) preload(wp, KT, OT, base, cnt);
        product(cnt, wp, KT, OT, base, cur, WIDE, false);
        const int tile = base + wave;
        if (tile < OT) {
          const f32x4 x = *reinterpret_cast<const f32x4 *>(
              net.pre + net.d_at(l - 1) + ((long)blockIdx.x * OT + tile) * 256 + lane * 4);
          f32x4 g;
#pragma unroll
          for (int v = 0; v < 4; ++v) {
            const float sg = 1.f / (1.f + expf(-x[v]));
            g[v] = acc[0][0][v] * sg * (1.f + x[v] * (1.f - sg));
          }
          *reinterpret_cast<uint2 *>(nxt + col * pitch + tile * 16 + 4 * kq) = f2bf4(g);
        }
      }
      if (!WIDE && l > 1)
        preload(net.wtp + net.w_at(l - 1), I / 32, net.in(l - 1) / 16, 0,
                tiles_of(net.in(l - 1) / 16));
      chain_barrier<WIDE>();
      pack_rows(I, net.dT + net.d_at(l - 1));
      uint16_t *swap = cur;
      cur = nxt;
      nxt = swap;
    }
  }
}

// Weight and bias gradients of every layer in one launch: gW = dpre^T a, the
// batch as k, a wave per 32 x 32 tile with eight k-steps of its operands in
// flight; then a wave per 32 biases.  `per` k-steps go into a sum of their own
// (a sixteenth of the batch where that divides), so that no chain of
// additions grows with the batch, and these sums are added in order; a bias
// is 16 sums, of every 16th column each, added in order.
// Bound by latency, with a wave for two SIMDs in three (644): 82 MB from L2 in
// 8.2 us at a batch of 1024 and 1536-256-256-256-384, a quarter of 64 bytes a
// clock and CU, where a launch per layer that transposed through LDS, its
// partial sums in memory and column sums by four workgroups took 134.
__global__ __launch_bounds__(64) void mlp_wgrad_kernel(MlpNet net, int SB, int per,
                                                       int tiles) {
  const int lane = threadIdx.x, row = lane & 15, kq = lane >> 4;
  int blk = blockIdx.x;
  if (blk >= tiles) {  // lane: bias o, octets of columns of one parity
    blk -= tiles;
    const int l = min(blk / (net.n_hidden / 32), net.nl - 1);
    blk -= l * (net.n_hidden / 32);
    const int o = lane & 31, par = lane >> 5;
    const uint16_t *d = net.dT + net.d_at(l) + ((long)(2 * blk + (o >> 4)) * SB * 64 + (o & 15)) * 8;
    float s[8] = {};
#pragma unroll 8
    for (int q = par; q < 4 * SB; q += 2) {
      const uint4 v = *reinterpret_cast<const uint4 *>(d + ((long)(q >> 2) * 64 + 16 * (q & 3)) * 8);
      const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
      for (int e = 0; e < 8; ++e)
        s[e] += __uint_as_float(e & 1 ? w[e >> 1] & 0xffff0000u : w[e >> 1] << 16);
    }
    float t = s[0];
#pragma unroll
    for (int e = 1; e < 8; ++e) t += s[e];
#pragma unroll
    for (int e = 0; e < 8; ++e) t += __shfl(s[e], lane | 32, 64);
    if (par == 0) net.gb[net.b_at(l) + 32 * blk + o] = t;
    return;
  }
  const int l = net.layer_of(blk), I = net.in(l), nti = I / 32;
  const int t = blk - net.tile_at(l), to = t / nti, ti = t - to * nti;
  const uint16_t *pa[2], *pb[2];
#pragma unroll
  for (int x = 0; x < 2; ++x) {
    pa[x] = net.dT + net.d_at(l) + (long)(to * 2 + x) * SB * 512 + lane * 8;
    pb[x] = net.aT + net.a_at(l) + (long)(ti * 2 + x) * SB * 512 + lane * 8;
  }
  const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
  f32x4 acc[2][2], sum[2][2];
#pragma unroll
  for (int x = 0; x < 2; ++x)
#pragma unroll
    for (int y = 0; y < 2; ++y) acc[x][y] = sum[x][y] = zero;
  constexpr int PD = 8;
  bf16x8 a[PD][2], b[PD][2];
  auto load = [&](int p, int s) {
    s = min(s, SB - 1);
#pragma unroll
    for (int x = 0; x < 2; ++x) {
      a[p][x] = *reinterpret_cast<const bf16x8 *>(pa[x] + (long)s * 512);
      b[p][x] = *reinterpret_cast<const bf16x8 *>(pb[x] + (long)s * 512);
    }
  };
#pragma unroll
  for (int p = 0; p < PD; ++p) load(p, p);
  int c = 0;
  auto one = [&](int p) {
#pragma unroll
    for (int x = 0; x < 2; ++x)
#pragma unroll
      for (int y = 0; y < 2; ++y) acc[x][y] = mfma(a[p][x], b[p][y], acc[x][y]);
    if (++c == per && per < SB) {
      c = 0;
#pragma unroll
      for (int x = 0; x < 2; ++x)
#pragma unroll
        for (int y = 0; y < 2; ++y) {
          sum[x][y] += acc[x][y];
          acc[x][y] = zero;
        }
    }
  };
  int s = 0;
  for (; s + PD < SB; s += PD)  // no branch past a load: see the chain's steps
#pragma unroll
    for (int p = 0; p < PD; ++p) {
      one(p);
      load(p, s + p + PD);
    }
#pragma unroll
  for (int p = 0; p < PD; ++p) {
    if (s + p >= SB) break;
    one(p);
  }
#pragma unroll
  for (int x = 0; x < 2; ++x)
#pragma unroll
    for (int y = 0; y < 2; ++y) {
      const f32x4 g = per < SB ? sum[x][y] : acc[x][y];
      float *gw = net.gw + net.w_at(l) + (long)(to * 32 + x * 16 + 4 * kq) * I + ti * 32 + y * 16 + row;
#pragma unroll
      for (int v = 0; v < 4; ++v) gw[(long)v * I] = g[v];
    }
}

// sums of squares of the misses, 256 consecutive values of the batch each
__global__ __launch_bounds__(256) void mlp_loss_kernel(const float *__restrict__ Y,
                                                       const float *__restrict__ T,
                                                       float *__restrict__ part, long n) {
  __shared__ float red[256];
  const long t = (long)blockIdx.x * 256 + threadIdx.x;
  const float d = t < n ? Y[t] - T[t] : 0.f;
  red[threadIdx.x] = d * d;
  __syncthreads();
  for (int s = 128; s > 0; s >>= 1) {
    if ((int)threadIdx.x < s) red[threadIdx.x] += red[threadIdx.x + s];
    __syncthreads();
  }
  if (threadIdx.x == 0) part[blockIdx.x] = red[0];
}

__device__ __forceinline__ float adam_step(float &w, float g, float &m1, float &m2,
                                           const MlpAdam &p, float wd) {
  const float gr = g + wd * w;
  const float a = p.b1 * m1 + (1.f - p.b1) * gr;
  const float b = p.b2 * m2 + (1.f - p.b2) * gr * gr;
  m1 = a;
  m2 = b;
  const float upd = (a / p.c1) / (sqrtf(b / p.c2) + p.eps);
  w = w - p.lr * upd;
  return w;
}

// Adam on the fp32 master weights and biases of the layers from l0 on, a
// workgroup per 32 x 32 tile, and the two packed bf16 copies of the tile: wp
// (rows = outputs, k = inputs) for the forward product, wtp (rows = inputs, k
// = outputs) for the way back.  UPDATE false: the copies alone.
// Bound by HBM or the last-level cache, 32 bytes a weight: 6.2 us for 622592
// weights (28 as eight launches).
template <bool UPDATE>
__global__ __launch_bounds__(256) void mlp_adam_kernel(MlpNet net, int l0, MlpAdam p) {
  __shared__ __attribute__((aligned(16))) uint16_t tile[32][40];
  const int blk = blockIdx.x + net.tile_at(l0), l = net.layer_of(blk);
  const int I = net.in(l), O = net.out(l), nti = I / 32;
  const int t = blk - net.tile_at(l), to = t / nti, ti = t - to * nti;
  const int tid = threadIdx.x, r = tid >> 3, c = 4 * (tid & 7);
  const long at = net.w_at(l) + (long)(to * 32 + r) * I + ti * 32 + c;
  f32x4 w = *reinterpret_cast<const f32x4 *>(net.w + at);
  if (UPDATE) {
    const f32x4 g = *reinterpret_cast<const f32x4 *>(net.gw + at);
    f32x4 m1 = *reinterpret_cast<const f32x4 *>(net.mw + at);
    f32x4 m2 = *reinterpret_cast<const f32x4 *>(net.vw + at);
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      float x = w[v], y = m1[v], z = m2[v];
      adam_step(x, g[v], y, z, p, p.wd);
      w[v] = x; m1[v] = y; m2[v] = z;
    }
    *reinterpret_cast<f32x4 *>(net.w + at) = w;
    *reinterpret_cast<f32x4 *>(net.mw + at) = m1;
    *reinterpret_cast<f32x4 *>(net.vw + at) = m2;
    if (ti == 0 && tid < 32) {
      const long o = net.b_at(l) + to * 32 + tid;
      adam_step(net.b[o], net.gb[o], net.mb[o], net.vb[o], p, 0.f);
    }
  }
  *reinterpret_cast<uint2 *>(&tile[r][c]) = f2bf4(w);
  __syncthreads();
  const int lane = tid & 63, row = lane & 15, k = 8 * (lane >> 4), h = (tid >> 6) & 1;
  if (tid < 128) {
    *reinterpret_cast<uint4 *>(net.wp + net.w_at(l) + ((long)(to * 2 + h) * nti + ti) * 512 + lane * 8) =
        *reinterpret_cast<const uint4 *>(&tile[16 * h + row][k]);
  } else {
    uint32_t v[4];
#pragma unroll
    for (int e = 0; e < 4; ++e)
      v[e] = (uint32_t)tile[k + 2 * e][16 * h + row] |
             (uint32_t)tile[k + 2 * e + 1][16 * h + row] << 16;
    *reinterpret_cast<uint4 *>(net.wtp + net.w_at(l) + ((long)(ti * 2 + h) * (O / 32) + to) * 512 + lane * 8) =
        make_uint4(v[0], v[1], v[2], v[3]);
  }
}

// Column features of the radiative box: for column (i, j) and cell kz of the
// interior, x[col][f*nz + kz] = (feat_f - mu[f*nz+kz]) / sd[f*nz+kz] with
// feat = (ln ro, ln T, |B|^2), T = (gm-1) ei, and with nfeat == 4 the
// horizontal Laplacian of ln T at stride FT_H (x and y periodic: neighbours
// wrap inside the interior).  Columns run i fastest.
// A block reads 64 consecutive x cells (one y row) x 32 heights with lanes
// along x, and ln T of the FT_H cells beside them, so that the x neighbours'
// logarithms are taken once, from LDS; then it writes each column's 32
// heights, four per lane.  Each XCD takes a contiguous range of blocks, x
// fastest, then y: the rows FT_H above and below are in its L2 (2.6 GB read
// at 384^3, of 2.3 without any row twice).
// Bound by HBM: 3.1 GB at 4.2 TB/s, 722 us at 384^3; with every neighbour's
// logarithm taken anew and the rows spread over the XCDs 943.
constexpr int FT_X = 64, FT_Z = 32, FT_H = 4;
typedef uint16_t u16x4u __attribute__((ext_vector_type(4), aligned(2)));

__global__ __launch_bounds__(256) void column_features_kernel(
    Fld<const double> q, Shape sh, double gm, const float *__restrict__ mu,
    const float *__restrict__ sd, uint16_t *__restrict__ X, float *__restrict__ Xf, int nfeat,
    int nbx, int nb) {
  __shared__ float tile[3][FT_Z][FT_X + 1];         // ln ro, |B|^2, Laplacian
  __shared__ float lnt[FT_Z][FT_X + 2 * FT_H + 1];  // ln T from x = i0 - FT_H on
  const int ni = sh.It - 2 * sh.mi, nj = sh.Jt - 2 * sh.mj, nz = sh.Kt - 2 * sh.mk;
  const int V = xcd_virtual_block(blockIdx.x, nb), rest = V / nbx;
  const int i0 = (V - rest * nbx) * FT_X, j = rest % nj, kz0 = rest / nj * FT_Z;
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  // the features end in FP32 (then BF16): logarithms in FP32 of the FP64
  // arguments, sums in FP64
  auto ln_t = [&](int c) { return logf((float)((gm - 1.0) * q.q[7][c])); };
  if (nfeat == 4) {
    static_assert(FT_Z * 2 * FT_H == 256, "a thread per cell beside the tile");
    const int r = threadIdx.x / (2 * FT_H), h = threadIdx.x % (2 * FT_H);
    const int p = h < FT_H ? h - FT_H : FT_X + h - FT_H;  // from i0
    const int i = ((i0 + p) % ni + ni) % ni;
    if (kz0 + r < nz) lnt[r][p + FT_H] = ln_t(sh.idx(sh.mi + i, sh.mj + j, sh.mk + kz0 + r));
  }
  const int i = (i0 + lane) % ni;  // lanes past the row's end: neighbours of its last cells
  const int up = ((j + FT_H) % nj - j) * sh.It, dn = ((j - FT_H % nj + nj) % nj - j) * sh.It;
  float y[FT_Z / 4][2];
#pragma unroll
  for (int m = 0; m < FT_Z / 4; ++m) {
    const int r = wv + 4 * m;
    if (kz0 + r >= nz) break;
    const int c = sh.idx(sh.mi + i, sh.mj + j, sh.mk + kz0 + r);
    const double bx = q.q[4][c], by = q.q[5][c], bz = q.q[6][c];
    tile[0][r][lane] = logf((float)q.q[0][c]);
    lnt[r][lane + FT_H] = ln_t(c);
    tile[1][r][lane] = (float)(bx * bx + by * by + bz * bz);
    if (nfeat == 4) {
      y[m][0] = ln_t(c + up);
      y[m][1] = ln_t(c + dn);
    }
  }
  __syncthreads();
  if (nfeat == 4) {
#pragma unroll
    for (int m = 0; m < FT_Z / 4; ++m) {
      const int r = wv + 4 * m;
      if (kz0 + r >= nz) break;
      const double s = (double)lnt[r][lane + 2 * FT_H] + (double)lnt[r][lane] + (double)y[m][0] +
                       (double)y[m][1];
      tile[2][r][lane] = (float)(s - 4.0 * (double)lnt[r][lane + FT_H]);
    }
    __syncthreads();
  }
  // write: 8 lanes along the heights of one (column, feature) pair
  const int zl = 4 * (threadIdx.x & 7), kz = kz0 + zl;
  if (kz >= nz) return;  // nz is a multiple of 8
  for (int f = 0; f < nfeat; ++f) {
    float m4[4], s4[4];
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      m4[v] = mu[f * nz + kz + v];
      s4[v] = sd[f * nz + kz + v];
    }
#pragma unroll
    for (int il = threadIdx.x >> 3; il < FT_X; il += 32) {
      if (i0 + il >= ni) break;
      f32x4 x;
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const float t = f == 1 ? lnt[zl + v][il + FT_H] : tile[f ? f - 1 : 0][zl + v][il];
        x[v] = (t - m4[v]) / s4[v];
      }
      const long at = ((long)j * ni + i0 + il) * nfeat * nz + f * nz + kz;
      const u16x4u h = {f2bf(x[0]), f2bf(x[1]), f2bf(x[2]), f2bf(x[3])};
      *reinterpret_cast<u16x4u *>(X + at) = h;
      if (Xf) *reinterpret_cast<f32x4u *>(Xf + at) = x;
    }
  }
}

// Sums over chosen rows of a row-major [..][W] array, by column, in FP64: of
// the values and of their magnitudes, or (SQ) of the squared distances from
// the mean.  A block takes 64 columns and a share of the rows; its sums go to
// p0 (p1) [share][column].
// Bound by HBM: the rows are read twice (the mean first, so that no digits
// cancel).  14746 x 1536 and their targets: 0.2 ms, where FP64 copies of the
// rows and library reductions took 1.1.
template <typename T, bool SQ>
__global__ __launch_bounds__(256) void moments_kernel(const T *__restrict__ x,
                                                      const long long *__restrict__ rows, long n,
                                                      int W, const double *__restrict__ mean,
                                                      double *__restrict__ p0,
                                                      double *__restrict__ p1, long share) {
  __shared__ double red[2][4][64];
  const int lane = threadIdx.x & 63;
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int col = blockIdx.x * 64 + lane, c = min(col, W - 1);
  const long r1 = min(n, (blockIdx.y + 1) * share);
  const double m = SQ ? mean[c] : 0.0;
  double a = 0.0, b = 0.0;
#pragma unroll 8
  for (long r = blockIdx.y * share + wv; r < r1; r += 4) {
    const double v = (double)x[rows[r] * W + c];
    if (SQ) {
      a += (v - m) * (v - m);
    } else {
      a += v;
      b += fabs(v);
    }
  }
  red[0][wv][lane] = a;
  red[1][wv][lane] = b;
  __syncthreads();
  if (wv == 0 && col < W) {
    const long at = (long)blockIdx.y * W + col;
    p0[at] = (red[0][0][lane] + red[0][1][lane]) + (red[0][2][lane] + red[0][3][lane]);
    if (!SQ) p1[at] = (red[1][0][lane] + red[1][1][lane]) + (red[1][2][lane] + red[1][3][lane]);
  }
}

// mean and mean magnitude, or (SQ) the standard deviation, from the shares
template <bool SQ>
__global__ __launch_bounds__(64) void moments_final_kernel(const double *__restrict__ p0,
                                                           const double *__restrict__ p1, long n,
                                                           int W, int shares,
                                                           double *__restrict__ o0,
                                                           double *__restrict__ o1) {
  const int col = blockIdx.x * 64 + threadIdx.x;
  if (col >= W) return;
  double a = 0.0, b = 0.0;
#pragma unroll 16
  for (int s = 0; s < shares; ++s) {
    a += p0[(long)s * W + col];
    if (!SQ) b += p1[(long)s * W + col];
  }
  if (SQ) {
    o0[col] = sqrt(a / (n ? (double)(n - 1) : 0.0));
  } else {
    o0[col] = a / (double)n;
    o1[col] = b / (double)n;
  }
}

// (x - mean) / sd in FP64, four columns a thread, to bf16 (by way of FP32) or
// FP32
template <typename T, bool BF>
__global__ __launch_bounds__(256) void normalize_kernel(const T *__restrict__ x, long n4, int W,
                                                        const double *__restrict__ mean,
                                                        const double *__restrict__ sd,
                                                        void *__restrict__ out) {
  typedef T x4 __attribute__((ext_vector_type(4), aligned(sizeof(T))));
  const long t = (long)blockIdx.x * 256 + threadIdx.x;
  if (t >= n4) return;
  const int c = (int)(4 * t % W);
  const x4 v = reinterpret_cast<const x4 *>(x)[t];
  f32x4 y;
#pragma unroll
  for (int e = 0; e < 4; ++e) y[e] = (float)(((double)v[e] - mean[c + e]) / sd[c + e]);
  if (BF)
    reinterpret_cast<uint2 *>(out)[t] = f2bf4(y);
  else
    reinterpret_cast<f32x4 *>(out)[t] = y;
}

// residual indicator per column: relative L2 of (mlp - rt) over the column
// above `tol` -> flag = 1; corr (optional) receives rt - mlp on every cell
__global__ void column_residual_kernel(const float *__restrict__ Y, Shape sh,
                                       const float *__restrict__ mu, const float *__restrict__ sd,
                                       const double *__restrict__ q_rt, int *__restrict__ flag,
                                       float tol, double *__restrict__ corr) {
  const int ni = sh.It - 2 * sh.mi, nj = sh.Jt - 2 * sh.mj, nz = sh.Kt - 2 * sh.mk;
  const long col = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (col >= (long)ni * nj) return;
  const int i = (int)(col % ni), j = (int)(col / ni);
  double num = 0.0, den = 0.0;
  for (int kz = 0; kz < nz; ++kz) {
    const int c = sh.idx(sh.mi + i, sh.mj + j, sh.mk + kz);
    const double qr = q_rt[c];
    const double qm = (double)(Y[col * nz + kz] * sd[kz] + mu[kz]);
    if (corr) corr[c] = qr - qm;
    num += (qm - qr) * (qm - qr);
    den += qr * qr;
  }
  flag[col] = (num > (double)tol * tol * den) ? 1 : 0;
}

// ------------------------------------------------------------- launchers
namespace {

// columns from which inference takes 64 to a workgroup: fewer leave CUs idle
constexpr int MLP_TALL = 8192;
// A layer of its own (WIDE) takes 64 columns to a workgroup where that still
// makes this many of them, 16 otherwise (1536-2048-2048-2048-384, 2048 columns:
// 118 and 162 us; 1024: 110 and 92; 1536-1024-1024-1024-384, 4096: 88 and 125,
// 2048: 81 and 68).
constexpr int MLP_LAYER_TALL = 192;
// Hidden widths above this go by layers in inference also where LDS would hold
// them: a small batch has a few workgroups, and each would read all weights
// (1536-1536-1536-1536-384, one column: 42 us for 160, 16384: 387 for 613).
// Training, 16 columns a workgroup, stays in one launch (batch of 4096: 428 us
// for 616).
constexpr int MLP_LAYERS = 1024;
constexpr int LDS_BYTES = 160 * 1024;
// features of X that a 16-column workgroup stages at a time
int x_width(int n_in) { return n_in < 2048 ? n_in : 2048; }
// LDS of a workgroup of ns columns: two activation buffers of width bw (none
// where they live in global memory) and, beside them, xw features of X
size_t chain_lds(int ns, int bw, int xw) {
  return sizeof(uint16_t) * ns * ((bw ? 2 * (bw + 8) : 0) + (xw ? xw + 8 : 0));
}

// workgroups per tile of columns for a layer of its own: `per` row tiles each
int wide_rows(const MlpNet &net, int phase, int per) {
  const int O = phase < net.nl ? net.out(phase) : net.in(2 * net.nl - 1 - phase);
  return (O / 16 + per - 1) / per;
}

template <int NT, int WAVES, int RT, int PD, bool TRAIN, bool WIDE>
hipError_t chain(hipStream_t st, const MlpNet &net, const uint16_t *X, int M, float *Y,
                 const MlpLoss &ls, const MlpField &fo, uint16_t *g0, uint16_t *g1, int bw,
                 int xoff, int xw, size_t bytes, int phase = 0) {
  auto k = mlp_chain_kernel<NT, WAVES, RT, PD, TRAIN, WIDE>;
  if (bytes > 65536) {
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(k),
                                       hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes);
    if (e != hipSuccess) return e;
  }
  const dim3 grid((M + 16 * NT - 1) / (16 * NT),
                  WIDE ? wide_rows(net, phase, WAVES * RT) : 1);
  hipLaunchKernelGGL(k, grid, dim3(64 * WAVES), bytes, st, net, X, M, Y, ls, fo, g0, g1, bw, xoff,
                     xw, phase);
  return hipGetLastError();
}

}  // namespace

bool mlp_is_wide(int n_in, int width) {
  return chain_lds(16, width, x_width(n_in)) + 1024 > (size_t)LDS_BYTES;
}
bool mlp_by_layers(int n_in, int n_hidden) {
  return n_hidden > MLP_LAYERS || mlp_is_wide(n_in, n_hidden);
}

hipError_t launch_mlp_forward(hipStream_t st, const MlpNet &net, int maxw, const uint16_t *X,
                              int M, float *Y, const MlpField &fo, uint16_t *g0, uint16_t *g1) {
  const int n_in = net.n_in, n_hidden = net.n_hidden;
  const MlpLoss none{};
  constexpr int NT = 4, NS = 16 * NT;
  if (mlp_by_layers(n_in, n_hidden)) {
    const int xw = x_width(std::max(n_in, n_hidden));
    hipError_t e = hipSuccess;
    for (int p = 0; p < net.nl && e == hipSuccess; ++p)
      e = (long)((M + NS - 1) / NS) * wide_rows(net, p, 16) >= MLP_LAYER_TALL
              ? chain<NT, 8, 2, 2, false, true>(st, net, X, M, Y, none, fo, g0, g1, maxw, 0,
                                                MLP_X_TALL,
                                                sizeof(uint16_t) * NS * 2 * (MLP_X_TALL + 8), p)
              : chain<1, 16, 1, 4, false, true>(st, net, X, M, Y, none, fo, g0, g1, maxw, 0, xw,
                                                chain_lds(16, 0, xw), p);
    return e;
  }
  // X passes through the place of the second buffer, two chunks of it (the
  // input layer writes the first buffer)
  const size_t tall = sizeof(uint16_t) * NS *
                      (n_hidden + 8 + std::max(n_hidden + 8, 2 * (MLP_X_TALL + 8)));
  if (M >= MLP_TALL && tall <= (size_t)LDS_BYTES)
    return chain<NT, 8, 2, 2, false, false>(st, net, X, M, Y, none, fo, g0, g1, n_hidden,
                                            NS * (n_hidden + 8), MLP_X_TALL, tall);
  const int xw = x_width(n_in);
  return chain<1, 16, 1, 4, false, false>(st, net, X, M, Y, none, fo, g0, g1, n_hidden,
                                          32 * (n_hidden + 8), xw, chain_lds(16, n_hidden, xw));
}

hipError_t launch_mlp_grad(hipStream_t st, const MlpNet &net, bool wide, int maxw,
                           const uint16_t *X, int M, const MlpLoss &ls, float *Y, uint16_t *g0,
                           uint16_t *g1) {
  const MlpField none{};
  const int xw = x_width(wide ? std::max(net.n_in, maxw) : net.n_in);
  hipError_t e = hipSuccess;
  if (wide)
    for (int p = 0; p < 2 * net.nl - 1 && e == hipSuccess; ++p)
      e = chain<1, 16, 1, 4, true, true>(st, net, X, M, Y, ls, none, g0, g1, maxw, 0, xw,
                                         chain_lds(16, 0, xw), p);
  else
    e = chain<1, 16, 1, 4, true, false>(st, net, X, M, Y, ls, none, g0, g1, maxw, 32 * (maxw + 8),
                                        xw, chain_lds(16, maxw, xw));
  if (e != hipSuccess) return e;
  int splits = 16;  // equal sums of whole k-steps
  while (M % (32 * splits)) --splits;
  hipLaunchKernelGGL(mlp_wgrad_kernel, dim3(net.tiles() + net.bias_tiles()), dim3(64), 0, st,
                     net, M / 32, M / 32 / splits, net.tiles());
  return hipGetLastError();
}

hipError_t launch_mlp_loss(hipStream_t st, const float *Y, const float *T, float *part, long n,
                           int *parts) {
  *parts = (int)((n + 255) / 256);
  hipLaunchKernelGGL(mlp_loss_kernel, dim3(*parts), dim3(256), 0, st, Y, T, part, n);
  return hipGetLastError();
}

hipError_t launch_mlp_adam(hipStream_t st, const MlpNet &net, const MlpAdam &p) {
  hipLaunchKernelGGL((mlp_adam_kernel<true>), dim3(net.tiles()), dim3(256), 0, st, net, 0, p);
  return hipGetLastError();
}

hipError_t launch_mlp_pack(hipStream_t st, const MlpNet &net, int layer) {
  const int tiles = net.in(layer) / 32 * (net.out(layer) / 32);
  hipLaunchKernelGGL((mlp_adam_kernel<false>), dim3(tiles), dim3(256), 0, st, net, layer,
                     MlpAdam{});
  return hipGetLastError();
}

hipError_t launch_column_features(hipStream_t st, const Fld<const double> &q, const Shape &sh,
                                  double gm, const float *mu, const float *sd, uint16_t *X,
                                  float *Xf, int nfeat) {
  const int ni = sh.It - 2 * sh.mi, nj = sh.Jt - 2 * sh.mj, nz = sh.Kt - 2 * sh.mk;
  if (nfeat < 3 || nfeat > 4 || nz % 4) return hipErrorInvalidValue;
  const int nbx = (ni + FT_X - 1) / FT_X;
  const long nb = (long)nbx * nj * ((nz + FT_Z - 1) / FT_Z);
  if (nb > 2147483647L) return hipErrorInvalidValue;
  hipLaunchKernelGGL(column_features_kernel, dim3((unsigned)nb), dim3(256), 0, st, q, sh, gm, mu,
                     sd, X, Xf, nfeat, nbx, (int)nb);
  return hipGetLastError();
}

template <typename T>
static hipError_t moments(hipStream_t st, const T *x, const long long *rows, long n, int W,
                          double *mean, double *sd, double *mean_abs, double *work) {
  const dim3 grid((W + 63) / 64, MLP_SHARES), one((W + 63) / 64);
  const long share = (n + MLP_SHARES - 1) / MLP_SHARES;
  double *p1 = work + (long)MLP_SHARES * W;
  hipLaunchKernelGGL((moments_kernel<T, false>), grid, dim3(256), 0, st, x, rows, n, W, nullptr,
                     work, p1, share);
  hipLaunchKernelGGL((moments_final_kernel<false>), one, dim3(64), 0, st, work, p1, n, W,
                     MLP_SHARES, mean, mean_abs);
  hipLaunchKernelGGL((moments_kernel<T, true>), grid, dim3(256), 0, st, x, rows, n, W, mean, work,
                     nullptr, share);
  hipLaunchKernelGGL((moments_final_kernel<true>), one, dim3(64), 0, st, work, nullptr, n, W,
                     MLP_SHARES, sd, nullptr);
  return hipGetLastError();
}

hipError_t launch_moments(hipStream_t st, const void *x, bool f64, const long long *rows, long n,
                          int W, double *mean, double *sd, double *mean_abs, double *work) {
  if (f64)
    return moments(st, static_cast<const double *>(x), rows, n, W, mean, sd, mean_abs, work);
  return moments(st, static_cast<const float *>(x), rows, n, W, mean, sd, mean_abs, work);
}

hipError_t launch_normalize(hipStream_t st, const void *x, bool f64, long n, int W,
                            const double *mean, const double *sd, void *out, bool bf16) {
  const long n4 = n * W / 4;
  const dim3 grid((unsigned)((n4 + 255) / 256));
  const double *xd = static_cast<const double *>(x);
  const float *xf = static_cast<const float *>(x);
  if (f64 && bf16)
    hipLaunchKernelGGL((normalize_kernel<double, true>), grid, dim3(256), 0, st, xd, n4, W, mean, sd, out);
  else if (f64)
    hipLaunchKernelGGL((normalize_kernel<double, false>), grid, dim3(256), 0, st, xd, n4, W, mean, sd, out);
  else if (bf16)
    hipLaunchKernelGGL((normalize_kernel<float, true>), grid, dim3(256), 0, st, xf, n4, W, mean, sd, out);
  else
    hipLaunchKernelGGL((normalize_kernel<float, false>), grid, dim3(256), 0, st, xf, n4, W, mean, sd, out);
  return hipGetLastError();
}

hipError_t launch_column_residual(hipStream_t st, const float *Y, const Shape &sh,
                                  const float *mu, const float *sd, const double *q_rt, int *flag,
                                  float tol, double *corr) {
  const long n = (long)(sh.It - 2 * sh.mi) * (sh.Jt - 2 * sh.mj);
  hipLaunchKernelGGL(column_residual_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st,
                     Y, sh, mu, sd, q_rt, flag, tol, corr);
  return hipGetLastError();
}

}  // namespace misohip
