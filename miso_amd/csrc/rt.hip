// Grey short-characteristics radiative transfer on the GPU (FP64), the
// counterpart of MISO's CPU-only rt::RT (miso/include/miso/rt_host.hpp).
//
// The sweep along a ray's dominant axis is sequential plane by plane, but
// within a plane every node is independent (its four upwind nodes all lie in
// the previous plane), and the 24 rays are independent.  So one launch
// advances all rays by one plane: rays x transverse nodes of that plane.
// Per-ray constants (dominant axis, sweep order, bilinear weights, ds) are
// computed on the host with the reference's expressions, float narrowing
// included (rt_host.hpp:461-508).
//
// Device layout: rint[(n * Kt + k) * Jt + j) * It + i] (x fastest); kappa
// and S as the MHD fields.  The RT lattice is ib0 = margin - is ...
// ib1 = ib0 + size on every axis (rt_host.hpp:127-154).
// A ray whose dominant axis is x sweeps planes of fixed i, whose nodes lie
// It apart in that layout; such rays ("transposed" rays, R.tr) keep their
// intensities y-fastest instead, rint[(n * Kt + k) * It + i) * Jt + j], and
// read kappa and S from copies in the same layout, so their planes are
// contiguous as well.  Per node the arithmetic does not change.
#include "launch.hpp"

namespace misohip {

// EVERY: the quotient is formed for every node and dropped where dtau is small:
// without a branch the nodes of a thread interleave (the patched sweep of 211 x
// 150 x 187, three iterations, 4.55 -> 3.91 ms).  A thread of one node has
// nothing to interleave and forms it only where it is used (one launch per
// plane, every ray x-fastest: 384^2 x 27 33.0 -> 25.3 ms, 128^3 6.86 -> 5.96).
template <bool EVERY>
__device__ __forceinline__ double rt_integrate(double Iu, double Su, double Sd, double dtau) {
  const double eps_tau = 1.e-4;
  const double exp_dtau = exp(-dtau);
  const double u0 = 1.0 - exp_dtau;
  double u1;
  if constexpr (EVERY) {
    double quot = u0 / dtau;
    asm("" : "+v"(quot));
    u1 = dtau < eps_tau ? 0.5 * dtau : 1.0 - quot;
  } else {
    u1 = dtau < eps_tau ? 0.5 * dtau : 1.0 - (u0 / dtau);
  }
  return Iu * exp_dtau + (u0 - u1) * Su + u1 * Sd;
}

// one node from its four upwind neighbours (00: same transverse position,
// 10: one step back along b, 01: along c, 11: both) and its own kappa, S
template <bool EVERY>
__device__ __forceinline__ double rt_node(const RtRay &R, double I00, double I10, double I01,
                                          double I11, double S00, double S10, double S01,
                                          double S11, double K00, double K10, double K01,
                                          double K11, double kc, double sc) {
  const double iu = R.w00 * I00 + R.w10 * I10 + R.w01 * I01 + R.w11 * I11;
  const double su = R.w00 * S00 + R.w10 * S10 + R.w01 * S01 + R.w11 * S11;
  const double ku = R.w00 * K00 + R.w10 * K10 + R.w01 * K01 + R.w11 * K11;
  const double dtau = 0.5 * (ku + kc) * R.ds;
  return rt_integrate<EVERY>(iu, su, sc, dtau);
}

// The solve's convergence measure is the max over lattice nodes of
// |I_end - I_start| of an iteration, float-narrowed as util::max2 does
// (rt_host.hpp:612-629); positive floats order like their bit patterns.
// Every lattice node of a ray is either swept (exactly once per iteration,
// so the sweep takes the change from the value it overwrites) or on one of
// the ray's upwind faces (written once, by rt_incoming_kernel, which takes
// the change as well).  Workgroup maxima go
// by atomicMax into one of RT_PARTS slots, 32 words apart, then one small
// kernel reduces them.
__device__ __forceinline__ unsigned rt_change(double now, double before) {
  return __float_as_uint((float)fabs(now - before));
}

__device__ __forceinline__ void rt_block_max(unsigned best, unsigned *part) {
  __shared__ unsigned red[16];
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) best = max(best, (unsigned)__shfl_xor((int)best, o, 64));
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = best;
  __syncthreads();
  if (threadIdx.x == 0) {
    unsigned b = red[0];
    for (int w = 1; w < (int)(blockDim.x >> 6); ++w) b = max(b, red[w]);
    if (b) atomicMax(part + 32 * ((blockIdx.x + 7 * blockIdx.y) % RT_PARTS), b);
  }
}

// plane p of every ray of `rays` (blockIdx.y = entry, R.id = its slot)
__global__ __launch_bounds__(256) void rt_sweep_plane_kernel(double *__restrict__ I,
                                                             const double *__restrict__ kap_x,
                                                             const double *__restrict__ S_x,
                                                             const double *__restrict__ kap_y,
                                                             const double *__restrict__ S_y,
                                                             RtRays rays, int p, long ray_stride,
                                                             unsigned *part) {
  const RtRay &R = rays.r[blockIdx.y];
  if (p >= R.nplanes) return;  // uniform over the block
  const double *__restrict__ kap = R.tr ? kap_y : kap_x;
  const double *__restrict__ S = R.tr ? S_y : S_x;
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  unsigned best = 0u;
  if (t < R.nb * R.nc) {
    const int ib = t % R.nb, ic = t / R.nb;
    const int c = R.start + p * R.da + ib * R.db + ic * R.dc;  // cell index (kappa, S)
    const int c00 = c - R.ua;
    const int c10 = c00 - R.ub, c01 = c00 - R.uc, c11 = c00 - R.ub - R.uc;
    double *Ir = I + ray_stride * R.id;
    const double before = Ir[c];
    const double now =
        rt_node<false>(R, Ir[c00], Ir[c10], Ir[c01], Ir[c11], S[c00], S[c10], S[c01], S[c11],
                       kap[c00], kap[c10], kap[c01], kap[c11], kap[c], S[c]);
    Ir[c] = now;
    best = rt_change(now, before);
  }
  rt_block_max(best, part);
}

// Planes p0 .. p0 + P - 1 of every ray of `rays` in one launch, for rays with
// neighbouring nodes of a plane in different cache lines (x rays kept x-fastest)
// and a short c axis (nc < RT_MULTI_ROWS).  Such a sweep is bound by the lines
// that its loads touch, so no node is loaded twice where it can be helped: a
// workgroup owns the RT_MULTI_COLS columns u in [U0, U0 + W) of a ray over the
// whole c range (u, v as in the patches below), and computes plane by plane the
// cone u in [U0 - P, U0 + W) of nodes that its last plane depends on; the plane
// is kept in LDS, column u = -1 and row v = -1 (the upwind boundary nodes, which
// the sweep never writes) are read from memory.  Every node is computed by
// rt_node from the same values as in rt_sweep_plane_kernel, so the results are
// the same bits; cone nodes outside the owned columns are recomputed, not
// stored, and the cone's stale edge (u below U0 - P + s + 1 at step s) never
// reaches them.  Patches load a row and eight columns more for each that they
// own: three iterations of 384^2 x 27 10.5 ms for 15.5, of 1024^2 x 3 11.1 for
// 24.2, of 300 x 300 x 2 1.2 for 3.1.
constexpr int RT_MULTI_THREADS = 1024;

__global__ __launch_bounds__(RT_MULTI_THREADS) void rt_sweep_multi_kernel(double *__restrict__ I,
                                                             const double *__restrict__ kap,
                                                             const double *__restrict__ S,
                                                             RtRays rays, int p0, int P,
                                                             long ray_stride, unsigned *part) {
  constexpr int W = RT_MULTI_COLS, X = RT_MULTI_COLS + RT_MULTI_PLANES, ROWS = RT_MULTI_ROWS;
  constexpr int NT = RT_MULTI_THREADS, CPT = (X * ROWS + NT - 1) / NT;
  __shared__ double Il[ROWS][X], Kl[ROWS][X], Sl[ROWS][X];
  const RtRay &R = rays.r[blockIdx.y];
  const int U0 = blockIdx.x * W;
  // uniform over the workgroup
  if (p0 >= R.nplanes || U0 >= R.nb || R.nc + 1 > ROWS || P < 1 || P > RT_MULTI_PLANES) return;
  double *Ir = I + ray_stride * R.id;
  const int ext = W + P, ncell = ext * (R.nc + 1);
  const int pend = min(p0 + P, R.nplanes);
  // per cell: memory index at plane 0, role (0 none, 1 boundary, read every
  // plane; 2 computed; 3 computed and owned, its value before the sweep read
  // for the change; 4 the cone's far edge e = 0,
  // read for the plane before p0 only: never valid after it, and its node
  // may be written by another workgroup meanwhile), LDS position
  int off[CPT], role[CPT], ce[CPT], cr[CPT];
#pragma unroll
  for (int q = 0; q < CPT; ++q) {
    const int idx = threadIdx.x + q * NT;
    const int e = idx % ext, r = idx / ext;
    const int u = U0 - P + e, v = r - 1;
    ce[q] = e;
    cr[q] = r;
    role[q] = 0;
    off[q] = 0;
    if (idx >= ncell || u < -1 || u >= R.nb) continue;
    const int ib = R.sb > 0 ? u : R.nb - 1 - u;
    const int ic = R.sc > 0 ? v : R.nc - 1 - v;
    off[q] = R.start + ib * R.db + ic * R.dc;
    if (u == -1 || v == -1) role[q] = 1;
    else if (e == 0) role[q] = 4;
    else role[q] = (u >= U0 && u < U0 + W) ? 3 : 2;
  }
  // the plane before p0
#pragma unroll
  for (int q = 0; q < CPT; ++q)
    if (role[q]) {
      const int c = off[q] + (p0 - 1) * R.da;
      Il[cr[q]][ce[q]] = Ir[c];
      Kl[cr[q]][ce[q]] = kap[c];
      Sl[cr[q]][ce[q]] = S[c];
    }
  // kappa, S and the boundary (role 1) or before-sweep (role 3) intensity of
  // a plane's cells; loads run two planes ahead of the computation
  auto load = [&](int p, double *k, double *s, double *b) {
#pragma unroll
    for (int q = 0; q < CPT; ++q) {
      k[q] = s[q] = b[q] = 0.0;
      if (p < pend && role[q] && role[q] < 4) {
        const int c = off[q] + p * R.da;
        k[q] = kap[c];
        s[q] = S[c];
        if (role[q] == 1 || role[q] == 3) b[q] = Ir[c];
      }
    }
  };
  double kc[CPT], sc[CPT], bnd[CPT], k1[CPT], s1[CPT], b1[CPT];
  load(p0, kc, sc, bnd);
  load(p0 + 1, k1, s1, b1);
  __syncthreads();
  unsigned best = 0u;
  for (int p = p0; p < pend; ++p) {
    double kn[CPT], sn[CPT], bn[CPT];
    load(p + 2, kn, sn, bn);
    double in[CPT];
#pragma unroll
    for (int q = 0; q < CPT; ++q) {
      in[q] = bnd[q];
      if (role[q] == 2 || role[q] == 3) {
        const int r = cr[q], e = ce[q];
        in[q] = rt_node<false>(R, Il[r][e], Il[r][e - 1], Il[r - 1][e], Il[r - 1][e - 1], Sl[r][e],
                        Sl[r][e - 1], Sl[r - 1][e], Sl[r - 1][e - 1], Kl[r][e], Kl[r][e - 1],
                        Kl[r - 1][e], Kl[r - 1][e - 1], kc[q], sc[q]);
      }
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < CPT; ++q)
      if (role[q] && role[q] < 4) {
        Il[cr[q]][ce[q]] = in[q];
        Kl[cr[q]][ce[q]] = kc[q];
        Sl[cr[q]][ce[q]] = sc[q];
        if (role[q] == 3) {
          best = max(best, rt_change(in[q], bnd[q]));
          Ir[off[q] + p * R.da] = in[q];
        }
      }
#pragma unroll
    for (int q = 0; q < CPT; ++q) {
      kc[q] = k1[q];
      sc[q] = s1[q];
      bnd[q] = b1[q];
      k1[q] = kn[q];
      s1[q] = sn[q];
      b1[q] = bn[q];
    }
    __syncthreads();
  }
  rt_block_max(best, part);
}

hipError_t launch_rt_sweep_multi(hipStream_t st, double *I, const double *kap, const double *S,
                                 const RtRays &rays, int nrays, int p0, long ray_stride,
                                 int max_nb, unsigned *part) {
  dim3 grid((max_nb + RT_MULTI_COLS - 1) / RT_MULTI_COLS, nrays);
  hipLaunchKernelGGL(rt_sweep_multi_kernel, grid, dim3(RT_MULTI_THREADS), 0, st, I, kap, S, rays,
                     p0, RT_MULTI_PLANES, ray_stride, part);
  return hipGetLastError();
}

// Planes p0 .. p0 + P - 1 of every ray of `rays` in one launch.  Node
// coordinates are mirrored so that upwind is always one step back: u = ib
// (sb > 0) or nb - 1 - ib, likewise v.  A workgroup takes a patch of 64
// columns x W R rows of one ray (W waves): lane l of wave w holds column
// u0 + l of the rows v0 + w R ... + R - 1, the plane before in registers;
// u - 1 comes by a DPP lane shift, v - 1 from the row above (the last row of
// the wave before, through LDS).  The patch's first column and row are the
// upwind boundary (u = -1, v = -1: loaded at every plane, the sweep never
// writes it) or, in the patches after the first, P columns and rows of the
// neighbouring patch, computed again: step s leaves the first s of them
// stale, so the columns and rows from P on are right after P planes, and
// only those are stored.  No workgroup uses what another one of the launch
// writes: the plane before p0 is not written, and of the planes after it a
// patch uses the old intensities of owned and boundary nodes alone (patches
// with a boundary on one side load those of the overlap on the other as well,
// while the neighbour stores there, and drop them).
// Three register sets hold the plane before, the current plane's kappa, S
// and old intensities, and the next plane's, in flight meanwhile.
// The four rays that go the same way along the planes read the same kappa
// and S: their workgroups of one patch sit on one XCD, next to each other in
// launch order, so that HBM is read once for the four; the patches of an XCD
// are neighbours.
// rt_node forms each value from the same operands as rt_sweep_plane_kernel:
// the same bits.
// No rate bounds it alone: at 256^3, where an iteration's sweeps take 3.0 ms
// of 5.2, VALU issue is at half of its rate (84 instructions for each of 1.72 x
// the nodes, for the repeated columns and rows; 1.55 to 1.75 along the axes of
// 211 x 150 x 187) and 4.1 TB/s pass the L2, 30 bytes a node and ray; the rest is
// the latency of a plane's FP64 chain, with four waves a SIMD to cover it.  A
// launch per plane read the plane before again, and kappa and S once per ray.
// Radiative step of 256^3 23.4 -> 17.0 ms, cold solve of 211 x 150 x 187 14.2 ->
// 8.2 ms.  (Tiles marched in wavefront order, which repeat nothing, read
// kappa and S once per ray and start and end with an idle chip: 19.4 and
// 10.6 ms.)
template <int R> struct RtTilePlane {
  double i[R], k[R], s[R];  // own rows; i: before the sweep, then after it
  double ih, kh, sh;        // the row above them
};

template <int R, int W, bool THIN>
__global__ __launch_bounds__(64 * W) void rt_sweep_tile_kernel(
    double *__restrict__ I, const double *__restrict__ kap_x, const double *__restrict__ S_x,
    const double *__restrict__ kap_y, const double *__restrict__ S_y, RtRays rays, RtPatches pt,
    int p0, int P, long ray_stride, unsigned *part) {
  constexpr int NR = W * R;
  __shared__ double edge[2][W][64];
  // blocks of one XCD (blockIdx % 8): consecutive patches, each for the
  // pt.same rays of its group in turn
  const int xcd = blockIdx.x % 8, idx = blockIdx.x / 8;
  const int patch = xcd * pt.per_xcd + idx / pt.same;
  int g = 0;
  while (g < pt.groups && patch >= pt.start[g + 1]) ++g;
  if (g == pt.groups) return;  // uniform over the workgroup, as are all below
  const RtRay &Q = rays.r[g * pt.same + idx % pt.same];
  const int na = rt_patches(Q.nb, 64, P);
  const int a = (patch - pt.start[g]) % na, b = (patch - pt.start[g]) / na;
  if (p0 >= Q.nplanes || b >= rt_patches(Q.nc, NR, P)) return;
  const double *__restrict__ kap = Q.tr ? kap_y : kap_x;
  const double *__restrict__ S = Q.tr ? S_y : S_x;
  double *Ir = I + ray_stride * Q.id;
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int pend = min(p0 + P, Q.nplanes);
  const int u0 = rt_patch_first(a, 64, P), v0 = rt_patch_first(b, NR, P);
  const int u_own = a ? u0 + P : 0, v_own = b ? v0 + P : 0;
  // columns and rows past the ray's end load its last ones and store nothing
  const int u = u0 + lane, uc = min(u, Q.nb - 1);
  const bool own = u >= u_own && u < Q.nb, bound = u < 0;
  // a node's address: a row's first node (ib = -1), uniform over the wave, and
  // the lane's byte offset from it (0 .. 8 (nb + 1) db, below 4 GiB: the host
  // checks that)
  auto byte_of = [&](int ub) {
    return (unsigned)((Q.sb > 0 ? ub + 1 : Q.nb - ub) * Q.db) * 8u;
  };
  // old intensities are of use in owned nodes and on the boundary: in a patch
  // without boundary rows the columns that are not owned load the nearest
  // owned one, in one without boundary columns the rows likewise
  const unsigned col = byte_of(uc);
  const unsigned col_i = byte_of(min(max(u, a && b ? u_own : -1), Q.nb - 1));
  auto row = [&](int v) {
    v = max(min(v, Q.nc - 1), -1);
    return Q.start - Q.db + (Q.sc > 0 ? v : Q.nc - 1 - v) * Q.dc;
  };
  const int vw = v0 + w * R;
  int off[R], off_i[R];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    off[r] = row(vw + r);
    off_i[r] = row(max(vw + r, a && b ? v_own : -1));
  }
  const int offh = row(vw - 1);
  // element q of the lane: the address as a scalar base (pinned, or the
  // compiler would fold the lane's part into it) plus 32 bits
  auto at = [](const double *q, unsigned byte) {
    unsigned long base = reinterpret_cast<unsigned long>(q);
    asm("" : "+s"(base));
    asm("" : "+v"(byte));
    return reinterpret_cast<__attribute__((address_space(1))) double *>(base + byte);
  };
  auto load = [&](RtTilePlane<R> &x, int p, const int *oi, unsigned ci) {
    const int d = p * Q.da;
    x.kh = *at(kap + (offh + d), col);
    x.sh = *at(S + (offh + d), col);
#pragma unroll
    for (int r = 0; r < R; ++r) {
      x.k[r] = *at(kap + (off[r] + d), col);
      x.s[r] = *at(S + (off[r] + d), col);
      x.i[r] = *at(Ir + (oi[r] + d), ci);
    }
    __builtin_amdgcn_sched_barrier(0);  // in flight before the plane is computed
  };
  auto exchange = [&](RtTilePlane<R> &x, int p) {
    edge[p & 1][w][lane] = x.i[R - 1];
    lds_barrier();
    x.ih = edge[p & 1][w ? w - 1 : 0][lane];
  };
  unsigned best = 0u;
  if (!THIN || vw < Q.nc) {
    RtTilePlane<R> x0, x1, x2;
    load(x0, p0 - 1, off, col);
    load(x1, p0, off_i, col_i);
    exchange(x0, p0 - 1);
    auto step = [&](const RtTilePlane<R> &b4, RtTilePlane<R> &x, RtTilePlane<R> &nx, int p) {
      load(nx, min(p + 1, pend - 1), off_i, col_i);
      double I01 = b4.ih, K01 = b4.kh, S01 = b4.sh;
      double I11 = lane_up(I01), K11 = lane_up(K01), S11 = lane_up(S01);
      double now[R];
#pragma unroll
      for (int r = 0; r < R; ++r) {
        const double I00 = b4.i[r], K00 = b4.k[r], S00 = b4.s[r];
        const double I10 = lane_up(I00), K10 = lane_up(K00), S10 = lane_up(S00);
        now[r] = rt_node<true>(Q, I00, I10, I01, I11, S00, S10, S01, S11, K00, K10, K01, K11,
                               x.k[r], x.s[r]);
        I01 = I00; K01 = K00; S01 = S00;
        I11 = I10; K11 = K10; S11 = S10;
      }
      if (own) {
#pragma unroll
        for (int r = 0; r < R; ++r)
          if (vw + r >= v_own && vw + r < Q.nc) {
            best = max(best, rt_change(now[r], x.i[r]));
            *at(Ir + (off[r] + p * Q.da), col) = now[r];
          }
      }
#pragma unroll
      for (int r = 0; r < R; ++r) x.i[r] = bound || vw + r < 0 ? x.i[r] : now[r];
      exchange(x, p);
    };
    for (int p = p0;;) {
      step(x0, x1, x2, p);
      if (++p >= pend) break;
      step(x1, x2, x0, p);
      if (++p >= pend) break;
      step(x2, x0, x1, p);
      if (++p >= pend) break;
    }
  } else {
    // THIN: rows past the ray's end: no stored node depends on them, and their
    // loads would be most of a thin ray's (elsewhere the branch costs more than
    // the few rows that it saves: slab solve of 384^2 x 27 2.95 -> 2.97 ms)
    for (int p = p0 - 1; p < pend; ++p) lds_barrier();
  }
  rt_block_max(best, part);
}

// Rows a wave holds, in patches of RT_ROWS and of RT_ROWS_SMALL rows.  Full
// launches read least with four (two: radiative step of 256^3 15.8 -> 17.2 ms,
// cold solve of 211 x 150 x 187 7.2 -> 7.9).  The short patches' launches leave
// most of the chip idle and run at the length of a plane's FP64 chain: ten
// waves of two rows instead of four of five hide more of it (slab solve of
// 384^2 x 27 3.21 -> 3.01 ms; five of four, uneven over the SIMDs, 3.31; loads
// two planes ahead 3.07).
constexpr int RT_R = 4, RT_R_SMALL = 2;

hipError_t launch_rt_sweep_tiles(hipStream_t st, double *I, const double *kap, const double *S,
                                 const double *kap_y, const double *S_y, const RtRays &rays,
                                 int nrays, int p0, int P, int rows, long ray_stride,
                                 unsigned *part) {
  RtPatches pt;
  pt.same = nrays % 4 == 0 ? 4 : 1;
  pt.groups = nrays / pt.same;
  pt.start[0] = 0;
  for (int g = 0; g < pt.groups; ++g) {
    int n = 0;
    for (int m = 0; m < pt.same; ++m) {
      const RtRay &Q = rays.r[g * pt.same + m];
      if (p0 < Q.nplanes) n = max(n, rt_patches(Q.nb, 64, P) * rt_patches(Q.nc, rows, P));
    }
    pt.start[g + 1] = pt.start[g] + n;
  }
  if (!pt.start[pt.groups]) return hipSuccess;
  pt.per_xcd = (pt.start[pt.groups] + 7) / 8;
  const dim3 grid(8 * pt.per_xcd * pt.same);
  if (rows == RT_ROWS_SMALL && P == RT_TILE_PLANES_THIN)
    hipLaunchKernelGGL((rt_sweep_tile_kernel<RT_R_SMALL, RT_ROWS_SMALL / RT_R_SMALL, true>), grid,
                       dim3(64 * RT_ROWS_SMALL / RT_R_SMALL), 0, st, I, kap, S, kap_y, S_y, rays,
                       pt, p0, P, ray_stride, part);
  else if (rows == RT_ROWS_SMALL)
    hipLaunchKernelGGL((rt_sweep_tile_kernel<RT_R_SMALL, RT_ROWS_SMALL / RT_R_SMALL, false>), grid,
                       dim3(64 * RT_ROWS_SMALL / RT_R_SMALL), 0, st, I, kap, S, kap_y, S_y, rays,
                       pt, p0, P, ray_stride, part);
  else
    hipLaunchKernelGGL((rt_sweep_tile_kernel<RT_R, RT_ROWS / RT_R, false>), grid,
                       dim3(64 * RT_ROWS / RT_R), 0, st, I, kap, S, kap_y, S_y, rays, pt, p0, P,
                       ray_stride, part);
  return hipGetLastError();
}

// The rays' upwind boundary nodes before a sweep (blockIdx.y = ray * 3 +
// axis): what the periodic halo self-exchange along z, y and x
// (rt_host.hpp:236-452: + rays copy node b1 into b0, - rays b0 into b1, over
// the full transverse extent), then the incoming boundaries of the physical
// faces in axis order (rt_host.hpp:50-101: the lattice's transverse range)
// leave there, in one pass: a node on several faces takes the value of the
// last physical one, or else the start value with every periodic coordinate
// moved to the far end.  That source lies on no face that this pass writes
// (where it would, so does the node itself, and takes the face's value), so
// the order of the threads does not matter.  Each node belongs to its lowest
// axis.  The change of the lattice nodes goes into the parts.
// Bound by the strided faces (x of an x-fastest ray, y of a y-fastest one: a
// cache line per node), which this pass reads and writes once.  As launches
// of their own, saving the faces, the exchange, the boundaries and the
// comparison read them four times: 155 us an iteration at 384^2 x 28, this
// pass 41 (radiative step of 256^3 17.0 -> 16.5 ms, cold solve of 211 x 150 x
// 187 8.2 -> 7.7 ms).
__global__ __launch_bounds__(256) void rt_incoming_kernel(double *__restrict__ I,
                                                          const double *__restrict__ S_x,
                                                          const double *__restrict__ S_y,
                                                          RtIncoming f, long ray_stride,
                                                          unsigned *part) {
  const int n = blockIdx.y / 3, a = blockIdx.y % 3;
  if (f.hi[a] <= f.lo[a]) return;  // uniform over the block
  const bool tr = (f.tr >> n) & 1u;
  // the face's nodes, the faster axis of the ray's layout first
  const int t0 = a == 0 ? 1 : a == 1 ? 0 : tr ? 1 : 0, t1 = 3 - a - t0;
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  unsigned best = 0u;
  if (t < f.tot[t0] * f.tot[t1]) {
    int x[3], up[3];
    bool on[3], in = true;
    x[t0] = t % f.tot[t0];
    x[t1] = t / f.tot[t0];
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      up[d] = ((f.pos[d] >> n) & 1u) ? f.lo[d] : f.hi[d];
      if (d == a) x[d] = up[d];
      on[d] = f.hi[d] > f.lo[d] && x[d] == up[d];
      in = in && x[d] >= f.lo[d] && x[d] <= f.hi[d];
    }
    if (!(a > 0 && on[0]) && !(a > 1 && on[1])) {
      auto at = [&](const int *q) {
        return tr ? ((long)q[2] * f.tot[0] + q[0]) * f.tot[1] + q[1]
                  : ((long)q[2] * f.tot[1] + q[1]) * f.tot[0] + q[0];
      };
      const long c = at(x);
      int kind = 0;
      double value = 0.0;
      int src[3];
      bool moved = false;
#pragma unroll
      for (int d = 0; d < 3; ++d) {
        src[d] = x[d];
        if (!on[d]) continue;
        const int side = up[d] == f.lo[d] ? 0 : 1;
        if (f.periodic[d]) {
          src[d] = side ? f.lo[d] : f.hi[d];
          moved = true;
        } else if (in && f.kind[2 * d + side] && ((f.moving[d] >> n) & 1u)) {
          kind = f.kind[2 * d + side];
          value = f.value[2 * d + side];
        }
      }
      if (kind || moved) {
        double *In = I + ray_stride * n;
        const double before = In[c];
        const double now = kind == 1 ? (tr ? S_y : S_x)[c] : kind == 2 ? 0.0
                         : kind ? value : In[at(src)];
        In[c] = now;
        if (in) best = rt_change(now, before);
      }
    }
  }
  rt_block_max(best, part);
}

// slot = max of the parts; the parts are cleared for the next iteration
__global__ __launch_bounds__(64) void rt_parts_reduce_kernel(unsigned *part, unsigned *slot,
                                                             int clear_only) {
  unsigned b = 0u;
  for (int s = threadIdx.x; s < RT_PARTS; s += 64) {
    b = max(b, part[32 * s]);
    part[32 * s] = 0u;
  }
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) b = max(b, (unsigned)__shfl_xor((int)b, o, 64));
  if (threadIdx.x == 0 && !clear_only) slot[0] = b;
}

// Q_rad = 4 pi kappa (J - S), J = sum_r w_r I_r in ray order, lattice nodes.
// A block covers 32 x 32 (i, j) nodes of one plane k; a ray kept y-fastest
// (tr_mask) is read along j into LDS and taken from there, the others along
// i, so every read is coalesced and each node sums its rays in order.
__global__ __launch_bounds__(256) void rt_qrad_kernel(const double *__restrict__ I,
                                                      const double *__restrict__ kap,
                                                      const double *__restrict__ S,
                                                      double *__restrict__ q, int lo_i, int lo_j,
                                                      int lo_k, int ni, int nj, int It, int Jt,
                                                      long ray_stride, int nrays, int tiles_i,
                                                      unsigned tr_mask, RtRays w) {
  __shared__ double tile[32][33];
  const int ti = blockIdx.x % tiles_i, tj = blockIdx.x / tiles_i, k = lo_k + blockIdx.y;
  const int l = threadIdx.x & 31, r0 = threadIdx.x >> 5;
  double J[4] = {0.0, 0.0, 0.0, 0.0};
  for (int n = 0; n < nrays; ++n) {
    const double *In = I + ray_stride * n;
    const double wq = w.r[n].wq;
    if ((tr_mask >> n) & 1u) {  // uniform over the block
      __syncthreads();
#pragma unroll
      for (int m = 0; m < 4; ++m) {
        const int il = r0 + 8 * m, i = ti * 32 + il, j = tj * 32 + l;
        if (i < ni && j < nj) tile[il][l] = In[((long)k * It + lo_i + i) * Jt + lo_j + j];
      }
      __syncthreads();
#pragma unroll
      for (int m = 0; m < 4; ++m) J[m] += wq * tile[l][r0 + 8 * m];
    } else {
#pragma unroll
      for (int m = 0; m < 4; ++m) {
        const int i = ti * 32 + l, j = tj * 32 + r0 + 8 * m;
        if (i < ni && j < nj) J[m] += wq * In[((long)k * Jt + lo_j + j) * It + lo_i + i];
      }
    }
  }
#pragma unroll
  for (int m = 0; m < 4; ++m) {
    const int i = ti * 32 + l, j = tj * 32 + r0 + 8 * m;
    if (i < ni && j < nj) {
      const long c = ((long)k * Jt + lo_j + j) * It + lo_i + i;
      q[c] = 4.0 * 3.14159265358979323846 * kap[c] * (J[m] - S[c]);
    }
  }
}

hipError_t launch_rt_sweep_plane(hipStream_t st, double *I, const double *kap, const double *S,
                                 const double *kap_y, const double *S_y, const RtRays &rays,
                                 int nrays, int p, long ray_stride, int max_nodes,
                                 unsigned *part) {
  dim3 grid((max_nodes + 255) / 256, nrays);
  hipLaunchKernelGGL(rt_sweep_plane_kernel, grid, dim3(256), 0, st, I, kap, S, kap_y, S_y, rays,
                     p, ray_stride, part);
  return hipGetLastError();
}

// (Kt, Jt, It) x-fastest -> (Kt, It, Jt) y-fastest, 32 x 32 tiles through LDS
__global__ __launch_bounds__(256) void rt_transpose_xy_kernel(const double *__restrict__ src,
                                                              double *__restrict__ dst, int It,
                                                              int Jt, int tiles_i) {
  __shared__ double tile[32][33];
  const int ti = blockIdx.x % tiles_i, tj = blockIdx.x / tiles_i, k = blockIdx.y;
  const long plane = (long)It * Jt * k;
  for (int r = threadIdx.x >> 5; r < 32; r += 8) {
    const int i = ti * 32 + (threadIdx.x & 31), j = tj * 32 + r;
    if (i < It && j < Jt) tile[r][threadIdx.x & 31] = src[plane + (long)j * It + i];
  }
  __syncthreads();
  for (int r = threadIdx.x >> 5; r < 32; r += 8) {
    const int j = tj * 32 + (threadIdx.x & 31), i = ti * 32 + r;
    if (i < It && j < Jt) dst[plane + (long)i * Jt + j] = tile[threadIdx.x & 31][r];
  }
}

// Every ray's field x-fastest (blockIdx.z = ray): 32 x 32 tiles of a plane,
// through LDS where the ray is kept y-fastest.  Bound by HBM (each value read
// and written once); a clone followed by a transpose of each y-fastest ray
// wrote those rays twice.  The others are copied 16 bytes a lane (by eights,
// through the same tiles: cold solve of 211 x 150 x 187 7.27 ms for 7.10, slab
// solve of 384^2 x 27 3.02 for 2.96).
__global__ __launch_bounds__(256) void rt_xfast_kernel(const double *__restrict__ I,
                                                       double *__restrict__ out, int It, int Jt,
                                                       int tiles_i, unsigned tr, long ray_stride) {
  __shared__ double tile[32][33];
  const int ti = blockIdx.x % tiles_i, tj = blockIdx.x / tiles_i, l = threadIdx.x & 31;
  const long plane = ray_stride * blockIdx.z + (long)It * Jt * blockIdx.y;
  if (!((tr >> blockIdx.z) & 1u)) {  // uniform over the block: a copy, 1024 values a block
    typedef double d2 __attribute__((ext_vector_type(2), aligned(8)));
    const int n = It * Jt, c0 = blockIdx.x * 1024 + 2 * threadIdx.x;
    const double *src = I + plane + c0;
    double *dst = out + plane + c0;
    if (c0 + 513 < n) {
      const d2 a = *reinterpret_cast<const d2 *>(src), b = *reinterpret_cast<const d2 *>(src + 512);
      *reinterpret_cast<d2 *>(dst) = a;
      *reinterpret_cast<d2 *>(dst + 512) = b;
    } else {
#pragma unroll
      for (int m = 0; m < 4; ++m) {
        const int q = (m & 1) + 512 * (m >> 1);
        if (c0 + q < n) dst[q] = src[q];
      }
    }
    return;
  }
#pragma unroll
  for (int m = 0; m < 4; ++m) {
    const int r = (threadIdx.x >> 5) + 8 * m, j = tj * 32 + l, i = ti * 32 + r;
    if (i < It && j < Jt) tile[r][l] = I[plane + (long)i * Jt + j];
  }
  __syncthreads();
#pragma unroll
  for (int m = 0; m < 4; ++m) {
    const int r = (threadIdx.x >> 5) + 8 * m, i = ti * 32 + l, j = tj * 32 + r;
    if (i < It && j < Jt) out[plane + (long)j * It + i] = tile[l][r];
  }
}

hipError_t launch_rt_xfast(hipStream_t st, const double *I, double *out, int It, int Jt, int Kt,
                           int nrays, unsigned tr) {
  const int ti = (It + 31) / 32, tj = (Jt + 31) / 32;
  hipLaunchKernelGGL(rt_xfast_kernel, dim3(ti * tj, Kt, nrays), dim3(256), 0, st, I, out, It, Jt,
                     ti, tr, (long)It * Jt * Kt);
  return hipGetLastError();
}

hipError_t launch_rt_transpose_xy(hipStream_t st, const double *src, double *dst, int It, int Jt,
                                  int Kt) {
  const int ti = (It + 31) / 32, tj = (Jt + 31) / 32;
  hipLaunchKernelGGL(rt_transpose_xy_kernel, dim3(ti * tj, Kt), dim3(256), 0, st, src, dst, It,
                     Jt, ti);
  return hipGetLastError();
}

hipError_t launch_rt_incoming(hipStream_t st, double *I, const double *S, const double *S_y,
                              const RtIncoming &f, long ray_stride, int nrays, unsigned *part) {
  int m = 1;
  for (int a = 0; a < 3; ++a)
    if (f.hi[a] > f.lo[a]) m = max(m, f.tot[(a + 1) % 3] * f.tot[(a + 2) % 3]);
  hipLaunchKernelGGL(rt_incoming_kernel, dim3((m + 255) / 256, 3 * nrays), dim3(256), 0, st, I, S,
                     S_y, f, ray_stride, part);
  return hipGetLastError();
}

hipError_t launch_rt_parts_reduce(hipStream_t st, unsigned *part, unsigned *slot,
                                  bool clear_only) {
  hipLaunchKernelGGL(rt_parts_reduce_kernel, dim3(1), dim3(64), 0, st, part, slot,
                     clear_only ? 1 : 0);
  return hipGetLastError();
}

hipError_t launch_rt_qrad(hipStream_t st, const double *I, const double *kap, const double *S,
                          double *q, const int lo[3], const int n[3], int It, int Jt,
                          long ray_stride, int nrays, unsigned tr_mask, const RtRays &w) {
  const int ti = (n[0] + 31) / 32, tj = (n[1] + 31) / 32;
  hipLaunchKernelGGL(rt_qrad_kernel, dim3(ti * tj, n[2]), dim3(256), 0, st, I, kap, S, q, lo[0],
                     lo[1], lo[2], n[0], n[1], It, Jt, ray_stride, nrays, ti, tr_mask, w);
  return hipGetLastError();
}

}  // namespace misohip

namespace misohip {

// T = (gm-1) ei, kappa = kappa0 ro T^3, S = s_rad T^4 on every cell
__global__ __launch_bounds__(256) void rt_source_kernel(const double *__restrict__ ro,
                                                        const double *__restrict__ ei,
                                                        double *__restrict__ kap,
                                                        double *__restrict__ S, long n, double gm,
                                                        double kappa0, double s_rad) {
  const long c = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= n) return;
  const double T = (gm - 1.0) * ei[c];
  const double T2 = T * T;
  kap[c] = kappa0 * ro[c] * (T2 * T);
  S[c] = s_rad * (T2 * T2);
}

// ei += dt * q / ro on the interior
__global__ __launch_bounds__(256) void rt_heat_kernel(const double *__restrict__ ro,
                                                      double *__restrict__ ei,
                                                      const double *__restrict__ q, Shape sh,
                                                      double dt) {
  const int ni = sh.It - 2 * sh.mi, nj = sh.Jt - 2 * sh.mj, nk = sh.Kt - 2 * sh.mk;
  const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= (long)ni * nj * nk) return;
  const int i = sh.mi + (int)(t % ni);
  const long r = t / ni;
  const int j = sh.mj + (int)(r % nj), k = sh.mk + (int)(r / nj);
  const int c = sh.idx(i, j, k);
  ei[c] = ei[c] + dt * q[c] / ro[c];
}

hipError_t launch_rt_source(hipStream_t st, const double *ro, const double *ei, double *kap,
                            double *S, long n, double gm, double kappa0, double s_rad) {
  hipLaunchKernelGGL(rt_source_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, ro, ei,
                     kap, S, n, gm, kappa0, s_rad);
  return hipGetLastError();
}

hipError_t launch_rt_heat(hipStream_t st, const double *ro, double *ei, const double *q,
                          const Shape &sh, double dt) {
  const long n = (long)(sh.It - 2 * sh.mi) * (sh.Jt - 2 * sh.mj) * (sh.Kt - 2 * sh.mk);
  hipLaunchKernelGGL(rt_heat_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, ro, ei,
                     q, sh, dt);
  return hipGetLastError();
}

}  // namespace misohip
