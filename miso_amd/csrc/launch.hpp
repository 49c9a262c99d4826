// Kernel launchers shared between the C ABI (capi.cpp) and the kernel files.
#pragma once

#include <hip/hip_runtime.h>

#include "device_common.hpp"

namespace misohip {

// Scalars of one RK stage (Integrator::update_sc4 arguments and members).
struct RkScalars {
  double dt, ch2, damp, gm, grav;
  int src_kind, grav_axis;
  int pencil_bx, pencil_by;  // pencil shape in blocks of 64 x 4 cells
  int variant;  // 3D kernel: 0 three load phases, 1 one per point, 2 = 1 at 4 waves/SIMD, 3 LDS tile,
                // 4 z-march over 64 x 4 columns, 5 over 64 x 8
  int zchunk;   // planes walked per block by the z-march kernel
  // z-march kernel: axes (bit 0 x, 1 y, 2 z) whose ghost cells it does not
  // read but maps to their periodic source cells, so that no ghost fill
  // needs to run before it on those axes
  int wrap = 0;
  // src_kind 2: src.vx, src.vy, src.vz, src.ei of the stage's argm (fields
  // of the grid's shape, the run's Real)
  const void *src_arr[4];
  GhostImg img;  // x-y runs: ghost cells stored with their sources
};

// Scalars of one AV sweep (ArtificialViscosity members plus dt).
struct AvScalars {
  double dt, ep, fh, gm, cs_fac, ca_fac, vv_fac;
  int chunk;  // cells walked per thread by the y/z sweeps
  // x-y walk and z walk: axes (bit 0 x, 1 y, 2 z) whose ghost cells they
  // map to periodic source cells instead of reading them
  int wrap = 0;
  int xy_waves = 3;  // FP64 x-y walk: waves per SIMD it is compiled for (3 or 2)
  // a launch over part of the grid: the z walk's chunks [part0, part0 +
  // nparts), the x-y walk's planes part0, part0 + 1, ... (nparts of them; a
  // range past the top z ring plane continues at the bottom one); 0: all
  int part0 = 0, nparts = 0;
  GhostImg img;  // x-y runs: ghost cells stored with their sources
  // x sweep, x-y walk: the CFL slot that this step's last sweep reduces into,
  // cleared on the way (none: null)
  unsigned *clear = nullptr;
};

// Boundary description on the device: axis kind (0 mirror, 1 periodic,
// 2 fixed from the `fixed` fields), mirror signs, fixed-value fields.
struct BcDev {
  int periodic[3];
  float sign[3][9];
  const void *fixed[9];
};

// The batched RK stage of runs with x and y axes and no z axis walks y:
// each wave owns RK_YWALK_OUT x outputs over RK_YWALK_ROWS rows, four waves
// per block (batch_rk_ywalk_kernel; the batch's block counts use these).
constexpr int RK_YWALK_OUT = 60;
constexpr int RK_YWALK_ROWS = 16;
// A single x-y run walks y only when that makes at least this many waves, about
// 2000^2: the one-plane kernel reads every cell at all its stencil points, and
// is the faster one while the run's fields come from the last-level cache (FP32
// stage of 1600 x 1500 66 us, the walk 79; FP64 of 1600 x 1590 170 and 174;
// 2400^2 203 and 171, 363 and 348; 4096^2 599 and 446, 1079 and 976).
constexpr int RK_YWALK_MIN_WAVES = 4096;

inline bool rk_walks_y(const Shape &sh, int variant) {
  const int ni = sh.It - 2 * sh.mi, nj = sh.Jt - 2 * sh.mj;
  return sh.is && sh.js && !sh.ks && variant >= 4 && variant <= 6 &&
         (long)((ni + RK_YWALK_OUT - 1) / RK_YWALK_OUT) *
                 ((nj + RK_YWALK_ROWS - 1) / RK_YWALK_ROWS) >= RK_YWALK_MIN_WAVES;
}

// The ghost cells of an x-y run that its passes can store themselves, where
// that costs less than the fills: those of the x faces are a few scattered
// stores of an end lane in every row, which the wave waits for.  They pay up to
// a number of rows, and in FP64 only beside the one-plane RK stage.  A step with
// and without: FP64 of 512 x 4096 766 and 810 us, 61 x 8192 273 and 261, 61 x
// 16384 487 and 434; FP32 of 61 x 16384 233 and 246, of 4 x 16384 285 and 298.
// With the walking stage FP64 of 1000 x 4096 1485 and 1403, 2048^2 1412 and
// 1403, 61 x 32790 1746 and 1443; FP32 of 2048^2 743 and 749, 1000 x 4096 740
// and 739, 4096^2 2563 and 2532, 61 x 32790 721 and 625.
inline GhostImg ghost_img(const Shape &sh, const BcDev &b, int variant, bool f64) {
  GhostImg m;
  const bool walk = rk_walks_y(sh, variant);
  const int rows = f64 ? (walk ? 0 : 6144) : (walk ? 3072 : 20480);
  m.on = sh.is && sh.js && !sh.ks && b.periodic[0] < 2 && b.periodic[1] < 2 &&
         sh.It >= 3 * sh.mi && sh.Jt >= 3 * sh.mj &&  // every image is a ghost cell
         sh.Jt - 2 * sh.mj <= rows;
  for (int a = 0; a < 2; ++a) {
    m.periodic[a] = b.periodic[a];
    for (int f = 0; f < 9; ++f)
      if (b.sign[a][f] < 0.f) m.flip[a] |= 1u << f;
  }
  return m;
}

// one ray of the sweep, everything the plane kernel needs
struct RtRay {
  int start;              // linear index (within the ray's block) of the first plane's (lo_b, lo_c) node
  int da, db, dc;         // linear step of the node along a (signed), b, c
  int ua, ub, uc;         // upwind offsets (linear) along a, b, c (0 if degenerate)
  int nb, nc;             // transverse node counts
  int sb, sc;             // upwind step along b, c in nodes (+1, -1, or 0 if degenerate)
  int nplanes;
  double w00, w10, w01, w11;  // bilinear weights
  double ds;
  double wq;              // quadrature weight
  int id;                 // the ray's slot in the intensity array
  int tr;                 // 1: intensities (and kappa, S) y-fastest, see rt.hip
};

struct RtRays {
  RtRay r[24];
};

// the lattice's ends, the arrays' extents, ray directions and layouts and the
// boundaries for rt_incoming_kernel
struct RtIncoming {
  int lo[3], hi[3], tot[3];
  int periodic[3], kind[6];
  double value[6];
  unsigned pos[3];     // bit r: ray r goes + along the axis
  unsigned moving[3];  // bit r: ray r has a component along it
  unsigned tr;         // bit r: ray r is kept y-fastest
};
constexpr int RT_PARTS = 64;  // change-reduction slots, 32 words apart

hipError_t launch_rt_sweep_plane(hipStream_t, double *, const double *, const double *,
                                 const double *, const double *, const RtRays &, int, int, long,
                                 int, unsigned *);
hipError_t launch_rt_transpose_xy(hipStream_t, const double *, double *, int, int, int);
// The patched sweep: RT_TILE_PLANES planes per launch (4, 6, 8 and 10: 17.4,
// 17.0, 17.0, 17.3 ms for a radiative step of 256^3 and 9.2, 8.6, 8.3, 8.5 ms
// for a cold solve of 211 x 150 x 187; three iterations of that solve in two
// planes a launch 5.8 ms, in eight 3.9), or RT_TILE_PLANES_THIN where a short
// patch holds the c axis of an axis' rays and nothing but columns repeats (three
// iterations in 8 and 16 planes: 300 x 300 x 2 1.90 and 0.97 ms, 384^2 x 6 2.52
// and 1.44, 1024 x 16 x 16 6.0 and 5.1, 1500 x 300 x 7 12.7 and 5.5, 900 x 800 x
// 18 11.3 and 10.7).  Patches have 64 x RT_ROWS nodes (48 rows: 17.0 ms for 16.0
// and 8.2 for 7.6; 36 of three a wave 16.8 and 8.3), or 64 x RT_ROWS_SMALL for
// thin rays and where an axis' launch would have fewer than RT_FEW workgroups,
// so that a thin slab's x and y rays, two patches high, reach the CUs that whole
// patches leave idle (slab solve of 384^2 x 27: 4.44 -> 3.56 ms; 16 rows, three
// patches high, 3.68; at 256^3, where the chip is full either way, the short
// patches' repeated rows make 19.1 ms of 17.0; a limit of 256 sends a 211 x 150 x
// 187 box there: 8.1 ms for 7.6).
// The first patch of an axis starts on the upwind boundary and owns size - 1
// nodes, the others start P nodes before the size - P they own.
constexpr int RT_TILE_PLANES = 8, RT_TILE_PLANES_THIN = 16;
constexpr int RT_ROWS = 32, RT_ROWS_SMALL = 20, RT_FEW = 128;
__host__ __device__ inline int rt_patches(int n, int size, int P) {
  return n < size ? 1 : 1 + (n - (size - 1) + size - P - 1) / (size - P);
}
__host__ __device__ inline int rt_patch_first(int a, int size, int P) {
  return a == 0 ? -1 : size - 1 + (a - 1) * (size - P) - P;
}
// The cones of x rays kept x-fastest (rt_sweep_multi_kernel): RT_MULTI_PLANES
// planes per launch, RT_MULTI_COLS columns of a plane to a workgroup, up to
// RT_MULTI_ROWS rows with the boundary.
constexpr int RT_MULTI_COLS = 32, RT_MULTI_PLANES = 16, RT_MULTI_ROWS = 33;
// How a ray advances where several planes per launch are allowed.  One with a
// degenerate axis, or a plane too large for a patch's 32-bit addresses: plane
// by plane.  One whose neighbouring nodes are neighbours in memory: in patches.
// The others, x rays kept x-fastest: in cones where these hold the c axis; in
// patches where launches count or the fields exceed the caches; plane by plane
// between (three iterations in patches and by planes: 48^3 0.67 and 1.04 ms,
// 64^3 1.39 and 1.42, 80^3 2.38 and 2.11, 96^3 3.6 and 2.97, 128^3 5.9 and 5.9,
// 500 x 30 x 40 4.3 and 8.6, 384^2 x 33 20.4 and 29.0, 211 x 150 x 187 13.5 and
// 19.7; in patches and in cones: 20^3 0.22 and 0.33, 32^3 0.34 and
// 0.47, 100^2 x 15 1.33 and 0.84).
enum RtWay { RT_BY_PLANES, RT_IN_PATCHES, RT_IN_CONES };
inline RtWay rt_way(const RtRay &R) {
  if (R.sb == 0 || R.sc == 0 || R.ua != R.da || (R.nb + 2L) * R.db >= 1L << 29)
    return RT_BY_PLANES;
  if (R.db == 1) return RT_IN_PATCHES;
  const long plane = (long)R.nb * R.nc, nodes = plane * R.nplanes;
  if (nodes < 65536) return RT_IN_PATCHES;
  if (R.nc < RT_MULTI_ROWS) return RT_IN_CONES;
  return plane >= 5000 && nodes <= 1300000 ? RT_BY_PLANES : RT_IN_PATCHES;
}
// the patches of a launch, by groups of `same` rays with the same planes:
// group g has patches start[g] .. start[g + 1] - 1, per_xcd go to each XCD
struct RtPatches {
  int same, groups, per_xcd;
  int start[25];
};
hipError_t launch_rt_sweep_tiles(hipStream_t, double *, const double *, const double *,
                                 const double *, const double *, const RtRays &, int, int, int,
                                 int, long, unsigned *);
hipError_t launch_rt_sweep_multi(hipStream_t, double *, const double *, const double *,
                                 const RtRays &, int, int, long, int, unsigned *);
hipError_t launch_rt_xfast(hipStream_t, const double *, double *, int, int, int, int, unsigned);
hipError_t launch_rt_incoming(hipStream_t, double *, const double *, const double *,
                              const RtIncoming &, long, int, unsigned *);
hipError_t launch_rt_parts_reduce(hipStream_t, unsigned *, unsigned *, bool);
hipError_t launch_rt_qrad(hipStream_t, const double *, const double *, const double *, double *,
                          const int[3], const int[3], int, int, long, int, unsigned,
                          const RtRays &);
hipError_t launch_rt_source(hipStream_t, const double *, const double *, double *, double *, long,
                            double, double, double);
hipError_t launch_rt_heat(hipStream_t, const double *, double *, const double *, const Shape &,
                          double);

// The next step's CFL reduction carried out by the last AV sweep of a step:
// metric, the run's constants and the reduction slot.
template <typename R> struct CflFuse {
  const R *dx, *dy, *dz;
  double gm, cfl;
  unsigned *slot;
  // optional radiative heating applied to each stored cell first (FP64
  // only): ei = ei + heat_dt * heat_q / ro, the operator-split heating
  const double *heat_q = nullptr;
  double heat_dt = 0.0;
};
hipError_t launch_cfl_init(hipStream_t, unsigned *);
// plain streaming kernels (calib.hip): kind 0 copy, 1 read, 2 write
hipError_t launch_stream(hipStream_t, const void *, void *, size_t, int, double *);

// Waves of a walking-sweep block laid along x: all four when the other
// transverse axis has fewer than four cells (2D runs), else one (the four
// waves then take four rows of that axis).
__host__ __device__ inline int walk_waves_x(int n_other) { return n_other < 4 ? 4 : 1; }

// ---------------------------------------------------------------- batches
// One instance of a batched launch: its three field sets (0 = qq, 1 = argm,
// 2 = rslt), frozen AV speed, metric and shape.  Stored in device memory;
// a block finds its instance by a binary search over per-phase block
// offsets.
template <typename R> struct BatchInst {
  Fld<R> st[3];
  R *cc;
  const R *dx, *dy, *dz, *dxi, *dyi, *dzi;
  Shape sh;
  double min_dxyz;
  int chunk;  // cells walked per thread by the y/z sweeps of this instance
};

// Per-instance step scalars, produced on the device from the CFL result.
template <typename R> struct BatchDyn {
  unsigned cfl_bits;  // float bits of the CFL minimum
  int exp_fallback;   // set if damp had to be evaluated on the device
  R dt;
  R dts[4];
  R ch2;
  R damp[4];
  double time;        // simulated time of the instance
  long steps;
};

// exp(-dt_s/tau) exactly as the host library evaluates it, tabulated for
// the quotients the four stages can produce (stage fractions 1/4, 1/2 and 1
// give -1/8, -1/4, -1/2 exactly; 1/3 gives a value within a few ulps of
// -1/6).
template <typename R> struct DampTable {
  R exact[4];      // stages 0, 2, 3 (index by stage; [1] unused)
  R third[33];     // stage 1: quotient bits q0 - 16 .. q0 + 16
  R q0;            // the quotient nearest -1/6
};

__device__ __forceinline__ int batch_find(const int *__restrict__ start, int n, int b) {
  int lo = 0, hi = n - 1;  // start[0] = 0 <= b < start[n]
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (start[mid] <= b) lo = mid; else hi = mid - 1;
  }
  return lo;
}

template <typename R>
hipError_t launch_batch_rk(hipStream_t, const BatchInst<R> *, const BatchDyn<R> *, const int *,
                           int, int, int, int, int, const RkScalars &, int);
template <typename R>
hipError_t launch_batch_ghost(hipStream_t, const BatchInst<R> *, const int *, int, int, int,
                              const BcDev &);
template <typename R>
hipError_t launch_batch_cfl(hipStream_t, const BatchInst<R> *, BatchDyn<R> *, const int *, int,
                            int, double, double);
template <typename R>
hipError_t launch_batch_params(hipStream_t, const BatchInst<R> *, BatchDyn<R> *, int, double,
                               const DampTable<R> &);
template <typename R>
hipError_t launch_batch_av(hipStream_t, int, int, const BatchInst<R> *, const BatchDyn<R> *,
                           const int *, int, int, int, int, const AvScalars &);

template <typename R>
hipError_t launch_rk_stage(hipStream_t, const Fld<const R> &, const Fld<const R> &,
                           const Fld<R> &, const R *, const R *, const R *, const Shape &,
                           const RkScalars &);
template <typename R>
hipError_t launch_av_sweep(hipStream_t, int, const Fld<const R> &, const Fld<R> &, R *, const R *,
                           const R *, const Shape &, const AvScalars &);
template <typename R>
hipError_t launch_av_sweep_y_degen_z(hipStream_t, const Fld<const R> &, const Fld<R> &,
                                     const R *, const R *, const R *, const Shape &,
                                     const AvScalars &);
// the last AV sweep of a step (z walk in 3D, y walk with the degenerate z
// sweep in 2D) also reducing the next step's CFL candidates into cf.slot
template <typename R>
hipError_t launch_av_last_sweep_cfl(hipStream_t, const Fld<const R> &, const Fld<R> &,
                                    const R *, const R *, const R *, const Shape &,
                                    const AvScalars &, const CflFuse<R> &);
template <typename R>
hipError_t launch_av_sweep_xy(hipStream_t, const Fld<const R> &, const Fld<R> &, R *, const R *,
                              const R *, const Shape &, const BcDev &, const AvScalars &);
// the chunks a y (dir 1) or z (dir 2) walk of this shape is cut into
template <typename R>
void av_walk_split(const Shape &sh, int dir, int chunk_req, int *chunk, int *nchunks);
template <typename R>
hipError_t launch_char_vel(hipStream_t, const Fld<const R> &, R *, int, const AvScalars &);
template <typename R>
hipError_t launch_table1d(hipStream_t, const R *, int, R, R, const R *, R *, long);
template <typename R>
hipError_t launch_table2d(hipStream_t, const R *, int, int, R, R, R, R, const R *, const R *, R *,
                          long);
template <typename R>
// axes: bit 0 x, 1 y, 2 z -- the faces to fill (edges of an axis left out
// keep their values)
hipError_t launch_ghost_fill(hipStream_t, const Fld<R> &, const Shape &, const BcDev &,
                             int axes = 7);
template <typename R>
hipError_t launch_cfl(hipStream_t, const Fld<const R> &, const R *, const R *, const R *,
                      const Shape &, double, double, unsigned *);
template <typename R>
hipError_t launch_transpose(hipStream_t, const R *, R *, int, int, int, bool);

}  // namespace misohip
