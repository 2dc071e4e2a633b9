// fv2d_march_device.h -- HIP kernel of the register-march stage (fv2d_march.h) and its launch.
#pragma once

#include "fv2d_device.h"
#include "fv2d_march.h"

namespace fv2d {

constexpr int MARCH_WAVES = 4;  // waves per workgroup (independent of each other)

// Lane l receives lane l-1's (shr) or l+1's (shl) value by DPP wave shifts; the lane without a
// neighbour gets 0.
__device__ inline int dpp_shr(int x) { return __builtin_amdgcn_update_dpp(0, x, 0x138, 0xf, 0xf, true); }
__device__ inline int dpp_shl(int x) { return __builtin_amdgcn_update_dpp(0, x, 0x130, 0xf, 0xf, true); }
__device__ inline double shr1(double x) { return __hiloint2double(dpp_shr(__double2hiint(x)), dpp_shr(__double2loint(x))); }
__device__ inline double shl1(double x) { return __hiloint2double(dpp_shl(__double2hiint(x)), dpp_shl(__double2loint(x))); }
__device__ inline float shr1(float x) { return __int_as_float(dpp_shr(__float_as_int(x))); }
__device__ inline float shl1(float x) { return __int_as_float(dpp_shl(__float_as_int(x))); }
// shl1 that leaves lane 63 its own value (in place when x dies here): a face state between real
// states keeps that lane off the division and square-root fallbacks, which the whole wave would
// run with it (Sedov 2048^2 FP64: 245 us per step with a zero state there, 230 without).
__device__ inline double shl1_keep(double x) {
  const int lo = __double2loint(x), hi = __double2hiint(x);
  return __hiloint2double(__builtin_amdgcn_update_dpp(hi, hi, 0x130, 0xf, 0xf, false),
                          __builtin_amdgcn_update_dpp(lo, lo, 0x130, 0xf, 0xf, false));
}
__device__ inline float shl1_keep(float x) {
  const int i = __float_as_int(x);
  return __int_as_float(__builtin_amdgcn_update_dpp(i, i, 0x130, 0xf, 0xf, false));
}

// Slots parked in LDS must stay there: without this the compiler forwards every stored value to
// its read of the next row in registers, which it then spills to scratch (KH FP64: 20 registers
// spilled, 1019 us per step at 4096^2; none, 927).
template <typename R>
__device__ inline LanePtr<R> opaque(LanePtr<R> p) {
#if defined(__HIP_DEVICE_COMPILE__)
  unsigned a = (unsigned)(size_t)p;
  asm volatile("" : "+v"(a));
  return (LanePtr<R>)a;
#else
  return p;
#endif
}

// Rows [jb, je) of the strip starting at output column i0, by one wave.
template <class K, typename R, typename S>
__device__ inline void march_rows(const KParams &kp, const StageIO<S> &io, int i0, int jb, int je, double dt,
                                  double dt_dx, double dt_dy, typename K::Lane &r) {
  const int lane = threadIdx.x & 63;
  K::set_column(lane, i0, kp, r);
  {
    S raw[4][4];
#pragma unroll
    for (int k = 0; k < 4; ++k) K::fetch_row(jb - 2 + k, kp, io, r, raw[k]);
    K::fetch_row(jb + 2, kp, io, r, r.raw);
    K::pro_rows(jb, raw, kp, io, r);
    if (K::kVISC) {
      r.u0l = shr1(r.um);
      r.v0l = shr1(r.vm);
      r.u1l = shr1(r.q0[IU]);
      r.v1l = shr1(r.q0[IV]);
      r.u1r = shl1(r.q0[IU]);
      r.v1r = shl1(r.q0[IV]);
      K::pro_visc(shl1(r.um), shl1(r.vm), kp, r);
    }
    K::put_low(r);
  }
  for (int j = jb; j < je; ++j) {
    r.low = opaque<R>(r.low);
    if (K::kRing) r.ring = opaque<S>(r.ring);
    K::row_begin(j, kp, io, r);
#pragma unroll
    for (int v = 0; v < 4; ++v) r.q0r[v] = shl1(r.q0[v]);
    if (K::kTC) r.t0r = shl1(r.t0);
    K::row_diffs(r);
    if (K::kPLM) {
#pragma unroll
      for (int v = 0; v < 4; ++v) r.dl[v] = shr1(r.d[v]);
    }
    if (K::kVISC) {
      r.eur = shl1(r.eu);
      r.evr = shl1(r.ev);
      r.u0l = shr1(r.q0[IU]);
      r.v0l = shr1(r.q0[IV]);
      r.u1l = shr1(r.q1[IU]);
      r.v1l = shr1(r.q1[IV]);
      r.u1r = shl1(r.q1[IU]);
      r.v1r = shl1(r.q1[IV]);
    }
    K::row_slopes(r);
    K::park(r);
#pragma unroll
    for (int v = 0; v < 4; ++v) r.bXr[v] = shl1_keep(r.bX[v]);
    K::row_fluxes(kp, r);
    S u[4];
    K::load_own(j, kp, io, r, u);
    K::fetch_row(j + 3, kp, io, r, r.raw);
#pragma unroll
    for (int v = 0; v < 4; ++v) r.fxl[v] = shr1(r.fx[v]);
    if (K::kTC) r.tcxl = shr1(r.tcx);
    if (K::kVISC) {
#pragma unroll
      for (int k = 0; k < 3; ++k) r.vxl[k] = shr1(r.vx[k]);
    }
    K::row_update(lane, j, i0, kp, io, dt, dt_dx, dt_dy, u, r);
    K::row_next(r);
  }
}

// One wave's task of a stage: rows [jb, je) of the strip at i0; `slot` picks its dt slot.
template <class K, typename R, typename S>
__device__ inline void march_task(const KParams &kp, const StageIO<S> &io, int i0, int jb, int je, int slot, double dt,
                                  double dt_dx, double dt_dy) {
  __shared__ R low[MARCH_WAVES][K::NLOW * 64];
  typename K::Lane r;
  r.low = (LanePtr<R>)(low[threadIdx.x >> 6] + (threadIdx.x & 63));
  if constexpr (K::kRing) {
    __shared__ S ring[MARCH_WAVES][K::NRING * 64];
    r.ring = (LanePtr<S>)(ring[threadIdx.x >> 6] + (threadIdx.x & 63));
  }
  march_rows<K, R, S>(kp, io, i0, jb, je, dt, dt_dx, dt_dy, r);
  if (io.epilogue) {
    const double m = wave_max(r.inv);
    if ((threadIdx.x & 63) == 0) acc_max(io.acc, slot, m);
  }
}

// How a stage of a single simulation gets its dt. The first stage of a step runs the loop control
// itself: each of its waves takes the maximum over the slots of the previous state and forms the
// same dt, and the wave of task 0 records it for the second stage and the next step, which read it
// after the launch boundary. A launch of its own for this took 4.2 us of every step. Control blocks
// alternate, the slots go round three sets: read by the step, filled by it, cleared for the next.
enum : int { MARCH_READ = 0, MARCH_ADVANCE = 1, MARCH_GIVEN = 2 };
struct MarchCtl {
  int mode;           // MARCH_READ: the step's dt is in `out`; else begin the step
  const StepCtl *in;  // control block of the previous step (MARCH_ADVANCE)
  StepCtl *out;       // of this step
  const unsigned long long *acc_in;  // slots of the state the step starts from (MARCH_ADVANCE)
  unsigned long long *acc_clear;     // slots the next step will fill
  double *dts_log;
  double dt;  // MARCH_GIVEN
};

// The step's dt, dt/dx, dt/dy; false when the loop has ended. acc: the slots this step fills.
__device__ inline bool march_begin(const MarchCtl &m, const KParams &kp, unsigned long long *acc, int task, double &dt,
                                   double &dt_dx, double &dt_dy) {
  if (m.mode == MARCH_READ) {
    dt = uni(m.out->dt);
    dt_dx = uni(m.out->dt_dx);
    dt_dy = uni(m.out->dt_dy);
    return uni(m.out->active) != 0;
  }
  StepCtl c;
  if (m.mode == MARCH_ADVANCE) {
    c = *m.in;
    if (c.active) advance_control(&c, acc_read(m.acc_in), kp, task == 0 && (threadIdx.x & 63) == 0 ? m.dts_log : nullptr);
  } else {
    c.dt = m.dt;
    c.dt_dx = m.dt / kp.dx;
    c.dt_dy = m.dt / kp.dy;
    c.t = c.tend = 0.0;
    c.active = 1;
    c.nsteps = c.max_steps = 0;
  }
  if (task == 0) {
    if ((threadIdx.x & 63) == 0) {
      StepCtl *o = m.out;  // (the reset counters and the reduced maximum are not part of the step)
      o->dt = c.dt;
      o->dt_dx = c.dt_dx;
      o->dt_dy = c.dt_dy;
      o->t = c.t;
      o->tend = c.tend;
      o->active = c.active;
      o->nsteps = c.nsteps;
      o->max_steps = c.max_steps;
    }
    acc_clear(m.acc_clear);
    if (!c.active) {  // no step: the state and its maximum stay
      const int s = (threadIdx.x & 63) * ACC_STRIDE;
      acc[s] = m.acc_in[s];
    }
  }
  dt = uni(c.dt);
  dt_dx = uni(c.dt_dx);
  dt_dy = uni(c.dt_dy);
  return uni(c.active) != 0;
}

template <class K, typename R, typename S>
__global__ void __launch_bounds__(64 * MARCH_WAVES) __attribute__((amdgpu_waves_per_eu(K::kWPE, K::kWPE)))
march_kernel(const KParams kp, const StageIO<S> io, const MarchGeom g, const MarchCtl mc) {
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  // XCD x (blocks b with b % 8 == x) takes band x or, with one band, a contiguous run of blocks, so
  // that neighbouring strips, which share halo columns, run on one L2
  const int x = blockIdx.x & 7, k = blockIdx.x >> 3;
  const int q = gridDim.x >> 3, rem = gridDim.x & 7;
  const int band = g.bands == 1 ? 0 : x;
  const int t = (k + (g.bands == 1 ? x * q + (x < rem ? x : rem) : 0)) * MARCH_WAVES + w;
  if (t >= g.per_band) return;
  double dt, dt_dx, dt_dy;
  // (the first band's first task records the step)
  if (!march_begin(mc, kp, io.acc, band + t, dt, dt_dx, dt_dy)) return;  // the device loop has ended
  int i0, jb, je;
  march_task_rows(g, kp.Ny, band, t, i0, jb, je);
  if (jb < je) march_task<K, R, S>(kp, io, i0, jb, je, t + 7 * band, dt, dt_dx, dt_dy);
}

// Batched stage: the waves of a persistent grid run the (job, task) pairs of one kernel class, each
// with the job's own parameters, buffers and dt. An item of the class's run of the work list stands
// for up to MARCH_GROUP tasks of a job. The tasks are split into 8 equal runs, one per XCD (block
// id % 8), with one atomic counter each in a cache line of its own: a wave's first task is its
// number in its run, the next ones come from the counter. One counter for the chip, read before
// every task, cost 8 ns per wave and task: 49 us per stage just for the waves of a full grid to
// learn that nothing is left. Waves do not wait for each other. stage as in batch_stage_kernel.
constexpr int MARCH_GROUP = 8;

// Tasks of a march job; rows: the work list's height.
__device__ inline int march_tasks(const BatchJob &J, int rows) {
  const int seg = J.seg > 0 ? J.seg : rows;
  return J.nsx * ((J.kp.Ny + seg - 1) / seg);
}

template <class K, typename R, typename S>
__global__ void __launch_bounds__(64 * MARCH_WAVES) __attribute__((amdgpu_waves_per_eu(K::kWPE, K::kWPE)))
batch_march_kernel(const BatchJob *__restrict__ jobs, const BatchItem *__restrict__ items, const int *range,
                   int *counter, int stage) {
  const int base = range[0], n = range[1] * MARCH_GROUP, rows = range[2];
  const int x = blockIdx.x & 7;
  const int lo = (int)((long long)n * x >> 3), hi = (int)((long long)n * (x + 1) >> 3);
  const int waves = ((int)(gridDim.x + 7 - x) >> 3) * MARCH_WAVES;  // of this XCD
  int it = lo + (int)(blockIdx.x >> 3) * MARCH_WAVES + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  for (bool first = true; it < hi; first = false) {
    if (!first) {
      if (hi - lo <= waves) return;
      int k = 0;
      if ((threadIdx.x & 63) == 0) k = atomicAdd(counter + x * COUNTER_STRIDE, 1);
      it = lo + waves + uni(k);
      if (it >= hi) return;
    }
    const BatchItem wi = items[base + it / MARCH_GROUP];
    const BatchJob &J = jobs[uni(wi.job)];
    const int task = uni(wi.blk) * MARCH_GROUP + it % MARCH_GROUP;
    StepCtl *ctl = J.ctl;
    const int seg = J.seg > 0 ? J.seg : rows;
    const int sy = task / J.nsx, jb = sy * seg;  // uniform segments
    if (jb >= J.kp.Ny || !uni(ctl->active) || (!J.rk2 && stage == 2)) continue;
    const StageIO<S> io = batch_stage_io<S>(J, stage, uni(ctl->fresh), uni(ctl->nsteps));
    march_task<K, R, S>(J.kp, io, (task - sy * J.nsx) * MARCH_OUT, jb, jb + seg < J.kp.Ny ? jb + seg : J.kp.Ny, task,
                        uni(ctl->dt), uni(ctl->dt_dx), uni(ctl->dt_dy));
  }
}

// Launch chain: run-time switches -> template arguments (DIVF fixed by the caller, as for
// launch_stage).
template <typename R, typename S, int DIVF>
struct MarchLaunch {
  const KParams &kp;
  const StageIO<S> &io;
  const MarchGeom &g;
  const MarchCtl &mc;
  hipStream_t st;
  template <int RC, int RM, bool TC, bool VI, bool XG>
  hipError_t operator()() {
    typedef MarchStage<R, S, RC, RM, TC, VI, XG, DIVF> K;
    hipLaunchKernelGGL((march_kernel<K, R, S>), dim3(g.bands * ((g.per_band + MARCH_WAVES - 1) / MARCH_WAVES)),
                       dim3(64 * MARCH_WAVES), 0, st, kp, io, g, mc);
    return hipGetLastError();
  }
};

template <typename R, typename S, int DIVF>
hipError_t launch_march(const StageClass &c, const KParams &kp, const StageIO<S> &io, const MarchGeom &g,
                        const MarchCtl &mc, hipStream_t st) {
  MarchLaunch<R, S, DIVF> f{kp, io, g, mc, st};
  return with_class(c, f);
}

// The batched kernels of a class: launch, and resident workgroups per CU (for the grid size).
template <typename R, typename S>
struct BatchMarchLaunch {
  const BatchJob *jobs;
  const BatchItem *items;
  const int *range;
  int *counter;
  int stage, grid;
  hipStream_t st;
  template <int RC, int RM, bool TC, bool VI, bool XG>
  hipError_t operator()() {
    typedef MarchStage<R, S, RC, RM, TC, VI, XG> K;
    hipLaunchKernelGGL((batch_march_kernel<K, R, S>), dim3(grid), dim3(64 * MARCH_WAVES), 0, st, jobs, items, range,
                       counter, stage);
    return hipGetLastError();
  }
};
template <typename R, typename S>
struct BatchMarchOcc {
  template <int RC, int RM, bool TC, bool VI, bool XG>
  int operator()() {
    typedef MarchStage<R, S, RC, RM, TC, VI, XG> K;
    int n = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, batch_march_kernel<K, R, S>, 64 * MARCH_WAVES, 0) != hipSuccess)
      n = 1;
    return n > 0 ? n : 1;
  }
};

// Defined in march_fp64.hip / march_fp64_exact.hip / march_fp32.hip.
hipError_t launch_march_fp64(const StageClass &c, const KParams &kp, const StageIO<double> &io,
                             const MarchGeom &g, const MarchCtl &mc, hipStream_t st);
hipError_t launch_march_fp64_exact(const StageClass &c, const KParams &kp, const StageIO<double> &io,
                             const MarchGeom &g, const MarchCtl &mc, hipStream_t st);
hipError_t launch_march_fp32s64(const StageClass &c, const KParams &kp, const StageIO<double> &io,
                                const MarchGeom &g, const MarchCtl &mc, hipStream_t st);
hipError_t launch_march_fp32(const StageClass &c, const KParams &kp, const StageIO<float> &io,
                             const MarchGeom &g, const MarchCtl &mc, hipStream_t st);

}  // namespace fv2d
