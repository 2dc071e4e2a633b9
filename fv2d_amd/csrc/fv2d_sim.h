// fv2d_sim.h -- the step sequence and the device-resident time loop of one simulation, on
// device buffers its owner provides: the handle's allocations (fv2d_capi.hip) or the
// no-allocation scratch (fv2d_noalloc.hip). Both entry points run exactly this code.
#pragma once

#include <hip/hip_runtime.h>

#include <string.h>

#include "../../include/fv2d_amd.h"
#include "fv2d_aux.h"
#include "fv2d_device.h"
#include "fv2d_march_device.h"
#include "fv2d_params.h"

namespace fv2d {

// Device buffers and geometry of one simulation.
struct SimDev {
  fv2d_params p;
  KParams kp;
  StripGeom geom;   // strip kernel (explicit chunk_rows)
  MarchGeom march;  // march kernel (ntasks = 0: the strip kernel runs)
  int nparts = 0;  // per-workgroup partial maxima of the dt reduction (= geom.nblocks)
  hipStream_t stream = nullptr;
  void *U = nullptr, *Us = nullptr, *Q0 = nullptr;  // SoA planes, row pitch kp.pitch
  StepCtl *ctl = nullptr;       // march kernel: two blocks (ctl[cur] is current), counters in the first
  StepCtl *host_ctl = nullptr;  // pinned copy the march path reports into (null: read back by a copy)
  int cur = 0;                  // march kernel: current control block
  int set = 0;                  // and the slots (0..2) of the current state's dt maximum
  double *partials = nullptr;
  const float *grav_row = nullptr;  // analytical gravity per row, else null
  bool fresh_q0 = false;            // the next first stage reads Q0 (main.cpp:57-58)
  // optional hook run before and after every stage launch (kernel timing)
  hipError_t (*mark)(void *ctx) = nullptr;
  void *mark_ctx = nullptr;
};

// The stage kernel and work split of the parameters.
inline void sim_set_geom(SimDev &d) {
  d.geom = sim_geom(&d.p);
  d.march = sim_march_geom(&d.p);
  d.nparts = d.geom.nblocks;
}

// The march kernel's three sets of slots share the buffer of the strip kernel's partials.
inline unsigned long long *sim_acc(const SimDev &d, int set = 0) {
  return d.march.ntasks ? (unsigned long long *)d.partials + set * ACC_WORDS : nullptr;
}
inline size_t sim_partials_bytes(const SimDev &d) {
  const size_t n = d.march.ntasks && d.nparts < 3 * ACC_WORDS ? 3 * ACC_WORDS : d.nparts;
  return n * sizeof(double);
}

// Sets the message fv2d_last_error(NULL) returns (fv2d_capi.hip).
void set_global_error(const char *msg);

// The state is stored in FP32 (FV2D_FP32), else in FP64.
inline bool sim_fp32(const SimDev &d) { return d.p.precision == FV2D_FP32; }
// FP32 arithmetic on an FP64 state (FV2D_FP32_STATE64).
inline bool sim_fp32s64(const SimDev &d) { return d.p.precision == FV2D_FP32_STATE64; }

// Max hyperbolic inverse dt of Q0 (from_q0) or of reset(consToPrim(src)) into the partials.
inline hipError_t sim_launch_dt_tiles(SimDev &d, const void *src, int from_q0) {
  const dim3 grid(d.nparts);
  unsigned long long *acc = sim_acc(d, d.set);
  if (sim_fp32(d))
    hipLaunchKernelGGL((dt_cells_kernel<float, float>), grid, dim3(256), 0, d.stream, d.kp, (const float *)src, from_q0,
                       d.partials, d.nparts, acc);
  else if (sim_fp32s64(d))
    hipLaunchKernelGGL((dt_cells_kernel<float, double>), grid, dim3(256), 0, d.stream, d.kp, (const double *)src,
                       from_q0, d.partials, d.nparts, acc);
  else
    hipLaunchKernelGGL((dt_cells_kernel<double, double>), grid, dim3(256), 0, d.stream, d.kp, (const double *)src,
                       from_q0, d.partials, d.nparts, acc);
  return hipGetLastError();
}

// Strip kernel: the dt reduction (and the loop control).
inline hipError_t sim_launch_reduce(SimDev &d, int advance, double *dts_log) {
  hipLaunchKernelGGL(reduce_kernel, dim3(1), dim3(1024), 0, d.stream, d.ctl, d.partials, d.nparts, d.kp, advance,
                     dts_log);
  return hipGetLastError();
}

// The control block, with the current state's inverse dt and the reset counters, on the host: waits
// for the stream.
inline hipError_t sim_report(SimDev &d, StepCtl &c) {
  hipError_t e;
  if (d.march.ntasks) {
    hipLaunchKernelGGL(report_kernel, dim3(1), dim3(64), 0, d.stream, d.ctl, d.ctl + d.cur, sim_acc(d, d.set), d.host_ctl);
    if ((e = hipGetLastError()) != hipSuccess) return e;
    d.cur = 0;
  }
  if (d.march.ntasks && d.host_ctl) {
    if ((e = hipStreamSynchronize(d.stream)) != hipSuccess) return e;
    c = *d.host_ctl;
    return hipSuccess;
  }
  if ((e = hipMemcpyAsync(&c, d.ctl, sizeof c, hipMemcpyDeviceToHost, d.stream)) != hipSuccess) return e;
  return hipStreamSynchronize(d.stream);
}

// The state's inverse dt after an upload (dt of Q0) or a step, for the next dt.
inline hipError_t sim_finish(SimDev &d, StepCtl &c) {
  hipError_t e;
  if (!d.march.ntasks && (e = sim_launch_reduce(d, 0, nullptr)) != hipSuccess) return e;
  return sim_report(d, c);
}

// One stage: out = [avg +] src + dt L(Q(src or Q0)).
inline hipError_t sim_launch_stage(SimDev &d, const void *src, int qsrc, const void *avg, void *out, int epilogue,
                                   const MarchCtl &mc) {
  const int recon = (d.p.reconstruction == FV2D_PLM) ? PLM : PCM;
  const bool tc = d.p.tc_active != 0, visc = d.p.visc_active != 0;
  const StageClass cls = {recon, d.p.riemann_solver, tc, visc, needs_xg(d.kp), 0};
  hipError_t e;
  if (d.mark && (e = d.mark(d.mark_ctx)) != hipSuccess) return e;
  if (sim_fp32(d)) {
    StageIO<float> io;
    io.src = (const float *)src;
    io.q0 = (const float *)d.Q0;
    io.avg = (const float *)avg;
    io.out = (float *)out;
    io.grav_row = d.grav_row;
    io.ctl = d.ctl;
    io.partials = d.partials;
    io.acc = sim_acc(d, d.set);
    io.qsrc = qsrc;
    io.epilogue = epilogue;
    e = d.march.ntasks ? launch_march_fp32(cls, d.kp, io, d.march, mc, d.stream)
                       : launch_stage_fp32(d.kp, io, d.geom, recon, d.p.riemann_solver, tc, visc, d.stream);
  } else {
    StageIO<double> io;
    io.src = (const double *)src;
    io.q0 = (const double *)d.Q0;
    io.avg = (const double *)avg;
    io.out = (double *)out;
    io.grav_row = d.grav_row;
    io.ctl = d.ctl;
    io.partials = d.partials;
    io.acc = sim_acc(d, d.set);
    io.qsrc = qsrc;
    io.epilogue = epilogue;
    if (sim_fp32s64(d))
      e = d.march.ntasks ? launch_march_fp32s64(cls, d.kp, io, d.march, mc, d.stream)
                         : launch_stage_fp32s64(d.kp, io, d.geom, recon, d.p.riemann_solver, tc, visc, d.stream);
    else
      e = d.march.ntasks ? launch_march_fp64(cls, d.kp, io, d.march, mc, d.stream)
                         : launch_stage_fp64(d.kp, io, d.geom, recon, d.p.riemann_solver, tc, visc, d.stream);
  }
  if (e != hipSuccess) return e;
  if (d.mark && (e = d.mark(d.mark_ctx)) != hipSuccess) return e;
  return hipSuccess;
}

// The stages of one step (UpdateFunctor::update, Update.h:193-222) plus the fused
// c2p / reset / dt epilogue. Euler ping-pongs U and Us; RK2 writes U* to Us and the final
// average in place into U. mode: MARCH_ADVANCE (loop control on the device; the strip kernel's
// reduce_kernel has run it) or MARCH_GIVEN (the dt is `dt`; the strip kernel's set_dt_kernel ran).
inline hipError_t sim_enqueue_step(SimDev &d, bool first_from_q0, bool &swapped, int mode, double dt, double *dts_log) {
  const int q1 = first_from_q0 ? QSRC_Q0 : QSRC_U_RESET;
  hipError_t e;
  swapped = false;
  MarchCtl mc;
  memset(&mc, 0, sizeof mc);
  if (d.march.ntasks) {
    mc.mode = mode;
    mc.dt = dt;
    mc.dts_log = dts_log;
    mc.in = d.ctl + d.cur;
    mc.out = d.ctl + (d.cur ^ 1);
    mc.acc_in = sim_acc(d, d.set);
    mc.acc_clear = sim_acc(d, (d.set + 2) % 3);
    d.cur ^= 1;
    d.set = (d.set + 1) % 3;
  }
  if (d.p.time_stepping == FV2D_TS_EULER) {
    if ((e = sim_launch_stage(d, d.U, q1, nullptr, d.Us, 1, mc)) != hipSuccess) return e;
    void *t = d.U;
    d.U = d.Us;
    d.Us = t;
    swapped = true;
  } else {
    if ((e = sim_launch_stage(d, d.U, q1, nullptr, d.Us, 0, mc)) != hipSuccess) return e;
    mc.mode = MARCH_READ;
    if ((e = sim_launch_stage(d, d.Us, QSRC_U, d.U, d.U, 1, mc)) != hipSuccess) return e;
  }
  return hipSuccess;
}

// Steps to queue before the host looks at the control block again: all that are left when only a
// number of steps ends the loop (up to 4096), else as many as the end time will take at the current
// dt, and one more (up to 64): steps past the end are no-ops, but two empty launches each.
inline int sim_chunk(const SimDev &d, int left, double t, double tend, double inv_hyp) {
  int n = 64;
  if (!(tend < FV2D_TEND_NONE)) n = 4096;
  else if (inv_hyp > 0.0) {
    double m = inv_hyp;
    if (m < d.kp.inv_tc) m = d.kp.inv_tc;
    if (m < d.kp.inv_visc) m = d.kp.inv_visc;
    const double est = (tend - t) * m / d.kp.CFL;  // steps to go
    if (est < 62.0) n = est > 0.0 ? (int)est + 2 : 1;
  }
  return (left > 0 && left < n) ? left : n;
}

// The time loop of main.cpp:62-84 without I/O, dt and t on the device: steps are queued in
// chunks (sim_chunk; steps past the end of the loop are no-ops on the device), the control block
// is read back after each chunk. inv_hyp: the current state's inverse dt (0: not known).
// dts_log (device, >= max_steps entries, or null) receives the dt of every step. On return c
// holds the final control block and d.U the state.
inline hipError_t sim_advance(SimDev &d, double t0, double tend, int max_steps, double inv_hyp, double *dts_log,
                              StepCtl &c) {
  hipError_t e;
  hipLaunchKernelGGL(set_loop_kernel, dim3(1), dim3(1), 0, d.stream, d.ctl + d.cur, t0, tend, max_steps);
  if ((e = hipGetLastError()) != hipSuccess) return e;
  double *log = (max_steps > 0) ? dts_log : nullptr;
  int done = 0;
  memset(&c, 0, sizeof c);
  c.t = t0;
  c.inv_hyp = inv_hyp;
  for (;;) {
    const int n = sim_chunk(d, max_steps > 0 ? max_steps - done : 0, c.t, tend, c.inv_hyp);
    void *U_start = d.U;
    int swaps = 0;
    for (int k = 0; k < n; ++k) {
      if (!d.march.ntasks && (e = sim_launch_reduce(d, 1, log)) != hipSuccess) return e;
      bool swapped;
      if ((e = sim_enqueue_step(d, d.fresh_q0 && done + k == 0, swapped, MARCH_ADVANCE, 0.0, log)) != hipSuccess) return e;
      swaps += swapped ? 1 : 0;
    }
    if ((e = sim_report(d, c)) != hipSuccess) return e;
    const int taken = c.nsteps - done;
    if (swaps) {
      // Euler ping-pong: the state is in U_start after an even number of taken steps.
      if (taken % 2 == 0) {
        if (d.U != U_start) {
          d.Us = d.U;
          d.U = U_start;
        }
      } else if (d.U == U_start) {
        void *x = d.U;
        d.U = d.Us;
        d.Us = x;
      }
    }
    if (c.nsteps > 0) d.fresh_q0 = false;
    done = c.nsteps;
    if (!c.active || (max_steps > 0 && done >= max_steps)) break;
  }
  if (d.march.ntasks) return hipSuccess;  // the report covers the last state
  return sim_finish(d, c);  // strip kernel: reduce the last epilogue for the next dt
}

}  // namespace fv2d
