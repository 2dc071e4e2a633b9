// fv2d_march.h -- the fused stage of the hydro step as a register march: one wave owns a strip
// of columns and a run of rows, and carries its whole y stencil in registers.
//
// Lane l of a wave stands for column i0-2+l (60 output columns, lanes 2..61; two halo lanes on
// each side). The wave walks up its rows one at a time; between rows it keeps the primitives
// of rows j and j+1, the left state, flux and viscous terms of the next y face. Values of the
// neighbouring columns come from the neighbouring lanes by DPP wave shifts (VALU moves). There
// is no LDS and no barrier: waves never wait for each other, so a SIMD always has other waves
// to issue from, and every interface is solved once. What a row needs late (the lower face's terms,
// the next row's left states, FP64: row j+2) waits in slots of LDS that only the lane itself uses.
// Bound by VALU issue: KH 4096^2 (PLM, HLLC, conduction, viscosity) FP64 697 VALU instructions per
// cell and stage, 88% busy over the launch, 890 us per step (strip kernel: 742, 75%, 1020); FP32 365,
// always busy, 345 us (389, 96%, 405). Per row j:
//   begin   row j+2 from storage values (loaded one row ahead) to primitives
//   diffs   differences along x, from column l+1            (shift: primitives of row j)
//   slopes  minmod slopes and face states of x (row j) and y (row j+1)   (shift: differences)
//   fluxes  x interface (l, l+1) and y interface (j, j+1), conduction and viscous face terms
//                                                            (shift: left-face states)
//   update  the cell, RK2 average, store, dt term            (shift: x-face fluxes and terms)
// The arithmetic of every value is StripStage's, operation for operation.
//
// The phase functions are plain host/device code on one lane's record; the kernel shifts the
// records' fields by DPP between phases, a host emulation by copies.
#pragma once

#include "fv2d_stage.h"

namespace fv2d {

constexpr int MARCH_OUT = 60;  // output columns per wave

// Waves per SIMD of the kernels: 4 with an FP64 state (84-128 VGPRs in FP64; FP32 on the FP64 state: 9.5
// KB of LDS per wave), FP32 at most 80 VGPRs (6 waves), or 96 (5 waves) where the gravity and wall
// terms come with viscosity or conduction (they spill at 80).
FV2D_HD constexpr int march_wpe(bool state64, bool xg_parabolic) { return state64 ? 4 : (xg_parabolic ? 5 : 6); }

// Work split of one grid: tasks (strip, segment of rows), one wave each. The rows are one band, or 8
// bands of `height` rows, one per XCD. A band's segments are `nlong` ones of `seg` rows from its first
// row on, then short ones of `sseg` rows up to its end; task t of a band is strip t % nsx of segment
// t / nsx. Tasks past a band's rows are empty. With one band all segments are long.
struct MarchGeom {
  int nsx;
  int bands, height;
  int nlong, seg, sseg;
  int per_band;  // tasks per band
  int ntasks;    // bands * per_band
};

FV2D_HD constexpr int march_strips(int Nx) { return (Nx + MARCH_OUT - 1) / MARCH_OUT; }

FV2D_HD MarchGeom march_geom(int Nx, int Ny, int seg) {
  MarchGeom g;
  g.nsx = march_strips(Nx);
  g.bands = 1;
  g.height = Ny;
  g.nlong = (Ny + seg - 1) / seg;
  g.seg = g.sseg = seg;
  g.per_band = g.ntasks = g.nsx * g.nlong;
  return g;
}

FV2D_HD MarchGeom march_geom_banded(int Nx, int Ny, int nlong, int seg, int sseg) {
  MarchGeom g = march_geom(Nx, Ny, seg);
  g.bands = 8;
  g.height = (Ny + 7) / 8;
  g.nlong = nlong;
  g.sseg = sseg;
  const int rest = g.height - nlong * seg;
  g.per_band = g.nsx * (nlong + (rest > 0 ? (rest + sseg - 1) / sseg : 0));
  g.ntasks = 8 * g.per_band;
  return g;
}

// Output columns from i0 and rows [jb, je) of task t of a band (je <= jb: an empty task).
FV2D_HD void march_task_rows(const MarchGeom &g, int Ny, int band, int t, int &i0, int &jb, int &je) {
  const int m = t / g.nsx;
  i0 = (t - m * g.nsx) * MARCH_OUT;
  const int b0 = band * g.height, b1 = (b0 + g.height < Ny) ? b0 + g.height : Ny;
  const bool lng = m < g.nlong;
  jb = b0 + (lng ? m * g.seg : g.nlong * g.seg + (m - g.nlong) * g.sseg);
  je = jb + (lng ? g.seg : g.sseg);
  je = je < b1 ? je : b1;
}

// A lane's own slots in LDS (device) or host memory; slot k of the lane is at [64 * k].
#if defined(__HIP_DEVICE_COMPILE__)
template <typename R>
using LanePtr = __attribute__((address_space(3))) R *;
#else
template <typename R>
using LanePtr = R *;
#endif

// One lane's record.
template <typename R, typename S>
struct MarchLane {
  // carried from row to row
  R q0[4], q1[4];    // primitives of rows j, j+1
  R t0, t1;          // p / rho of rows j, j+1
  R um, vm;          // velocities of row j-1
  LanePtr<R> low;    // the lane's slots (stride 64) of the y face (j-1, j): flux, viscous terms,
                     // conduction flux, interface pressure
  LanePtr<S> ring;   // the lane's slots of U of rows j .. j+2 (kRing)
  S raw[4];          // storage values of row j+2
  // within a row
  R q2[4], t2;       // primitives of row j+2
  R q0r[4], t0r;     // row j, lane l+1
  R u1l, v1l, u1r, v1r, u0l, v0l;  // velocities of rows j+1, j at lanes l-1, l+1
  R d[4], dl[4];     // row j: q(l+1) - q(l), and that of lane l-1
  R eu, ev, eur, evr;  // u, v: row j+1 minus row j-1, and that of lane l+1
  R aX[4], bX[4], bXr[4];  // row j's face states at its right / left face; the latter of lane l+1
  R bY[4], aLn[4];   // row j+1's face states at its lower / upper face
  R fx[4], fxl[4];   // flux of the x face (l, l+1), and that of lane l-1
  R fy[4], py;       // flux and interface pressure of the y face (j, j+1)
  R tcx, tcxl;       // conduction flux of the x faces
  R vx[3], vxl[3];   // viscous terms of the x faces
  R vy[3];           // viscous terms of the y face (j, j+1)
  R fc;              // conduction flux of the y face (j, j+1)
  // the wave's column
  int si;            // source column of this lane (ghosts mapped)
  bool flip;         // u changes sign there
  double inv;
};

template <typename R, typename S, int RECON, int RIEM, bool TC, bool VISC, bool XG, int DIVF_ = DIVF_RUNTIME>
struct MarchStage : StageOps<R, S, TC, DIVF_> {
  typedef StageOps<R, S, TC, DIVF_> Ops_;
  using typename Ops_::A;
  using Ops_::add_flux;
  using Ops_::add_gravity;
  using Ops_::exact_dxdy;
  typedef MarchLane<R, S> Lane;
  static constexpr bool kTC = TC, kVISC = VISC, kPLM = RECON == PLM;
  static constexpr bool kParkQ2 = sizeof(R) == 8;
  // U of a row is kept from its load to its update, two rows later (the FP32 forms, where the slots
  // fit): the rows in flight outgrow an XCD's 4 MB L2, so reading it again was a third of the HBM reads
  // at 4096^2 (FP32 733 -> 491 MB per stage).
  static constexpr bool kRing = sizeof(R) == 4;
  static constexpr int NRING = kRing ? 12 : 0;
  static constexpr int kWPE = march_wpe(sizeof(S) == 8, XG && (TC || VISC));

  // Slots of Lane::low.
  static constexpr int LFY = 0, LVY = 4, LFC = LVY + (VISC ? 3 : 0), LPY = LFC + (TC ? 1 : 0);
  static constexpr int LAL = LPY + (XG ? 1 : 0), LQ2 = LAL + 4;
  static constexpr int NLOW = LQ2 + (kParkQ2 ? 5 : 0);

  // The lane's column i0-2+lane, ghosts mapped to their source.
  static FV2D_HD void set_column(int lane, int i0, const KParams &kp, Lane &r) {
    const int gi = i0 - 2 + lane;
    r.flip = false;
    r.si = (gi >= 0 && gi < kp.Nx) ? gi : map_ghost(gi, kp.Nx, kp.bcx, r.flip);
    r.inv = 0.0;
  }

  // Storage values of row gj (wave-uniform; ghosts mapped).
  static FV2D_HD void fetch_row(int gj, const KParams &kp, const StageIO<S> &io, const Lane &r, S raw[4]) {
    bool fy;
    const int sj = (gj >= 0 && gj < kp.Ny) ? gj : map_ghost(gj, kp.Ny, kp.bcy, fy);
    const S *row = ((io.qsrc == QSRC_Q0) ? io.q0 : io.src) + (long long)sj * kp.pitch;
#pragma unroll
    for (int v = 0; v < 4; ++v) raw[v] = URow<S>(row + (long long)v * kp.plane)[r.si];
  }

  // Primitives (and T) of row gj from its storage values.
  static FV2D_HD void row_prim(int gj, const S raw[4], const KParams &kp, const StageIO<S> &io, const Lane &r,
                               R q[4], R &t) {
    bool fy = false;
    if (gj < 0 || gj >= kp.Ny) map_ghost(gj, kp.Ny, kp.bcy, fy);
    St<R> s;
    t = R(0);
    Ops_::raw_to_q(raw, r.flip, fy, kp, io, s, t);
#pragma unroll
    for (int v = 0; v < 4; ++v) q[v] = s.v[v];
  }

  // Lanes whose cell this wave updates.
  static FV2D_HD bool owns(int lane, int i0, const KParams &kp) {
    return lane >= 2 && lane < 2 + MARCH_OUT && i0 - 2 + lane < kp.Nx;
  }
  static FV2D_HD void ring_put(int j, const S raw[4], Lane &r) {
    if (!kRing) return;
    const LanePtr<S> p = r.ring + 64 * 4 * int((unsigned)j % 3u);
#pragma unroll
    for (int v = 0; v < 4; ++v) p[64 * v] = raw[v];
  }
  // Own-cell U of row j (the other lanes read a column inside the grid and drop it).
  static FV2D_HD void load_own(int j, const KParams &kp, const StageIO<S> &io, const Lane &r, S u[4]) {
    if (kRing && io.qsrc != QSRC_Q0) {
      const LanePtr<S> p = r.ring + 64 * 4 * int((unsigned)j % 3u);
#pragma unroll
      for (int v = 0; v < 4; ++v) u[v] = p[64 * v];
      return;
    }
    const long long k = (long long)j * kp.pitch;
#pragma unroll
    for (int v = 0; v < 4; ++v) u[v] = URow<S>(io.src + (k + (long long)v * kp.plane))[r.si];
  }

  // Face values q +- slope / 2: one rounding of slope * 0.5 shared by both sides (FP64), one FMA
  // each (FP32); the same bits as q + slope * (+-1) * 0.5.
  static FV2D_HD R hi_face(R q, R s) { return q + s * R(0.5); }
  static FV2D_HD R lo_face(R q, R s) { return q - s * R(0.5); }

  static FV2D_HD void y_riemann(const R a[4], const R b[4], const KParams &kp, R f[4], R &pout) {
    St<R> l, h, fs;
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      l.v[v] = a[v];
      h.v[v] = b[v];
    }
    riemann<RIEM>(swap_uv(l), swap_uv(h), R(kp.gamma0), R(kp.gm1), R(kp.entho), kp.divg, R(kp.fslp_K), R(kp.gdx_y), fs, pout);
    fs = swap_uv(fs);
#pragma unroll
    for (int v = 0; v < 4; ++v) f[v] = fs.v[v];
  }

  // Viscous terms of a y face between a lower row a and an upper row b (Viscosity.h:87-106):
  // own column u/v and those of lanes l-1 (m), l+1 (p).
  static FV2D_HD void visc_y(R ua, R va, R uam, R vam, R uap, R vap, R ub, R vb, R ubm, R vbm, R ubp, R vbp,
                             const KParams &kp, R vy[3]) {
    const R mu = R(kp.mu), ody = R(kp.inv_dy);
    const R qiu = (ub + ua) * R(0.5);
    const R qiv = (vb + va) * R(0.5);
    const R dudy = ody * (ub - ua);
    const R dvdy = ody * (vb - va);
    const R dudx = R(kp.qdx) * (ubp - ubm + uap - uam);
    const R dvdx = R(kp.qdx) * (vbp - vbm + vap - vam);
    const R tau_yy = R(4.0 / 3.0) * dvdy - R(2.0 / 3.0) * dudx;
    const R tau_xy = dvdx + dudy;
    vy[0] = mu * tau_xy;
    vy[1] = mu * tau_yy;
    vy[2] = mu * (tau_xy * qiu + tau_yy * qiv);
  }

  // ---------------------------------------------------------------- segment prologue
  // From the raw rows jb-2 .. jb+1: the carried state at j = jb. The viscous terms of the
  // bottom face need the neighbours' velocities of rows jb-1 (u0l ..) and jb (u1l ..): the
  // first function leaves row jb-1's velocities in um, vm; the caller shifts.
  static FV2D_HD void pro_rows(int jb, const S raw[4][4], const KParams &kp, const StageIO<S> &io, Lane &r) {
    R qa[4], qb[4], ta, tb;
    row_prim(jb - 2, raw[0], kp, io, r, qa, ta);
    row_prim(jb - 1, raw[1], kp, io, r, qb, tb);
    row_prim(jb, raw[2], kp, io, r, r.q0, r.t0);
    row_prim(jb + 1, raw[3], kp, io, r, r.q1, r.t1);
    ring_put(jb, raw[2], r);
    ring_put(jb + 1, raw[3], r);
    R lo[4], hi[4];
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      if (kPLM) {
        const R d0 = r.q0[v] - qb[v];
        const R s = minmod(d0, r.q1[v] - r.q0[v]);
        lo[v] = hi_face(qb[v], minmod(qb[v] - qa[v], d0));
        hi[v] = lo_face(r.q0[v], s);
        r.low[64 * (LAL + v)] = hi_face(r.q0[v], s);
      } else {
        lo[v] = qb[v];
        hi[v] = r.q0[v];
        r.low[64 * (LAL + v)] = r.q0[v];
      }
    }
    y_riemann(lo, hi, kp, r.fy, r.py);
    r.um = qb[IU];
    r.vm = qb[IV];
    if (TC) {
      const R kf = R(kp.kf);
      r.fc = Ops<R>::div_c(kf * (r.t0 - tb), R(kp.dy), R(kp.inv_dy), divy(kp));
    }
  }
  // Bottom-face viscous terms (u0l.. = row jb-1 at the neighbours, u1l.. = row jb).
  static FV2D_HD void pro_visc(R uap, R vap, const KParams &kp, Lane &r) {
    visc_y(r.um, r.vm, r.u0l, r.v0l, uap, vap, r.q0[IU], r.q0[IV], r.u1l, r.v1l, r.u1r, r.v1r, kp, r.vy);
  }

  // ---------------------------------------------------------------- row phases
  static FV2D_HD int divx(const KParams &kp) { return exact_dxdy(kp) ? int(DIV_EXACT) : kp.divx; }
  static FV2D_HD int divy(const KParams &kp) { return exact_dxdy(kp) ? int(DIV_EXACT) : kp.divy; }

  // Row j+2's primitives. Then the caller shifts q0, t0 (q0r, t0r) and, with viscosity, the
  // velocities of rows j and j+1 (u0l, u1l, u1r, ...).
  static FV2D_HD void row_begin(int j, const KParams &kp, const StageIO<S> &io, Lane &r) {
    row_prim(j + 2, r.raw, kp, io, r, r.q2, r.t2);
    ring_put(j + 2, r.raw, r);
  }
  // Differences along x; then the caller shifts d (dl) and eu, ev (eur, evr).
  static FV2D_HD void row_diffs(Lane &r) {
#pragma unroll
    for (int v = 0; v < 4; ++v) r.d[v] = r.q0r[v] - r.q0[v];
    if (VISC) {
      r.eu = r.q1[IU] - r.um;
      r.ev = r.q1[IV] - r.vm;
    }
  }
  // Face states of x (row j) and y (row j+1); then the caller shifts bX (bXr).
  static FV2D_HD void row_slopes(Lane &r) {
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      if (kPLM) {
        const R sx = minmod(r.dl[v], r.d[v]);
        r.aX[v] = hi_face(r.q0[v], sx);
        r.bX[v] = lo_face(r.q0[v], sx);
        const R sy = minmod(r.q1[v] - r.q0[v], r.q2[v] - r.q1[v]);
        r.bY[v] = lo_face(r.q1[v], sy);
        r.aLn[v] = hi_face(r.q1[v], sy);
      } else {
        r.aX[v] = r.bX[v] = r.q0[v];
        r.bY[v] = r.aLn[v] = r.q1[v];
      }
    }
  }
  // Row j+2 is not used again before it becomes row j+1.
  static FV2D_HD void park(Lane &r) {
    if (!kParkQ2) return;
#pragma unroll
    for (int v = 0; v < 4; ++v) r.low[64 * (LQ2 + v)] = r.q2[v];
    if (TC) r.low[64 * (LQ2 + 4)] = r.t2;
  }
  // Fluxes and face terms; then the caller shifts fx, tcx, vx (fxl, tcxl, vxl).
  static FV2D_HD void row_fluxes(const KParams &kp, Lane &r) {
    St<R> a, b, f;
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      a.v[v] = r.aX[v];
      b.v[v] = r.bXr[v];
    }
    R px;
    riemann<RIEM>(a, b, R(kp.gamma0), R(kp.gm1), R(kp.entho), kp.divg, R(kp.fslp_K), R(kp.gdx_x), f, px);
#pragma unroll
    for (int v = 0; v < 4; ++v) r.fx[v] = f.v[v];
    R aL[4];
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      aL[v] = r.low[64 * (LAL + v)];
      r.low[64 * (LAL + v)] = r.aLn[v];
    }
    y_riemann(aL, r.bY, kp, r.fy, r.py);
    if (TC) {
      const R kf = R(kp.kf);
      r.tcx = Ops<R>::div_c(kf * (r.t0r - r.t0), R(kp.dx), R(kp.inv_dx), divx(kp));
      r.fc = Ops<R>::div_c(kf * (r.t1 - r.t0), R(kp.dy), R(kp.inv_dy), divy(kp));
    }
    if (VISC) {
      const R mu = R(kp.mu), odx = R(kp.inv_dx);
      const R ub = r.q0r[IU], ua = r.q0[IU], vb = r.q0r[IV], va = r.q0[IV];
      const R qiu = (ub + ua) * R(0.5);
      const R qiv = (vb + va) * R(0.5);
      const R dudx = odx * r.d[IU];
      const R dvdx = odx * r.d[IV];
      const R dudy = R(kp.qdy) * (r.eur + r.q1[IU] - r.um);
      const R dvdy = R(kp.qdy) * (r.evr + r.q1[IV] - r.vm);
      const R tau_xx = R(4.0 / 3.0) * dudx - R(2.0 / 3.0) * dvdy;
      const R tau_xy = dvdx + dudy;
      r.vx[0] = mu * tau_xx;
      r.vx[1] = mu * tau_xy;
      r.vx[2] = mu * (tau_xx * qiu + tau_xy * qiv);
      visc_y(ua, va, r.u0l, r.v0l, ub, vb, r.q1[IU], r.q1[IV], r.u1l, r.v1l, r.u1r, r.v1r, kp, r.vy);
    }
  }
  // Reset counters (rare).
  static FV2D_HD void count_resets(StepCtl *ctl, unsigned nr, unsigned np, unsigned nn) {
#if defined(__HIP_DEVICE_COMPILE__)
    if (nr) atomicAdd(&ctl->neg_rho, (unsigned long long)nr);
    if (np) atomicAdd(&ctl->neg_prs, (unsigned long long)np);
    if (nn) atomicAdd(&ctl->nan_cnt, (unsigned long long)nn);
#else
    ctl->neg_rho += nr;
    ctl->neg_prs += np;
    ctl->nan_cnt += nn;
#endif
  }
  // The cell of row j.
  static FV2D_HD void row_update(int lane, int j, int i0, const KParams &kp, const StageIO<S> &io, double dt,
                                 double dt_dx, double dt_dy, const S u[4], Lane &r) {
    if (!owns(lane, i0, kp)) return;
    S u0[4];
    if (io.avg) {
      const long long k = (long long)j * kp.pitch;
#pragma unroll
      for (int v = 0; v < 4; ++v) u0[v] = URow<S>(io.avg + (k + (long long)v * kp.plane))[r.si];
    }
    const int dvx = divx(kp), dvy = divy(kp);
    const R rho = r.q0[IR];
    A acc[4];
#pragma unroll
    for (int v = 0; v < 4; ++v) acc[v] = (sizeof(R) == 8) ? A(u[v]) : A(0);

    double gX = 0.0, gY = 0.0;
    if (XG) {
      if (kp.grav == GRAV_CONSTANT) {
        gX = kp.gxf;
        gY = kp.gyf;
      } else if (kp.grav == GRAV_ANALYTICAL) {
        gX = gY = (double)io.grav_row[j];
      }
    }

    // x sweep (Update.h:171)
    add_flux(acc, r.fxl, r.fx, dt, dt_dx, kp.dx, kp.inv_dx, dvx);
    if (XG && kp.grav != GRAV_NONE) add_gravity(acc, rho, r.fxl[IR], r.fx[IR], dt, gX);

    // y sweep (Update.h:172)
    {
      R FL[4], FR[4];
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        FL[v] = r.low[64 * (LFY + v)];
        FR[v] = r.fy[v];
      }
      // well-balanced wall flux (Update.h:149-156), with the pout of the other face
      if (XG && kp.wb && (j == 0 || j == kp.Ny - 1)) {
        const R g = R(gY);
        if (j == 0) {
          FL[0] = R(0);
          FL[1] = R(0);
          FL[2] = r.py - rho * g * R(kp.dy);
          FL[3] = R(0);
        } else {
          FR[0] = R(0);
          FR[1] = R(0);
          FR[2] = r.low[64 * LPY] + rho * g * R(kp.dy);
          FR[3] = R(0);
        }
      }
      add_flux(acc, FL, FR, dt, dt_dy, kp.dy, kp.inv_dy, dvy);
      if (XG && kp.grav != GRAV_NONE) add_gravity(acc, rho, FL[IR], FR[IR], dt, gY);
    }

    // thermal conduction into E (ThermalConduction.h:42-106)
    if (TC) {
      R FL = r.tcxl;
      R FR = r.tcx;
      // wall modes replace the x fluxes on the first / last row (ThermalConduction.h:75-103)
      if (XG) {
        const R kf = R(kp.kf);
        const R dy = R(kp.dy);
        if (j == 0 && kp.bctc_ymin != BCTC_NONE) {
          if (kp.bctc_ymin == BCTC_FIXED_TEMPERATURE)
            FL = Ops<R>::div_c(kf * R(2) * (r.t0 - R(kp.bctc_ymin_value)), dy, R(kp.inv_dy), dvy);
          else if (kp.bctc_ymin == BCTC_FIXED_GRADIENT)
            FL = kf * R(kp.bctc_ymin_value);
        }
        if (j == kp.Ny - 1 && kp.bctc_ymax != BCTC_NONE) {
          if (kp.bctc_ymax == BCTC_FIXED_TEMPERATURE)
            FR = Ops<R>::div_c(kf * R(2) * (R(kp.bctc_ymax_value) - r.t0), dy, R(kp.inv_dy), dvy);
          else if (kp.bctc_ymax == BCTC_FIXED_GRADIENT)
            FR = kf * R(kp.bctc_ymax_value);
        }
      }
      acc[IE] = acc[IE] + (A(dt_dx) * A(FR - FL) + A(dt_dy) * A(r.fc - r.low[64 * LFC]));
    }

    // viscosity (Viscosity.h:33-117). The reference accumulates 0 + (-low) + high per direction,
    // which is high - low but for the sign of a zero.
    if (VISC) {
      R f[3];
#pragma unroll
      for (int k = 0; k < 3; ++k) f[k] = (r.vx[k] - r.vxl[k]) + (r.vy[k] - r.low[64 * (LVY + k)]);
      if (sizeof(R) == 8) acc[IR] = acc[IR] + A(0) * A(dt);
      acc[IU] = acc[IU] + A(f[0]) * A(dt);
      acc[IV] = acc[IV] + A(f[1]) * A(dt);
      acc[IE] = acc[IE] + A(f[2]) * A(dt);
    }
    unsigned nr = 0, np = 0, nn = 0;
    Ops_::finish_cell(i0 - 2 + lane, j, acc, u, u0, kp, io, dvx, dvy, nr, np, nn, r.inv);
    if (nr | np | nn) count_resets(io.ctl, nr, np, nn);
  }
  // The y face (j, j+1) becomes the lower one.
  static FV2D_HD void put_low(Lane &r) {
#pragma unroll
    for (int v = 0; v < 4; ++v) r.low[64 * (LFY + v)] = r.fy[v];
    if (VISC) {
#pragma unroll
      for (int k = 0; k < 3; ++k) r.low[64 * (LVY + k)] = r.vy[k];
    }
    if (TC) r.low[64 * LFC] = r.fc;
    if (XG) r.low[64 * LPY] = r.py;
  }
  // Row j+1 becomes the current row.
  static FV2D_HD void row_next(Lane &r) {
    r.um = r.q0[IU];
    r.vm = r.q0[IV];
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      r.q0[v] = r.q1[v];
      r.q1[v] = kParkQ2 ? r.low[64 * (LQ2 + v)] : r.q2[v];
    }
    r.t0 = r.t1;
    r.t1 = kParkQ2 && TC ? r.low[64 * (LQ2 + 4)] : r.t2;
    put_low(r);
  }
};

}  // namespace fv2d
