// march_emu.cpp -- TEST INFRASTRUCTURE: host emulation of the register-march stage.
//
// Runs the phase functions of fv2d_march.h lane by lane, with the kernel's DPP wave shifts as
// copies between lane records, inside the step sequence and C interface of tile_emu.cpp (its
// stage dispatch is replaced by march_stage below). Lane records and slots are filled with
// garbage and NaN before use, so a read of anything not written first shows up in the results;
// the sanitized build checks every index.
#include <array>

#include "tile_emu.h"

#include "../../fv2d_amd/csrc/fv2d_march.h"

namespace emu {

template <class K, typename R, typename S>
void march_run(Sim &s, const StageIO<S> &io) {
  const KParams &kp = s.kp;
  const MarchGeom g = sim_march_geom(&s.p);
  typedef typename K::Lane Lane;
  std::vector<Lane> L(64);
  std::vector<R> low((size_t)K::NLOW * 64);
  std::vector<S> ring((size_t)K::NRING * 64);
  double best = 0.0;
#define EACH(stmt)                                                                                                     \
  for (int lane = 0; lane < 64; ++lane) {                                                                              \
    Lane &r = L[lane];                                                                                                 \
    (void)r;                                                                                                           \
    stmt;                                                                                                              \
  }
  // dst of lane l = src of lane l - 1 (SHR) or l + 1 (SHL), 0 past the ends
#define SHR(dst, src) EACH(r.dst = lane > 0 ? L[lane - 1].src : R(0))
#define SHL(dst, src) EACH(r.dst = lane < 63 ? L[lane + 1].src : R(0))
  for (int task = 0; task < g.ntasks; ++task) {
    int i0, jb, je;
    march_task_rows(g, kp.Ny, task / g.per_band, task % g.per_band, i0, jb, je);
    if (jb >= je) continue;
    for (auto &x : low) x = std::numeric_limits<R>::quiet_NaN();
    for (auto &x : ring) x = std::numeric_limits<S>::quiet_NaN();
    for (int lane = 0; lane < 64; ++lane) {
      memset((void *)&L[lane], 0xff, sizeof(Lane));
      L[lane].low = low.data() + lane;
      L[lane].ring = K::kRing ? ring.data() + lane : nullptr;
      K::set_column(lane, i0, kp, L[lane]);
    }
    for (int lane = 0; lane < 64; ++lane) {
      Lane &r = L[lane];
      S raw[4][4];
      for (int k = 0; k < 4; ++k) K::fetch_row(jb - 2 + k, kp, io, r, raw[k]);
      K::fetch_row(jb + 2, kp, io, r, r.raw);
      K::pro_rows(jb, raw, kp, io, r);
    }
    if (K::kVISC) {
      SHR(u0l, um) SHR(v0l, vm) SHR(u1l, q0[IU]) SHR(v1l, q0[IV]) SHL(u1r, q0[IU]) SHL(v1r, q0[IV])
      std::vector<R> up(64), vp(64);
      for (int l = 0; l < 64; ++l) {
        up[l] = l < 63 ? L[l + 1].um : R(0);
        vp[l] = l < 63 ? L[l + 1].vm : R(0);
      }
      EACH(K::pro_visc(up[lane], vp[lane], kp, r))
    }
    EACH(K::put_low(r))
    for (int j = jb; j < je; ++j) {
      EACH(K::row_begin(j, kp, io, r))
      for (int v = 0; v < 4; ++v) SHL(q0r[v], q0[v])
      if (K::kTC) SHL(t0r, t0)
      EACH(K::row_diffs(r))
      if (K::kPLM)
        for (int v = 0; v < 4; ++v) SHR(dl[v], d[v])
      if (K::kVISC) {
        SHL(eur, eu) SHL(evr, ev)
        SHR(u0l, q0[IU]) SHR(v0l, q0[IV]) SHR(u1l, q1[IU]) SHR(v1l, q1[IV]) SHL(u1r, q1[IU]) SHL(v1r, q1[IV])
      }
      EACH(K::row_slopes(r))
      EACH(K::park(r))
      for (int v = 0; v < 4; ++v) EACH(r.bXr[v] = L[lane < 63 ? lane + 1 : lane].bX[v])
      EACH(K::row_fluxes(kp, r))
      std::vector<std::array<S, 4>> u(64);
      EACH(K::load_own(j, kp, io, r, u[lane].data()))
      EACH(K::fetch_row(j + 3, kp, io, r, r.raw))
      for (int v = 0; v < 4; ++v) SHR(fxl[v], fx[v])
      if (K::kTC) SHR(tcxl, tcx)
      if (K::kVISC)
        for (int k = 0; k < 3; ++k) SHR(vxl[k], vx[k])
      EACH(K::row_update(lane, j, i0, kp, io, s.ctl.dt, s.ctl.dt_dx, s.ctl.dt_dy, u[lane].data(), r))
      EACH(K::row_next(r))
    }
    for (auto &r : L) best = fmax(best, r.inv);
  }
#undef EACH
#undef SHR
#undef SHL
  if (io.epilogue) {
    for (auto &x : s.partials) x = 0.0;
    s.partials[0] = best;
  }
}

template <typename R, typename S, int RC, int RM, bool XG>
void march_rr(Sim &s, const StageIO<S> &io) {
  const bool tc = s.p.tc_active, vi = s.p.visc_active;
  if (tc && vi) march_run<MarchStage<R, S, RC, RM, true, true, XG>, R, S>(s, io);
  else if (tc) march_run<MarchStage<R, S, RC, RM, true, false, XG>, R, S>(s, io);
  else if (vi) march_run<MarchStage<R, S, RC, RM, false, true, XG>, R, S>(s, io);
  else march_run<MarchStage<R, S, RC, RM, false, false, XG>, R, S>(s, io);
}

// MARCH_EMU_FEW: only PLM / HLLC with conduction and viscosity (the sanitized build).
template <typename R, typename S, int RC>
void march_r(Sim &s, const StageIO<S> &io) {
  const KParams &kp = s.kp;
  const bool xg = kp.grav != GRAV_NONE || kp.wb || kp.bctc_ymin || kp.bctc_ymax;
#ifdef MARCH_EMU_FEW
  if (xg) march_run<MarchStage<R, S, PLM, HLLC, true, true, true>, R, S>(s, io);
  else march_run<MarchStage<R, S, PLM, HLLC, true, true, false>, R, S>(s, io);
#else
#define EMU_RM(RM) (xg ? march_rr<R, S, RC, RM, true>(s, io) : march_rr<R, S, RC, RM, false>(s, io))
  switch (s.p.riemann_solver) {
  case HLL: EMU_RM(HLL); break;
  case FSLP: EMU_RM(FSLP); break;
  default: EMU_RM(HLLC); break;
  }
#undef EMU_RM
#endif
}

template <typename R, typename S, int NW>
void march_stage(Sim &s, const StageIO<S> &io) {
#ifdef MARCH_EMU_FEW
  march_r<R, S, PLM>(s, io);
#else
  if (s.p.reconstruction == FV2D_PLM) march_r<R, S, PLM>(s, io);
  else march_r<R, S, PCM>(s, io);
#endif
}

}  // namespace emu

#define stage_nw march_stage
#include "tile_emu.cpp"

// Tasks of the split the march kernel takes for these parameters: returns their number and fills (i0,
// jb, je) of each into out (when not NULL); bands into *bands.
extern "C" int emu_march_tasks(const fv2d_params *p, int *out, int *bands) {
  const MarchGeom g = sim_march_geom(p);
  *bands = g.bands;
  if (out)
    for (int t = 0; t < g.ntasks; ++t)
      march_task_rows(g, p->Ny, t / g.per_band, t % g.per_band, out[3 * t], out[3 * t + 1], out[3 * t + 2]);
  return g.ntasks;
}
