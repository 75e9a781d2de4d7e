// Host-side operands of the fused 2-D kernels.
#pragma once

#include <cmath>

#include "lee_bc.h"
#include "lee_device.h"
#include "lee_internal.h"

namespace lee {

namespace {

inline BcArgs make_bc_args(const lee_handle *h, const Block &b, const BcFace &f, double he) {
  BcArgs a{};
  a.he = he;
  a.hg = f.hg;
  a.type = f.type;
  a.dir = f.dir;
  a.end = f.end;
  a.i0 = f.is[0];
  a.i1 = f.ie[0];
  a.j0 = f.is[1];
  a.j1 = f.ie[1];
  a.ni = b.ni;
  a.nj = b.nj;
  a.sb = h->fd.sb;
  a.nsc = h->cfg.num_scalar;
  for (int q = 0; q < 9; q++) a.neu[q] = h->fd.bnd[0][q];
  return a;
}

// The points face a writes, grown by those its rows read.
struct BcReach {
  int lo[2], hi[2];
};
inline BcReach bc_reach(const BcArgs &a) {
  BcReach r{{a.i0, a.j0}, {a.i1, a.j1}};
  if (a.end == 0) r.hi[a.dir] += a.sb - 1;
  else r.lo[a.dir] -= a.sb - 1;
  return r;
}
inline bool bc_apart(const BcReach &r, const BcReach &o) {
  return r.lo[0] > o.hi[0] || o.lo[0] > r.hi[0] || r.lo[1] > o.hi[1] || o.lo[1] > r.hi[1];
}

template <typename T>
inline void fill_zones(StageArgs<T> &a, const Block &b) {
  a.nz = 0;
  for (const auto &z : b.zones) {
    if (a.nz >= MAX_ZONES) break;
    ZoneT<T> &q = a.z[a.nz++];
    q.i0 = z.is[0];
    q.i1 = z.ie[0];
    q.j0 = z.is[1];
    q.j1 = z.ie[1];
    q.nzi = z.nz[0];
    if constexpr (sizeof(T) == 8) q.sig = (const T *)z.sigma64;
    else q.sig = (const T *)z.sigma32;
    q.harm = z.harmonic ? 1 : 0;
    q.hg = z.hg;
  }
}

// Stage kind of RK stage `stage`; below 0, runs on scratch buffers: -1 the
// right-hand side (a middle stage), -2 and -3 the tuner's first and last stage.
inline int stage_kind(const lee_handle *h, int stage) {
  const int last = h->cfg.rk_stages - 1;
  if (stage < 0) return stage == -2 ? STAGE_FIRST : (stage == -3 ? STAGE_LAST : STAGE_MID);
  return stage == 0 ? STAGE_FIRST : (stage == last ? STAGE_LAST : STAGE_MID);
}

// Operands of one RK stage on block b with R rows per thread.
template <typename T>
inline StageArgs<T> make_stage_args(const lee_handle *h, const Block &b, int stage, T *const *Y, T *rho, int R,
                                    const StageScalars &sc) {
  StageArgs<T> a{};
  a.ni = b.ni;
  a.nj = b.nj;
  a.ntx = (b.ni + ST_TX - 1) / ST_TX;
  a.nty = (b.nj + 4 * R - 1) / (4 * R);
  a.ntiles = a.ntx * a.nty;
  a.chunk = (a.ntiles + 7) / 8;
  // stage 0 reads Y0 and writes Y1 (accumulator) and Y2; odd stages read
  // Y2 and write Y3, even stages read Y3 and write Y2; y_n stays in Y0.
  // stage < 0 (lee_compute_rhs): y in Y[2], zeroed accumulator Y[3] with
  // h = b = 1 receives the RHS, Y[1] is scratch
  const int in_idx = stage == 0 ? 0 : (stage % 2 == 1 ? 2 : 3);
  const int out_idx = stage % 2 == 0 ? 2 : 3;
  a.yin = Y[in_idx];
  a.yn = Y[0];
  a.acc = Y[1];
  a.yout = Y[out_idx];
  if (stage < 0) {
    a.yin = Y[2];
    a.yn = Y[2];
    a.acc = Y[3];
    a.yout = Y[1];
  }
  a.rho_in = rho;
  a.rho_out = stage < 0 ? Y[1] : rho;
  a.met = b.met;
  a.jac = b.jac;
  a.iblank = b.iblank;
  a.code = b.code_fd;
  a.clean = b.clean_fd;
  a.mean = b.mean;
  a.mgrad = b.mgrad;
  a.rhob = b.rhobar;
  a.mc = sizeof(T) == 8 ? (const T *)b.mc64 : (const T *)b.mc32;
  a.u0 = b.umean[IUX];
  a.v0 = b.umean[IUY];
  a.gamma = h->cfg.gamma;
  a.axi = h->cfg.axisym;
  a.gi = 1.0 / h->cfg.gamma;
  a.gp0 = h->cfg.gamma * b.umean[IP];
  {
    const double pbar = b.umean[IP], sbar = b.umean[IS];
    a.rhob0 = std::pow(h->cfg.gamma * pbar, 1.0 / h->cfg.gamma) * std::exp(-sbar);
  }
  fill_zones(a, b);
  a.si0 = b.src.i0;
  a.si1 = b.src.i1;
  a.sj0 = b.src.j0;
  a.sj1 = b.src.j1;
  a.g = b.src.g;
  a.s1 = sc.s1;
  a.s2 = sc.s2;
  a.he = sc.he;
  a.h = (T)sc.h;
  a.b = (T)sc.b;
  a.a = (T)sc.a;
  a.fdw = h->fdw;
  return a;
}

template <typename T>
struct BatchStageArgs {
  const StageArgs<T> *args;      // nsolve entries for this stage
  const int *map;                // (solve, tile) per list entry
  const BatchSched *sched;       // [step][solve][stage]
  const int *counter;            // step index within the schedule
  int nsolve, nstage, stage, total, chunk;
  T b, a;
};

// A device table as a constant-address-space pointer (the kernels' view).
template <typename P>
inline const LEE_CONST_AS P *CA(const P *p) {
  return (const LEE_CONST_AS P *)p;
}

}  // namespace

}  // namespace lee
