// The right-hand side of one point of the fused 2-D stages, shared by the
// kernels that run one RK stage per launch, two of them, or a batch.
#pragma once

#include "lee_device.h"

namespace lee {

namespace {

// Chain rule and LEE right-hand side of a point from its values yc and
// index-space derivatives dx, dy (s', u', v', p'), its FP64 metrics m and J
// and, for a non-uniform mean, its coefficients mc(f), f an MC_* index (STALE:
// with the carried aux density rho() instead of that of yc).  They are asked
// for after the chain rule, where a caller may read them from memory (see
// stage_rhs).  Every fusion is written out (fmx), so all callers round alike.
template <typename T, bool MEANF, bool STALE, typename AT, typename Mean, typename Rho>
__device__ __forceinline__ void stage_terms(const AT &a, const double (&m)[4], double J, Mean mc, Rho stale_rho,
                                            const T (&yc)[4], const T (&dx)[4], const T (&dy)[4], T (&r)[4]) {
#pragma clang fp contract(off)
  // chain rule with FP64 metrics (spatial:1810-1820)
  const double mxx = m[0], mxy = m[1], myx = m[2], myy = m[3];
  T fx[4], fy[4];
#pragma unroll
  for (int v = 0; v < 4; v++) {
    fx[v] = (T)(fmx(mxx, (double)dx[v], myx * (double)dy[v]) * J);
    fy[v] = (T)(fmx(mxy, (double)dx[v], myy * (double)dy[v]) * J);
  }
  // LEE right-hand side (spatial:2053-2130), reference term order
  const T sv = yc[0], uv = yc[1], vv = yc[2], pv = yc[3];
  T rs, ru, rv, rp;
  if (!MEANF) {
    const T u0 = (T)a.u0, v0 = (T)a.v0, gp0 = (T)a.gp0;
    rs = -(u0 * fx[0]);
    rs = fmx(-v0, fy[0], rs);
    ru = -(u0 * fx[1]);
    ru = fmx(-v0, fy[1], ru);
    rv = -(u0 * fx[2]);
    rv = fmx(-v0, fy[2], rv);
    if (sizeof(T) == 8) {
      ru -= fx[3] / (T)a.rhob0;
      rv -= fy[3] / (T)a.rhob0;
    } else {
      const T irb = (T)(1.0 / a.rhob0);
      ru = fmx(-fx[3], irb, ru);
      rv = fmx(-fy[3], irb, rv);
    }
    rp = -(u0 * fx[3]);
    rp = fmx(-gp0, fx[1], rp);
    rp = fmx(-v0, fy[3], rp);
    rp = fmx(-gp0, fy[2], rp);
  } else {
    // per-point mean coefficients (MC_* order): u, v, gamma p, 1/rho,
    // the eight mean gradients, rho gi / p and rho (all at the point)
    const T u0 = mc(MC_U), v0 = mc(MC_V), gp = mc(MC_GP), irb = mc(MC_IRB);
    const T gsx = mc(MC_GSX), gsy = mc(MC_GSY), gux = mc(MC_GUX), guy = mc(MC_GUY);
    const T gvx = mc(MC_GVX), gvy = mc(MC_GVY), gpx = mc(MC_GPX), gpy = mc(MC_GPY);
    const T rho = STALE ? stale_rho() : fmx(pv, mc(MC_RP), -(sv * mc(MC_RB)));
    const T g = (T)a.gamma;
    const T ru_fac = rho * irb;
    const T uf = fmx(ru_fac, u0, uv), vf = fmx(ru_fac, v0, vv), gpv = g * pv;
    rs = -(u0 * fx[0]);
    rs = fmx(-uv, gsx, rs);
    rs = fmx(-v0, fy[0], rs);
    rs = fmx(-vv, gsy, rs);
    ru = -(u0 * fx[1]);
    ru = fmx(-uf, gux, ru);
    ru = fmx(-v0, fy[1], ru);
    ru = fmx(-vf, guy, ru);
    ru = fmx(-fx[3], irb, ru);
    rv = -(u0 * fx[2]);
    rv = fmx(-uf, gvx, rv);
    rv = fmx(-v0, fy[2], rv);
    rv = fmx(-vf, gvy, rv);
    rv = fmx(-fy[3], irb, rv);
    rp = -(u0 * fx[3]);
    rp = fmx(-uv, gpx, rp);
    rp = fmx(-gp, fx[1], rp);
    rp = fmx(-gpv, gux, rp);
    rp = fmx(-v0, fy[3], rp);
    rp = fmx(-vv, gpy, rp);
    rp = fmx(-gp, fy[2], rp);
    rp = fmx(-gpv, gvy, rp);
    // axisymmetry (spatial:2119-2126): -gamma (pbar v' + p' vbar) / (r + 1e-99)
    if (a.axi) rp -= fmx(gp, vv, g * v0 * pv) / mc(MC_R);
  }
  r[0] = rs;
  r[1] = ru;
  r[2] = rv;
  r[3] = rp;
}

// One Freund sponge of strength sg (source.cpp:136-201): s' relaxes by ds,
// the other variables to 0.
template <typename T>
__device__ __forceinline__ void sponge_relax(T sg, T ds, const T (&yc)[4], T (&r)[4]) {
  r[0] = fmx(-sg, ds, r[0]);
  r[1] = fmx(-sg, yc[1], r[1]);
  r[2] = fmx(-sg, yc[2], r[2]);
  r[3] = fmx(-sg, yc[3], r[3]);
}

// The whole right-hand side of block point p = (gi, gj): stage_terms, the
// source and the sponges, zone by zone, with the entropy factor he.
template <typename T, bool MEANF, bool STALE, typename AT>
__device__ __forceinline__ void stage_rhs(const AT &a, double s1, double s2, double he, int gi, int gj, int p, int n,
                                          const double (&m)[4], double J, const T (&yc)[4], const T (&dx)[4],
                                          const T (&dy)[4], T (&r)[4]) {
#pragma clang fp contract(off)
  // the mean coefficients straight from memory: gathered before the chain rule
  // they take the middle 11-point stage in FP64 from 152 to 238 registers, and
  // 11-point steps were 5 to 11 % slower (1025 x 769 FP64 249 -> 275 us)
  stage_terms<T, MEANF, STALE>(a, m, J, [&](int f) { return a.mc[f * n + p]; }, [&]() { return a.rho_in[p]; }, yc, dx, dy,
                               r);
  // physical source (source.cpp:22-107), pressure equation
  if (gi >= a.si0 && gi <= a.si1 && gj >= a.sj0 && gj <= a.sj1) {
    const double gval = a.g[(gj - a.sj0) * (a.si1 - a.si0 + 1) + (gi - a.si0)];
    r[3] += (T)(s1 * gval * s2);
  }
  // Freund sponges, zone by zone (source.cpp:136-201), sol_ref = 0
#pragma unroll 1
  for (int z = 0; z < a.nz; z++) {
    const auto &zz = a.z[z];
    if (gi >= zz.i0 && gi <= zz.i1 && gj >= zz.j0 && gj <= zz.j1) {
      const int zp = (gj - zz.j0) * zz.nzi + (gi - zz.i0);
      const T sg = zz.sig[zp];
      // a harmonic-wave zone relaxes s' to e(t) g (source.cpp:264-320)
      const T ds = zz.harm ? yc[0] - (T)(zz.hg ? he * zz.hg[zp] : he) : yc[0];
      sponge_relax(sg, ds, yc, r);
    }
  }
}

}  // namespace

}  // namespace lee
