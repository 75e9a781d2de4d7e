// Boundary conditions of one face point (boundary_condition.cpp:46-545), for
// kernels that keep the state in global memory or in LDS.
#pragma once

#include "lee_device.h"

namespace lee {

namespace {

struct BcArgs {
  int type, dir, end;
  int i0, i1, j0, j1;   // face box (collapsed along dir)
  int ni, nj;
  double neu[9];        // closure row 0 of the FD operator (sb entries)
  int sb;
  double he;            // dirichlet_harmonicwave: entropy factor e(t) at the BC time
  const double *hg;     // and g per face point (null: 1)
  int nsc;              // passive scalars (variables NV .. NV + nsc - 1)
};

__device__ __forceinline__ bool bc_is_neumann(const BcArgs &a) {
  return a.type == LEE_BC_NEUMANN || a.type == LEE_BC_WALL_SLIP_KINEMATIC ||
         (a.type >= LEE_BC_CENTERLINE_CART_NORM2X && a.type <= LEE_BC_CENTERLINE_AXISYM);
}

// bc_neumann (boundary_condition.cpp:348-444): the face value whose closure
// row vanishes, from the values nb[s - 1] at s points inward; c is the face
// coordinate on a line of length len.  NS: the most entries past the first
// that a row of the operator has (2 for OA4 alone, 8 with FDO11P).
template <typename T, int NS>
__device__ __forceinline__ double bc_neumann_value(const BcArgs &a, int c, int len, const T (&nb)[NS]) {
#pragma clang fp contract(off)
  const int sg = a.end == 0 ? 1 : -1;
  double d = 0.0;
#pragma unroll
  for (int s = 1; s <= NS; s++) {
    const int cs = c + sg * s;
    const bool use = (NS == 2 || s < a.sb) && cs >= 0 && cs < len;
    const double t1 = a.end == 0 ? d - a.neu[s] * (double)nb[s - 1] : d + a.neu[s] * (double)nb[s - 1];
    d = use ? t1 : d;
  }
  d /= a.end == 0 ? a.neu[0] : -a.neu[0];
  return d;
}

// bc::apply_BC of one face point (boundary_condition.cpp:46-209) with
// bc_neumann (:348-444), bc_wall_slip_kinematic (:448-494), dirichlet_allzero
// and the centerline conditions.  Arithmetic in FP64 for both precisions.
// Face point q of the face box (i fastest), block point p; get(v, s) is the
// value of variable v at s points inward (s = 0: the face point; clamped to
// the face point where that leaves the block).  Only s < a.sb is asked for:
// the points that bc_reach counts.
template <typename T, int NS, typename Get>
__device__ __forceinline__ void bc_face_data(const BcArgs &a, int q, int p, int c, int len, const double *met,
                                             const double *jac, Get get, double (&data)[NV]) {
#pragma clang fp contract(off)
  const int n = a.ni * a.nj;
  for (int v = 0; v < NV; v++) data[v] = 1.0e9 * (double)(a.dir + 1);
  if (a.type == LEE_BC_DIRICHLET_ALLZERO)
    for (int v = 0; v < NV; v++) data[v] = 0.0;
  if (a.type == LEE_BC_DIRICHLET_HARMONICWAVE) {  // WAVE_ENTROPY: s' = e(t) g, the rest 0 (bc:250-334)
    for (int v = 0; v < NV; v++) data[v] = 0.0;
    data[IS] = a.hg ? a.he * a.hg[q] : a.he;
  }
  if (bc_is_neumann(a)) {
    // every neighbour value is requested first (clamped addresses), then the
    // closure row is solved in the reference's order with the skipped
    // entries masked: one memory latency instead of one per entry
    T nb[NV][NS];
#pragma unroll
    for (int s = 1; s <= NS; s++)
#pragma unroll
      for (int v = 0; v < NV; v++) nb[v][s - 1] = get(v, NS == 2 || s < a.sb ? s : 0);
    for (int v = 0; v < NV; v++) {
      if (a.type == LEE_BC_WALL_SLIP_KINEMATIC && v >= IUX && v <= IUZ) continue;
      data[v] = bc_neumann_value<T, NS>(a, c, len, nb[v]);
    }
  }
  if (a.type == LEE_BC_WALL_SLIP_KINEMATIC) {
    const double m00 = met[p], m01 = met[(size_t)n + p], m10 = met[(size_t)2 * n + p], m11 = met[(size_t)3 * n + p];
    const double u = (double)get(IUX, 0), v = (double)get(IUY, 0);
    double k0 = 0.0, k1 = 0.0;
    k0 += m00 * u;
    k0 += m01 * v;
    k1 += m10 * u;
    k1 += m11 * v;
    if (a.dir == 0) k0 = 0.0; else k1 = 0.0;
    // metricsInverse (metrics.cpp:375-381): [X][XI] = eta_y, [X][ETA] = -xi_y,
    // [Y][XI] = -eta_x, [Y][ETA] = xi_x
    const double J = jac[p];
    double ux = 0.0, uy = 0.0;
    ux += m11 * k0;
    ux += -m01 * k1;
    ux *= J;
    uy += -m10 * k0;
    uy += m00 * k1;
    uy *= J;
    data[IUX] = ux;
    data[IUY] = uy;
    data[IUZ] = (double)get(IUZ, 0);
  }
  if (a.type >= LEE_BC_CENTERLINE_CART_NORM2X && a.type <= LEE_BC_CENTERLINE_CART_NORM2Z)
    data[IUX + (a.type - LEE_BC_CENTERLINE_CART_NORM2X)] = 0.0;
  if (a.type == LEE_BC_CENTERLINE_AXISYM) data[IUY] = 0.0;  // u_r on the axis (bc:498-545, IVAR_UR)
}

}  // namespace

}  // namespace lee
