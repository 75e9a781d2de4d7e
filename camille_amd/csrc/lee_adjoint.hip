// Discrete adjoint of the fused 2-D LEE time advance (no reference
// counterpart: the reference has no adjoint).
//
// The forward step with stage inputs u_i, stage RHS k_i = L(u_i, rho_i) + q s_i,
// accumulator acc_{i+1} = acc_i + b_i h k_i (acc_0 = y_n), next input
// u_{i+1} = y_n + a_i h k_i, filtered state y_{n+1} = F(acc_S) and the
// stale aux density rho_{n+1} = R(acc_S) (R(y) = rho_bar (p'/(gamma p_bar) - s'),
// consumed by stage 0 of the next step) is linear in (y_n, rho_n) and
// affine in the source field q.  Its exact transpose, step by step
// backwards, is
//   lambda* = F^T lambda_{n+1} + R^T mu_{n+1}
//   kappa_i = b_i h lambda* + a_i h lambda_u{i+1}        (last stage: b_i h lambda*)
//   lambda_u_i = L_u^T kappa_i + R^T L_rho^T kappa_i     (i >= 1)
//   lambda_n = lambda* + sum_{i>=1} lambda_u_i + L_u^T kappa_0,   mu_n = L_rho^T kappa_0
//   dJ/dq += sum_i s_i kappa_i[p']
// with the transposed operators built from the same row codes as the
// forward: (D^T f)_i = sum over rows j touching i of w(code_j, i - j) f_j.
// L^T applies D_xi^T and D_eta^T to per-point flux fields
// J (m_xi,x A + m_xi,y B), J (m_eta,x A + m_eta,y B), where A, B are the
// coefficients of d/dx and d/dy in each RHS term times kappa, evaluated at
// the row's own point.  The filter transposes as rem I + blend F_xi^T F_eta^T.
#include <hip/hip_runtime.h>

#include <cmath>

#include "lee_device.h"
#include "lee_internal.h"

namespace lee {

namespace {

// Weight of the FD row with code `code` (at point j) on point j + d: the
// rows of fd_row (lee_device.h) written out by offset.
template <typename T>
__device__ __forceinline__ T fd_wt(int code, int d) {
  const T c1 = (T)(8.0 / 12.0), c2 = (T)(-1.0 / 12.0);
  switch (code) {
    case CODE_INTERIOR:
      return d == -2 ? -c2 : d == -1 ? -c1 : d == 1 ? c1 : d == 2 ? c2 : (T)0;
    case CODE_ZERO:
      return (T)0;
    case CODE_LEFT + 0:
      return d == 0 ? (T)(-3.0 / 2.0) : d == 1 ? (T)(4.0 / 2.0) : d == 2 ? (T)(-1.0 / 2.0) : (T)0;
    case CODE_LEFT + 1:
      return d == -1 ? (T)(-1.0 / 2.0) : d == 1 ? (T)(1.0 / 2.0) : (T)0;
    case CODE_LEFT + 2:
      return d == 0 ? (T)(3.0 / 2.0) : d == -1 ? (T)(-4.0 / 2.0) : d == -2 ? (T)(1.0 / 2.0) : (T)0;
    default:
      return d == 1 ? (T)(1.0 / 2.0) : d == -1 ? (T)(-1.0 / 2.0) : (T)0;
  }
}

// Transposed FD row where every neighbour's row is interior: D^T = -D there
// (fusions as in row_t5_sum).
template <typename T>
__device__ __forceinline__ T fd_row_t_inner(const T *f, int st) {
#pragma clang fp contract(off)
  const T c1 = (T)(8.0 / 12.0), c2 = (T)(-1.0 / 12.0);
  T acc = c2 * f[-2 * st];
  acc = fmx(c1, f[-st], acc);
  acc = fmx(-c1, f[st], acc);
  return fmx(-c2, f[2 * st], acc);
}

// Transposed FD row at block point p (coordinate c of a line of length
// len, stride gs in the block, st in LDS) with the per-point codes of a
// block with holes: the rows of the neighbours c + o, o in [-2, 2].
template <typename T>
__device__ __forceinline__ T fd_row_t_codes(const T *f, int st, int c, int len, const int8_t *code, int p, int gs) {
  T acc = 0;
#pragma unroll
  for (int o = -2; o <= 2; o++) {
    const int j = c + o;
    if (j < 0 || j >= len) continue;
    acc += fd_wt<T>((int)code[p + o * gs], -o) * f[o * st];
  }
  return acc;
}

template <typename T, int ORDER>
__device__ __forceinline__ T flt_row_t_codes(const T *f, int st, int c, int len, const int8_t *code, int p, int gs) {
  constexpr int H = ORDER / 2;
  T acc = 0;
#pragma unroll
  for (int o = -H; o <= H; o++) {
    const int j = c + o;
    if (j < 0 || j >= len) continue;
    acc += flt_wt<T, ORDER>((int)code[p + o * gs], -o) * f[o * st];
  }
  return acc;
}

template <typename T>
struct AdjArgs {
  int ni, nj, ntx, nty, ntiles, chunk;
  const T *lacc;   // adjoint of the accumulator after the last stage (5n)
  const T *lin;    // adjoint of the next stage input (null at the last stage)
  const T *lyin;   // running adjoint of y_n (null when nothing has reached it yet)
  T *lout;         // adjoint of this stage's input; at stage 0 the adjoint of y_n
  T *lyout;        // running adjoint of y_n (middle stages; may equal lyin)
  T *mu;           // adjoint of the stale aux density (stage 0, non-uniform mean)
  double *grad;    // adjoint of the source field (n), accumulated (null: none)
  const double *met, *jac, *mean, *mgrad, *rhob;
  double u0, v0, gp0, rhob0, gamma, gi;
  int nz;
  ZoneT<T> z[MAX_ZONES];
  double hb, ha;   // b_i h and a_i h
  double src;      // s1 s2 of this stage
  const int8_t *iblank, *code;  // holes only: iblank, FD codes (xi then eta)
  const int *clean;             // holes only: integral image of points off the interior FD rows
  const T *rad;                 // axisymmetric runs: the forward's radius field r + 1e-99 (null: none)
};

constexpr int ADJ_TX = 32, ADJ_TY = 8;  // points of a tile

// What bounds it: latency, of the fluxes' operands and of each tile's serial
// work, more than its 296 bytes a point (FP64, general mean).  Tiles of 32 x
// 8 points, their halo one direction a lane (1.3 evaluations a point), the
// point's operands requested before the barrier, transposed closure rows
// without branches.  Middle stage of 385 x 257 FP64: 25 us with 64 x 8 tiles
// whose halo went eight lanes at a time, 12.7 with 64 x 4 tiles and the whole
// region in both directions, 11.4 now; whole reverse step of 1025 x 513 268
// -> 255, of 2049 x 1025 1087 -> 1051 against the second form.
// One reversed RK stage on a tile: kappa and the flux fields on the tile and
// its 2-point halo go to LDS, then the transposed stencils, the point-local
// transposed terms and the accumulations of the running adjoints.
// Blocks with holes (HOLES): the forward stage writes 0 at BLANKED points
// whatever its inputs, so the adjoints arriving there (lacc, lin) count as 0
// and kappa vanishes there; the transposed rows take the per-point codes.
template <typename T, bool MEANF, int KIND, bool HOLES>
__global__ void __launch_bounds__(TPB) k_adj_stage(AdjArgs<T> a) {
  constexpr int H = ST_H;
  __shared__ T FX[4][ADJ_TY][ADJ_TX + 2 * H];  // xi fluxes with their halo columns
  __shared__ T FE[4][ADJ_TY + 2 * H][ADJ_TX];  // eta fluxes with their halo rows
  const int tile = xcd_tile(blockIdx.x, a.chunk);
  if (tile >= a.ntiles) return;
  const int tx = threadIdx.x, ty = threadIdx.y, tid = ty * ADJ_TX + tx;
  const int i0 = (tile % a.ntx) * ADJ_TX, j0 = (tile / a.ntx) * ADJ_TY;
  const int ni = a.ni, nj = a.nj, n = ni * nj;
  const int VOFF[4] = {IS * n, IUX * n, IUY * n, IP * n};
  const bool inner = HOLES ? box_clean(a.clean, ni, nj, i0 - H, i0 + ADJ_TX + H, j0 - H, j0 + ADJ_TY + H)
                           : (i0 >= 2 * H && i0 + ADJ_TX + 2 * H <= ni && j0 >= 2 * H && j0 + ADJ_TY + 2 * H <= nj);
  const T hb = (T)a.hb, ha = (T)a.ha;
  // sponge zones of the tile: the boxes are kernel arguments at fixed places,
  // read all at once
  unsigned zmask = 0;
#pragma unroll
  for (int z = 0; z < MAX_ZONES; z++)
    zmask |= z < a.nz && a.z[z].i0 < i0 + ADJ_TX && a.z[z].i1 >= i0 && a.z[z].j0 < j0 + ADJ_TY && a.z[z].j1 >= j0
                 ? 1u << z : 0;

  // (1) kappa and fluxes: every thread's own point in both directions, then
  // a point of the halo, in the direction that reads it, by 160 lanes (four
  // rows by waves 0 and 1, four columns by half of wave 2); points outside
  // the block evaluate the nearest one inside and store 0
  struct Point {
    double k[4], u0, v0, c, irb, J;  // c = gamma p kappa_p; J the negative Jacobian
    bool ok;
  };
  auto point = [&](int ri, int rj, int p) {
    Point q;
    q.ok = rj >= 0 && rj < nj && ri >= 0 && ri < ni && !(HOLES && a.iblank[p] == BLANKED);
#pragma unroll
    for (int v = 0; v < 4; v++) {
      T kv = hb * a.lacc[VOFF[v] + p];
      if (KIND != STAGE_LAST && a.lin) kv += ha * a.lin[VOFF[v] + p];
      q.k[v] = kv;
    }
    double gp = a.gp0;
    q.u0 = a.u0;
    q.v0 = a.v0;
    q.irb = 1.0 / a.rhob0;
    if (MEANF) {
      q.u0 = a.mean[IUX * n + p];
      q.v0 = a.mean[IUY * n + p];
      gp = a.gamma * a.mean[IP * n + p];
      q.irb = 1.0 / a.rhob[p];
    }
    q.c = gp * q.k[3];
    q.J = -a.jac[p];
    return q;
  };
  // F_l = -J (U_l kappa + ...) with the contravariant velocity U_l
  auto flux = [&](const Point &q, double mx, double my, T (&f)[4]) {
    const double U = mx * q.u0 + my * q.v0;
    f[0] = (T)(U * q.k[0] * q.J);
    f[1] = (T)((U * q.k[1] + mx * q.c) * q.J);
    f[2] = (T)((U * q.k[2] + my * q.c) * q.J);
    f[3] = (T)((U * q.k[3] + (mx * q.k[1] + my * q.k[2]) * q.irb) * q.J);
  };
  const int gi = i0 + tx, gj = j0 + ty;
  const int p = min(gj, nj - 1) * ni + min(gi, ni - 1);
  {
    const Point q = point(gi, gj, p);
    T f[2][4];
#pragma unroll
    for (int l = 0; l < 2; l++)
      flux(q, a.met[(size_t)(2 * l) * n + p], a.met[(size_t)(2 * l + 1) * n + p], f[l]);
#pragma unroll
    for (int v = 0; v < 4; v++) {
      FX[v][ty][tx + H] = q.ok ? f[0][v] : (T)0;
      FE[v][ty + H][tx] = q.ok ? f[1][v] : (T)0;
    }
  }
  static_assert(ADJ_TX == 32 && ADJ_TY == 8 && TPB == 256, "halo lanes");
  if (tid < 160) {
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), hq = wave < 2 ? tid >> 5 : tid & 3;
    const int hr = wave < 2 ? (hq < 2 ? hq : hq + ADJ_TY) : (tid >> 2) & 7;  // row of FE or FX
    const int hc = wave < 2 ? tx : (hq < 2 ? hq : hq + ADJ_TX);              // and column
    const int hj = wave < 2 ? j0 - H + hr : j0 + hr, hi = wave < 2 ? i0 + hc : i0 - H + hc;
    const int hp = min(max(hj, 0), nj - 1) * ni + min(max(hi, 0), ni - 1);
    const double *hm = a.met + (wave < 2 ? (size_t)2 * n : 0);
    const Point q = point(hi, hj, hp);
    T f[4];
    flux(q, hm[hp], hm[(size_t)n + hp], f);
#pragma unroll
    for (int v = 0; v < 4; v++) {
      T *to = wave < 2 ? &FE[v][hr][hc] : &FX[v][hr][hc];
      *to = q.ok ? f[v] : (T)0;
    }
  }

  // (2) the operands of the thread's point, requested before the barrier
  T lacc[4], lin[4], lyin[4], mg[8];
  double mb[4];
  const bool hole = HOLES && a.iblank[p] == BLANKED;
#pragma unroll
  for (int v = 0; v < 4; v++) {
    lacc[v] = a.lacc[VOFF[v] + p];
    lin[v] = KIND != STAGE_LAST && a.lin ? a.lin[VOFF[v] + p] : (T)0;
    lyin[v] = KIND != STAGE_LAST && a.lyin ? a.lyin[VOFF[v] + p] : (T)0;
  }
  const double gr = a.grad ? a.grad[p] : 0.0;
  if (MEANF) {
    mb[0] = a.mean[IUX * n + p];
    mb[1] = a.mean[IUY * n + p];
    mb[2] = a.rhob[p];
    mb[3] = a.mean[IP * n + p];
    constexpr int GV[4] = {IS, IUX, IUY, IP};
#pragma unroll
    for (int v = 0; v < 4; v++)
#pragma unroll
      for (int d = 0; d < 2; d++) mg[2 * v + d] = (T)a.mgrad[(2 * GV[v] + d) * n + p];
  }
  __syncthreads();

  // (3) the point of the thread
  if (gi >= ni || gj >= nj) return;
  T lam[4];
  if (inner) {
#pragma unroll
    for (int v = 0; v < 4; v++) {
      lam[v] = fd_row_t_inner<T>(&FX[v][ty][tx + H], 1);
      lam[v] += fd_row_t_inner<T>(&FE[v][ty + H][tx], ADJ_TX);
    }
  } else if (HOLES) {
#pragma unroll
    for (int v = 0; v < 4; v++) {
      lam[v] = fd_row_t_codes<T>(&FX[v][ty][tx + H], 1, gi, ni, a.code, p, 1);
      lam[v] += fd_row_t_codes<T>(&FE[v][ty + H][tx], ADJ_TX, gj, nj, a.code + n, p, ni);
    }
  } else {
    const RowT5<T> rx = row_t5<T>(gi, ni), ry = row_t5<T>(gj, nj);
#pragma unroll
    for (int v = 0; v < 4; v++) {
      lam[v] = row_t5_sum<T>(rx, &FX[v][ty][tx + H], 1);
      lam[v] += row_t5_sum<T>(ry, &FE[v][ty + H][tx], ADJ_TX);
    }
  }
  // kappa at the point (recomputed from the same operands)
  T kap[4];
#pragma unroll
  for (int v = 0; v < 4; v++) {
    if (hole) lacc[v] = lin[v] = (T)0;
    T kv = hb * lacc[v];
    if (KIND != STAGE_LAST && a.lin) kv += ha * lin[v];
    kap[v] = kv;
  }
  // sponges: r_v -= sigma y_v
  for (unsigned zm = zmask; zm; zm &= zm - 1) {
    const ZoneT<T> &zz = a.z[__builtin_ctz(zm)];
    if (gi >= zz.i0 && gi <= zz.i1 && gj >= zz.j0 && gj <= zz.j1) {
      const T sg = zz.sig[(gj - zz.j0) * zz.nzi + (gi - zz.i0)];
#pragma unroll
      for (int v = 0; v < 4; v++) lam[v] += -sg * kap[v];
    }
  }
  T mur = 0;
  if (MEANF) {
    const T u0 = (T)mb[0], v0 = (T)mb[1], rb = (T)mb[2];
    const T g = (T)a.gamma;
    const T gsx = mg[0], gsy = mg[1], gux = mg[2], guy = mg[3];
    const T gvx = mg[4], gvy = mg[5], gpx = mg[6], gpy = mg[7];
    const T ks = kap[0], ku = kap[1], kv = kap[2], kp = kap[3];
    lam[1] += -(gsx * ks) - gux * ku - gvx * kv - gpx * kp;
    lam[2] += -(gsy * ks) - guy * ku - gvy * kv - gpy * kp;
    lam[3] += -(g * gux * kp) - g * gvy * kp;
    mur = -((u0 * gux + v0 * guy) * ku + (u0 * gvx + v0 * gvy) * kv) / rb;
    if (a.rad) {
      // axisymmetric term r_p -= (gamma pbar v' + gamma vbar p') / r
      // (spatial:2119-2126), with the forward's gamma pbar and r fields
      const T rr = a.rad[p], gpb = (T)(a.gamma * mb[3]);
      lam[2] += -(gpb / rr) * kp;
      lam[3] += -(g * v0 / rr) * kp;
    }
    if (KIND != STAGE_FIRST) {  // rho' of this stage's input: R(u)
      lam[0] += -(rb * mur);
      lam[3] += (T)((double)mur * mb[2] * a.gi / mb[3]);
    }
  }
  if (a.grad) a.grad[p] = gr + a.src * (double)kap[3];
  if (KIND == STAGE_FIRST) {
#pragma unroll
    for (int v = 0; v < 4; v++) {
      T out = lam[v] + lacc[v] + lin[v];
      if (a.lyin) out += lyin[v];
      a.lout[VOFF[v] + p] = out;
    }
    if (MEANF) a.mu[p] = mur;
  } else {
#pragma unroll
    for (int v = 0; v < 4; v++) a.lout[VOFF[v] + p] = lam[v];
    if (a.lyout) {
#pragma unroll
      for (int v = 0; v < 4; v++) {
        T y = lin[v];
        if (a.lyin) y += lyin[v];
        a.lyout[VOFF[v] + p] = y;
      }
    }
  }
}

template <typename T>
struct AdjFilterArgs {
  int ni, nj, ntx, nty, ntiles, chunk;
  const T *src;    // adjoint of the filtered state (5n)
  T *dst;          // adjoint of the unfiltered state (5n)
  const T *mu;     // adjoint of the stale aux density taken from the unfiltered state (null: none)
  const double *mean, *rhob;
  double gi;
  T rem, blend;
  const int8_t *iblank, *code;  // holes only: iblank, filter codes (xi then eta)
  const int *clean;             // holes only: integral image of points off the interior filter rows
};

// Transposed filter on a 64 x TY tile: eta^T sweep of the (TY + 8) x 72
// region into LDS, then the xi^T sweep, blend, and R^T mu.
// Blocks with holes (HOLES): the forward filter is followed by the hole
// reset, so the adjoint arriving at a BLANKED point counts as 0, and the
// transposed rows take the per-point filter codes.
// What bounds it: latency.  Region and middle sweep go round the threads in
// line order, and closure rows are weights chosen once per line instead of a
// branch per tap: 385 x 257 FP64 16.5 -> 6.5 us.
template <typename T, int ORDER, int TY, bool HOLES>
__global__ void __launch_bounds__(TPB) k_adj_filter(AdjFilterArgs<T> a) {
  constexpr int NR = TY + 2 * FL_H, NC = FL_TX + 2 * FL_H;
  __shared__ T in[4][NR][NC];
  __shared__ T mid[4][TY][NC];
  const int tile = xcd_tile(blockIdx.x, a.chunk);
  if (tile >= a.ntiles) return;
  const int tx = threadIdx.x, ty = threadIdx.y, tid = ty * 64 + tx;
  const int i0 = (tile % a.ntx) * FL_TX, j0 = (tile / a.ntx) * TY;
  const int ni = a.ni, nj = a.nj, n = ni * nj;
  const int VOFF[4] = {IS * n, IUX * n, IUY * n, IP * n};
  // (no filter codes when the filter is off: blend is 0 and only the
  // masked identity part counts)
  const bool inner = HOLES ? (a.clean && box_clean(a.clean, ni, nj, i0 - FL_H, i0 + FL_TX + FL_H, j0 - FL_H,
                                                   j0 + TY + FL_H))
                           : (i0 >= 2 * FL_H && i0 + FL_TX + 2 * FL_H <= ni && j0 >= 2 * FL_H &&
                              j0 + TY + 2 * FL_H <= nj);
  // points outside the block read the nearest one inside and store 0
  auto load = [&](int idx) {
    const int r = idx / NC, c = idx - r * NC;
    const int gj = j0 - FL_H + r, gi = i0 - FL_H + c;
    const int p = min(max(gj, 0), nj - 1) * ni + min(max(gi, 0), ni - 1);
    const bool ok = gj >= 0 && gj < nj && gi >= 0 && gi < ni && !(HOLES && a.iblank[p] == BLANKED);
#pragma unroll
    for (int v = 0; v < 4; v++) {
      const T x = a.src[VOFF[v] + p];
      in[v][r][c] = ok ? x : (T)0;
    }
  };
#pragma unroll
  for (int q = 0; q < NR * NC / TPB; q++) load(tid + q * TPB);
  if (tid + NR * NC / TPB * TPB < NR * NC) load(tid + NR * NC / TPB * TPB);
  // the operands of R^T mu, requested before the barriers
  const int gi = i0 + tx;
  double mu[TY / 4], mp[TY / 4], rb[TY / 4];
#pragma unroll
  for (int k = 0; k < TY / 4; k++) {
    const int p = min(j0 + ty + 4 * k, nj - 1) * ni + min(gi, ni - 1);
    mu[k] = a.mu ? (double)a.mu[p] : 0.0;
    rb[k] = a.mu ? a.rhob[p] : 0.0;
    mp[k] = a.mu ? a.mean[IP * n + p] : 1.0;
  }
  __syncthreads();
  // eta^T over the tile rows, every column of the region
  auto eta = [&](int idx) {
    const int r = idx / NC, c = idx - r * NC;
    const int gj = j0 + r, gc = i0 - FL_H + c;
    if (inner) {  // symmetric interior rows: F^T = F
#pragma unroll
      for (int v = 0; v < 4; v++) mid[v][r][c] = filter_row<T, ORDER>(&in[v][r + FL_H][c], NC, CODE_INTERIOR);
    } else if (HOLES) {
      const bool ok = gj < nj && gc >= 0 && gc < ni && a.code;
#pragma unroll
      for (int v = 0; v < 4; v++)
        mid[v][r][c] =
            ok ? flt_row_t_codes<T, ORDER>(&in[v][r + FL_H][c], NC, gj, nj, a.code + n, gj * ni + gc, ni) : (T)0;
    } else {
      const FltRowT<T, ORDER> w = flt_row_t<T, ORDER>(gj, nj);
#pragma unroll
      for (int v = 0; v < 4; v++) mid[v][r][c] = flt_row_t_sum<T, ORDER>(w, &in[v][r + FL_H][c], NC);
    }
  };
#pragma unroll
  for (int q = 0; q < TY * NC / TPB; q++) eta(tid + q * TPB);
  if (tid + TY * NC / TPB * TPB < TY * NC) eta(tid + TY * NC / TPB * TPB);
  __syncthreads();
  FltRowT<T, ORDER> wx{};
  if (!HOLES && !inner) wx = flt_row_t<T, ORDER>(gi, ni);
#pragma unroll
  for (int k = 0; k < TY / 4; k++) {
    const int r = ty + 4 * k;
    const int gj = j0 + r;
    if (gi >= ni || gj >= nj) continue;
    const int p = gj * ni + gi;
    T out[4];
#pragma unroll
    for (int v = 0; v < 4; v++) {
      const T *m = &mid[v][r][tx + FL_H];
      T f;
      if (inner) f = filter_row<T, ORDER>(m, 1, CODE_INTERIOR);
      else if (HOLES) f = a.code ? flt_row_t_codes<T, ORDER>(m, 1, gi, ni, a.code, p, 1) : (T)0;
      else f = flt_row_t_sum<T, ORDER>(wx, m, 1);
      out[v] = a.rem * in[v][r + FL_H][tx + FL_H] + a.blend * f;
    }
    if (a.mu) {
      const double m = mu[k] * rb[k];
      out[0] += (T)(-m);
      out[3] += (T)(m * a.gi / mp[k]);
    }
#pragma unroll
    for (int v = 0; v < 4; v++) a.dst[VOFF[v] + p] = out[v];
  }
}

// Observer functional: J_k = sum_l w_l p'(l)^2 for one state, one workgroup,
// fixed summation order.
template <typename T>
__global__ void __launch_bounds__(1024) k_obs_energy(const T *__restrict__ y, const int *__restrict__ l,
                                                     const double *__restrict__ w, int nobs, int n,
                                                     double *__restrict__ out) {
  __shared__ double part[1024];
  double acc = 0.0;
  for (int q = threadIdx.x; q < nobs; q += 1024) {
    const double pv = (double)y[(size_t)IP * n + l[q]];
    acc += w[q] * pv * pv;
  }
  part[threadIdx.x] = acc;
  __syncthreads();
  for (int s = 512; s > 0; s >>= 1) {
    if ((int)threadIdx.x < s) part[threadIdx.x] += part[threadIdx.x + s];
    __syncthreads();
  }
  if (threadIdx.x == 0) out[0] += part[0];
}

// p' at the observer points of one state.
template <typename T>
__global__ void __launch_bounds__(TPB) k_obs_gather(const T *__restrict__ y, const int *__restrict__ l, int nobs,
                                                    int n, double *__restrict__ out) {
  const int q = blockIdx.x * TPB + threadIdx.x;
  if (q < nobs) out[q] = (double)y[(size_t)IP * n + l[q]];
}

// lambda_p += scale 2 w p' at the observer points.
template <typename T>
__global__ void __launch_bounds__(TPB) k_obs_seed(T *__restrict__ lam, const int *__restrict__ l,
                                                  const double *__restrict__ w, const double *__restrict__ samp,
                                                  int nobs, int n, double scale) {
  const int q = blockIdx.x * TPB + threadIdx.x;
  if (q < nobs) {
    const size_t p = (size_t)IP * n + l[q];
    lam[p] = (T)((double)lam[p] + scale * 2.0 * w[q] * samp[q]);
  }
}

// lambda += R^T mu: the aux density of the initial state, R(y) =
// rho_bar (p' gi / p_bar - s'), is the stale density of the first step.
template <typename T>
__global__ void __launch_bounds__(TPB) k_add_rt_mu(T *__restrict__ lam, const T *__restrict__ mu,
                                                   const double *__restrict__ mean, const double *__restrict__ rhob,
                                                   double gi, int n) {
  const int p = blockIdx.x * TPB + threadIdx.x;
  if (p >= n) return;
  const double m = (double)mu[p] * rhob[p];
  lam[(size_t)IS * n + p] = (T)((double)lam[(size_t)IS * n + p] - m);
  lam[(size_t)IP * n + p] = (T)((double)lam[(size_t)IP * n + p] + m * gi / mean[(size_t)IP * n + p]);
}

template <typename T>
__global__ void __launch_bounds__(TPB) k_fill_t(T *__restrict__ a, size_t n) {
  const size_t p = (size_t)blockIdx.x * TPB + threadIdx.x;
  if (p < n) a[p] = (T)0;
}

inline unsigned nblk(size_t n) { return (unsigned)((n + TPB - 1) / TPB); }

// ------------------------------------------- transposed boundary update
//
// The forward boundary update after a stage (spatial::update_boundary,
// spatial:2162-2187) is linear: each BC face replaces the values at its
// points, then the overset interpolation replaces every receiver by the
// weighted sum of its donors, all donor sums formed first.  Its transpose
// runs backwards: the overset part, then the faces of each block in reverse
// order.

template <typename T>
struct AdjOvTables {
  T *lam[MAX_OV_BLOCKS];
  int ni[MAX_OV_BLOCKS], nn[MAX_OV_BLOCKS];
};

// Overset transpose, part 1: each receiver's adjoint is kept in buf and
// zeroed (the forward overwrote the receiver's value).
template <typename T>
__global__ void __launch_bounds__(TPB) k_adj_ov_take(AdjOvTables<T> t, const int *__restrict__ rb,
                                                     const int *__restrict__ rl, double *__restrict__ buf,
                                                     int nrecv) {
  const int gid = blockIdx.x * TPB + threadIdx.x;
  if (gid >= NV * nrecv) return;
  const int v = gid / nrecv, r = gid - v * nrecv;
  const int b = rb[r], p = rl[r];
  if (p < 0 || p >= t.nn[b]) {
    buf[gid] = 0.0;
    return;
  }
  T *lam = t.lam[b] + (size_t)v * t.nn[b] + p;
  buf[gid] = (double)*lam;
  *lam = (T)0;
}

// Overset transpose, part 2: each receiver's adjoint goes to its donors
// with the normalised weights (the forward's donors outside the block were
// skipped, and are here).  Receivers sharing a donor add atomically.
template <typename T>
__global__ void __launch_bounds__(TPB) k_adj_ov_give(AdjOvTables<T> t, const int *__restrict__ db,
                                                     const int *__restrict__ dl, const int *__restrict__ w,
                                                     const double *__restrict__ coef, int stride,
                                                     const double *__restrict__ buf, int nrecv) {
  const int gid = blockIdx.x * TPB + threadIdx.x;
  if (gid >= NV * nrecv) return;
  const int v = gid / nrecv, r = gid - v * nrecv;
  const double lr = buf[gid];
  if (lr == 0.0) return;
  const int b = db[r];
  const int ni = t.ni[b], n = t.nn[b];
  const int w1 = w[3 * b], w2 = w[3 * b + 1];
  const double *c = coef + (size_t)r * stride;
  T *lam = t.lam[b] + (size_t)v * n;
  int q = 0;
  for (int b2 = 0; b2 < w2; b2++)
    for (int b1 = 0; b1 < w1; b1++, q++) {
      const int l1 = dl[r] + b1 + b2 * ni;
      if (l1 >= 0 && l1 < n) atomicAdd(&lam[l1], (T)(c[q] * lr));
    }
}

struct AdjBcArgs {
  int type, dir, end;
  int i0, i1, j0, j1;   // face box (collapsed along dir)
  int ni, nj;
  double neu[9];        // closure row 0 of the FD operator
  int sb;
};

// Transpose of one BC face (bc::apply_BC, boundary_condition.cpp:46-209):
// at a face point that is not a hole, the variables a Neumann closure
// (bc:348-444) sets hand their adjoint to the points along the normal
// (weights -neu[s] / neu[0]); wall-slip velocities (bc:448-494) take the
// transposed 2 x 2 map J Minv Z M; dirichlet_allzero and a centerline's
// normal velocity (bc:498-545) pass nothing on.  Points of one face reach
// distinct points along their normals, so no two threads touch one value.
template <typename T>
__global__ void __launch_bounds__(TPB) k_adj_bc_face(T *__restrict__ lam, const double *__restrict__ met,
                                                     const double *__restrict__ jac,
                                                     const int8_t *__restrict__ iblank, AdjBcArgs a) {
  const int fw = a.i1 - a.i0 + 1, fh = a.j1 - a.j0 + 1;
  const int q = blockIdx.x * TPB + threadIdx.x;
  if (q >= fw * fh) return;
  const int i = a.i0 + q % fw, j = a.j0 + q / fw;
  const int n = a.ni * a.nj;
  const int p = j * a.ni + i;
  if (iblank && iblank[p] == BLANKED) return;
  const int mf = a.dir == 0 ? 1 : a.ni;
  const int c = a.dir == 0 ? i : j, len = a.dir == 0 ? a.ni : a.nj;
  const int sg = a.end == 0 ? 1 : -1;
  double lv[NV];
  for (int v = 0; v < NV; v++) lv[v] = (double)lam[(size_t)v * n + p];
  bool neu[NV] = {false, false, false, false, false};
  double keep[NV] = {0.0, 0.0, 0.0, 0.0, 0.0};  // adjoint left at the face point
  switch (a.type) {
    case LEE_BC_NEUMANN:
      for (int v = 0; v < NV; v++) neu[v] = true;
      break;
    case LEE_BC_WALL_SLIP_KINEMATIC: {
      neu[IS] = neu[IP] = true;
      const double m00 = met[p], m01 = met[(size_t)n + p], m10 = met[(size_t)2 * n + p], m11 = met[(size_t)3 * n + p];
      const double J = jac[p];
      // forward: k = M u, k[dir] = 0, u' = J Minv k with Minv = [[m11, -m01], [-m10, m00]]
      double g0 = J * (m11 * lv[IUX] - m10 * lv[IUY]);
      double g1 = J * (-m01 * lv[IUX] + m00 * lv[IUY]);
      if (a.dir == 0) g0 = 0.0; else g1 = 0.0;
      keep[IUX] = m00 * g0 + m10 * g1;
      keep[IUY] = m01 * g0 + m11 * g1;
      keep[IUZ] = lv[IUZ];
      break;
    }
    case LEE_BC_CENTERLINE_CART_NORM2X:
    case LEE_BC_CENTERLINE_CART_NORM2Y:
    case LEE_BC_CENTERLINE_CART_NORM2Z:
      for (int v = 0; v < NV; v++) neu[v] = true;
      neu[IUX + (a.type - LEE_BC_CENTERLINE_CART_NORM2X)] = false;
      break;
    case LEE_BC_CENTERLINE_AXISYM:  // u_r = u_y' set to 0 on the axis (bc:498-545)
      for (int v = 0; v < NV; v++) neu[v] = true;
      neu[IUY] = false;
      break;
    default:  // dirichlet_allzero, and dirichlet_harmonicwave (its data do not depend on the state)
      break;
  }
  for (int v = 0; v < NV; v++) lam[(size_t)v * n + p] = (T)keep[v];
  for (int v = 0; v < NV; v++) {
    if (!neu[v] || lv[v] == 0.0) continue;
    for (int s = 1; s < a.sb && s <= 8; s++) {
      const int cs = c + sg * s;
      if (cs < 0 || cs >= len) continue;
      T *t = &lam[(size_t)v * n + p + sg * s * mf];
      *t = (T)((double)*t - a.neu[s] / a.neu[0] * lv[v]);
    }
  }
}

}  // namespace

// ------------------------------------------------------------- launchers

template <typename T>
static hipError_t adj_stage_t(hipStream_t s, lee_handle *h, Block &b, const AdjStage &st) {
  AdjArgs<T> a{};
  a.ni = b.ni;
  a.nj = b.nj;
  a.ntx = (b.ni + ADJ_TX - 1) / ADJ_TX;
  a.nty = (b.nj + ADJ_TY - 1) / ADJ_TY;
  a.ntiles = a.ntx * a.nty;
  a.chunk = (a.ntiles + 7) / 8;
  T *const *L = sizeof(T) == 8 ? (T *const *)b.A64 : (T *const *)b.A32;
  auto buf = [&](int k) -> T * { return k < 0 ? nullptr : L[k]; };
  a.lacc = buf(st.lacc);
  a.lin = buf(st.lin);
  a.lyin = buf(st.lyin);
  a.lout = buf(st.lout);
  a.lyout = buf(st.lyout);
  a.mu = sizeof(T) == 8 ? (T *)b.amu64 : (T *)b.amu32;
  a.grad = st.grad ? b.agrad : nullptr;
  a.met = b.met;
  a.jac = b.jac;
  a.mean = b.mean;
  a.mgrad = b.mgrad;
  a.rhob = b.rhobar;
  a.u0 = b.umean[IUX];
  a.v0 = b.umean[IUY];
  a.gamma = h->cfg.gamma;
  a.gi = 1.0 / h->cfg.gamma;
  a.gp0 = h->cfg.gamma * b.umean[IP];
  a.rhob0 = std::pow(h->cfg.gamma * b.umean[IP], 1.0 / h->cfg.gamma) * std::exp(-b.umean[IS]);
  a.nz = 0;
  for (const auto &z : b.zones) {
    if (a.nz >= MAX_ZONES) break;
    ZoneT<T> &q = a.z[a.nz++];
    q.i0 = z.is[0];
    q.i1 = z.ie[0];
    q.j0 = z.is[1];
    q.j1 = z.ie[1];
    q.nzi = z.nz[0];
    q.sig = sizeof(T) == 8 ? (const T *)z.sigma64 : (const T *)z.sigma32;
  }
  a.hb = st.hb;
  a.ha = st.ha;
  a.src = st.src;
  a.iblank = b.iblank;
  a.code = b.code_fd;
  a.clean = b.clean_fd;
  if (h->cfg.axisym) {  // an axisymmetric block always has its coefficient fields
    const T *mc = sizeof(T) == 8 ? (const T *)b.mc64 : (const T *)b.mc32;
    a.rad = mc + (size_t)MC_R * b.n;
  }
  const dim3 grid(a.chunk * 8), block(ADJ_TX, ADJ_TY);
  const bool mf = !b.uniform_mean, ho = b.has_holes;
#define LEE_ADJ(MF, K, HO)                                                                     \
  do {                                                                                         \
    hipLaunchKernelGGL((k_adj_stage<T, MF, K, HO>), grid, block, 0, s, a);                     \
  } while (0)
#define LEE_ADJK(MF, HO)                                          \
  do {                                                            \
    if (st.kind == STAGE_FIRST) LEE_ADJ(MF, STAGE_FIRST, HO);     \
    else if (st.kind == STAGE_MID) LEE_ADJ(MF, STAGE_MID, HO);    \
    else LEE_ADJ(MF, STAGE_LAST, HO);                             \
  } while (0)
  if (mf && ho) LEE_ADJK(true, true);
  else if (mf) LEE_ADJK(true, false);
  else if (ho) LEE_ADJK(false, true);
  else LEE_ADJK(false, false);
#undef LEE_ADJK
#undef LEE_ADJ
  return hipGetLastError();
}

hipError_t adjoint_stage(hipStream_t s, lee_handle *h, Block &b, const AdjStage &st) {
  if (h->cfg.precision == LEE_FP32) return adj_stage_t<float>(s, h, b, st);
  return adj_stage_t<double>(s, h, b, st);
}

template <typename T>
static hipError_t adj_filter_t(hipStream_t s, lee_handle *h, Block &b, int src, int dst, bool with_mu) {
  AdjFilterArgs<T> a{};
  const int TY = sizeof(T) == 8 ? 4 : 8;
  a.ni = b.ni;
  a.nj = b.nj;
  a.ntx = (b.ni + FL_TX - 1) / FL_TX;
  a.nty = (b.nj + TY - 1) / TY;
  a.ntiles = a.ntx * a.nty;
  a.chunk = (a.ntiles + 7) / 8;
  T *const *L = sizeof(T) == 8 ? (T *const *)b.A64 : (T *const *)b.A32;
  a.src = L[src];
  a.dst = L[dst];
  a.mu = with_mu ? (sizeof(T) == 8 ? (const T *)b.amu64 : (const T *)b.amu32) : nullptr;
  a.mean = b.mean;
  a.rhob = b.rhobar;
  a.gi = 1.0 / h->cfg.gamma;
  // without a filter the step's output is the accumulator itself
  const double blend = h->cfg.filter_order > 0 ? h->cfg.filter_blend : 0.0;
  a.blend = (T)blend;
  a.rem = (T)(1.0 - blend);
  a.iblank = b.iblank;
  a.code = b.code_flt;
  a.clean = b.clean_flt;
  const dim3 grid(a.chunk * 8), block(64, 4);
  // without a filter there are no filter codes: the hole reset alone
  // (blend 0 takes the identity part only)
  const bool ho = b.has_holes;
  if (h->cfg.filter_order == 8) {
    if (ho) hipLaunchKernelGGL((k_adj_filter<T, 8, TY, true>), grid, block, 0, s, a);
    else hipLaunchKernelGGL((k_adj_filter<T, 8, TY, false>), grid, block, 0, s, a);
  } else {
    if (ho) hipLaunchKernelGGL((k_adj_filter<T, 4, TY, true>), grid, block, 0, s, a);
    else hipLaunchKernelGGL((k_adj_filter<T, 4, TY, false>), grid, block, 0, s, a);
  }
  return hipGetLastError();
}

hipError_t adjoint_filter(hipStream_t s, lee_handle *h, Block &b, int src, int dst, bool with_mu) {
  if (h->cfg.precision == LEE_FP32) return adj_filter_t<float>(s, h, b, src, dst, with_mu);
  return adj_filter_t<double>(s, h, b, src, dst, with_mu);
}

hipError_t adjoint_zero(hipStream_t s, lee_handle *h, Block &b, int buf) {
  const size_t cnt = (size_t)NV * b.n;
  if (h->cfg.precision == LEE_FP32) {
    float *p = buf < 0 ? b.amu32 : b.A32[buf];
    hipLaunchKernelGGL(k_fill_t<float>, dim3(nblk(buf < 0 ? b.n : cnt)), dim3(TPB), 0, s, p, buf < 0 ? (size_t)b.n : cnt);
  } else {
    double *p = buf < 0 ? b.amu64 : b.A64[buf];
    hipLaunchKernelGGL(k_fill_t<double>, dim3(nblk(buf < 0 ? b.n : cnt)), dim3(TPB), 0, s, p, buf < 0 ? (size_t)b.n : cnt);
  }
  return hipGetLastError();
}

hipError_t adjoint_add_rt_mu(hipStream_t s, lee_handle *h, Block &b, int buf) {
  if (h->cfg.precision == LEE_FP32)
    hipLaunchKernelGGL(k_add_rt_mu<float>, dim3(nblk(b.n)), dim3(TPB), 0, s, b.A32[buf], b.amu32, b.mean, b.rhobar,
                       1.0 / h->cfg.gamma, b.n);
  else
    hipLaunchKernelGGL(k_add_rt_mu<double>, dim3(nblk(b.n)), dim3(TPB), 0, s, b.A64[buf], b.amu64, b.mean, b.rhobar,
                       1.0 / h->cfg.gamma, b.n);
  return hipGetLastError();
}

hipError_t adjoint_zero_grad(hipStream_t s, Block &b) {
  hipLaunchKernelGGL(k_fill_t<double>, dim3(nblk(b.n)), dim3(TPB), 0, s, b.agrad, (size_t)b.n);
  return hipGetLastError();
}

template <typename T>
static hipError_t adj_boundary_t(hipStream_t s, lee_handle *h, int buf) {
  const Overset &o = h->ov;
  if (o.nrecv > 0) {
    AdjOvTables<T> t{};
    for (int ib = 0; ib < h->nblk; ib++) {
      t.lam[ib] = sizeof(T) == 8 ? (T *)h->b[ib].A64[buf] : (T *)h->b[ib].A32[buf];
      t.ni[ib] = h->b[ib].ni;
      t.nn[ib] = h->b[ib].n;
    }
    const unsigned g = nblk((size_t)NV * o.nrecv);
    hipLaunchKernelGGL(k_adj_ov_take<T>, dim3(g), dim3(TPB), 0, s, t, o.rb, o.rl, o.buf, o.nrecv);
    hipLaunchKernelGGL(k_adj_ov_give<T>, dim3(g), dim3(TPB), 0, s, t, o.db, o.dl, o.w, o.coef, o.stride, o.buf,
                       o.nrecv);
  }
  for (int ib = 0; ib < h->nblk; ib++) {
    Block &b = h->b[ib];
    T *lam = sizeof(T) == 8 ? (T *)b.A64[buf] : (T *)b.A32[buf];
    for (int k = (int)b.faces.size() - 1; k >= 0; k--) {
      const BcFace &f = b.faces[k];
      AdjBcArgs a{};
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
      for (int q = 0; q < 9; q++) a.neu[q] = h->fd.bnd[0][q];
      const size_t cnt = (size_t)(a.i1 - a.i0 + 1) * (a.j1 - a.j0 + 1);
      hipLaunchKernelGGL(k_adj_bc_face<T>, dim3(nblk(cnt)), dim3(TPB), 0, s, lam, b.met, b.jac,
                         b.has_holes ? b.iblank : nullptr, a);
    }
  }
  return hipGetLastError();
}

hipError_t adjoint_boundary(hipStream_t s, lee_handle *h, int buf) {
  if (h->cfg.precision == LEE_FP32) return adj_boundary_t<float>(s, h, buf);
  return adj_boundary_t<double>(s, h, buf);
}

hipError_t observer_energy(hipStream_t s, lee_handle *h, Block &b, double *out) {
  if (b.nobs == 0) return hipSuccess;
  if (h->cfg.precision == LEE_FP32)
    hipLaunchKernelGGL(k_obs_energy<float>, dim3(1), dim3(1024), 0, s, b.Y32[0], b.obs_l, b.obs_w, b.nobs, b.n, out);
  else
    hipLaunchKernelGGL(k_obs_energy<double>, dim3(1), dim3(1024), 0, s, b.Y64[0], b.obs_l, b.obs_w, b.nobs, b.n, out);
  return hipGetLastError();
}

hipError_t observer_gather(hipStream_t s, lee_handle *h, Block &b, double *out) {
  if (b.nobs == 0) return hipSuccess;
  if (h->cfg.precision == LEE_FP32)
    hipLaunchKernelGGL(k_obs_gather<float>, dim3(nblk(b.nobs)), dim3(TPB), 0, s, b.Y32[0], b.obs_l, b.nobs, b.n, out);
  else
    hipLaunchKernelGGL(k_obs_gather<double>, dim3(nblk(b.nobs)), dim3(TPB), 0, s, b.Y64[0], b.obs_l, b.nobs, b.n, out);
  return hipGetLastError();
}

hipError_t observer_seed(hipStream_t s, lee_handle *h, Block &b, int buf, const double *samp, double scale) {
  if (b.nobs == 0) return hipSuccess;
  if (h->cfg.precision == LEE_FP32)
    hipLaunchKernelGGL(k_obs_seed<float>, dim3(nblk(b.nobs)), dim3(TPB), 0, s, b.A32[buf], b.obs_l, b.obs_w, samp,
                       b.nobs, b.n, scale);
  else
    hipLaunchKernelGGL(k_obs_seed<double>, dim3(nblk(b.nobs)), dim3(TPB), 0, s, b.A64[buf], b.obs_l, b.obs_w, samp,
                       b.nobs, b.n, scale);
  return hipGetLastError();
}

}  // namespace lee
