// Discrete adjoint of the 3-D fused time advance (no reference counterpart).
//
// Same transposition as the 2-D adjoint (lee_adjoint.hip): per reversed RK
// stage, kappa = b_i h lambda_acc + a_i h lambda_in, then
// lambda_u = sum_l D_l^T F_l + point-local terms, with the flux fields
// F_l,v = J sum_d m[l][d] A_d,v built from the coefficients A_d,v of
// d/dx_d in each right-hand-side term:
//   s:    A_d = -u_d kappa_s
//   u_i:  A_d = -u_d kappa_ui - delta_id gamma p kappa_p
//   p:    A_d = -u_d kappa_p - kappa_ud / rho
// The stage kernel marches a 32 x 8 column tile through z like the forward
// one: the xi fluxes of each plane with two halo columns a side and the eta
// fluxes with two halo rows a side are staged in LDS, the zeta fluxes of the
// thread's own column sit in a 5-plane register window.  The transposed filter is rem I + blend F_xi^T F_eta^T
// F_zeta^T: a zeta^T column pass into scratch, then the eta^T, xi^T plane
// pass with the blend and R^T mu.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>

#include "lee_device.h"
#include "lee_internal.h"

namespace lee {

namespace {

constexpr int A3_TX = 32, A3_TY = 8;  // points of a stage tile
constexpr int A3_ZC = 16;      // most planes per chunk of the zeta^T filter pass (at least 4, z_chunk)
// Planes per workgroup of the adjoint stage (z_chunk_rounds): the start of a
// column costs about two planes; up to 10, past which little is shared.
// Whole reverse step with 4 planes whatever the block and with this rule,
// FP32 / FP64: 112 x 96 x 80 640 / 960 -> 516 / 906 us (5 and 8 planes),
// 144 x 120 x 112 1389 / 2515 -> 1332 / 2376 (6 and 6), 256 x 200 x 256 7770 /
// 13339 -> 7402 / 12877; 48 x 40 x 32 208 / 275 -> 147 / 185 (1).
constexpr int ADJ_Z_CHUNK = 10;
constexpr double ADJ_Z_START = 2.0;

inline unsigned nba(size_t n) { return (unsigned)((n + TPB - 1) / TPB); }

template <typename T>
struct Zone3A {
  int i0, i1, j0, j1, k0, k1, nzi, nzj;
  const T *sig;
};

template <typename T>
struct Adj3Args {
  int ni, nj, nk, ntx, nty, nzc, zc;
  const T *lacc, *lin, *lyin;
  T *lout, *lyout, *mu;
  double *grad;
  const double *met, *jac;
  const T *mc;               // MC3_COUNT coefficient fields (non-uniform mean)
  unsigned varies;           // and which of them are not constant
  double u0, v0, w0, gp0, rhob0, gamma;
  int nz;
  Zone3A<T> z[MAX_ZONES];
  double hb, ha, src;
};

// kappa and the mean flow at a point, and from them the flux vector of one
// direction with its metrics m: F_l = -J (U_l kappa + ...) with the
// contravariant velocity U_l = m . ubar.
struct AdjPoint3 {
  double kap[5], ub[3], c, irb, J;  // c = gamma p kappa_p; J the negative Jacobian
};

template <typename T, bool MEANF, int KIND>
__device__ __forceinline__ AdjPoint3 adj_point3(const Adj3Args<T> &a, size_t p, size_t n) {
  AdjPoint3 q;
  const T hb = (T)a.hb, ha = (T)a.ha;
#pragma unroll
  for (int v = 0; v < 5; v++) {
    T kv = hb * a.lacc[v * n + p];
    if (KIND != STAGE_LAST && a.lin) kv += ha * a.lin[v * n + p];
    q.kap[v] = kv;
  }
  double gp = a.gp0;
  q.ub[0] = a.u0;
  q.ub[1] = a.v0;
  q.ub[2] = a.w0;
  if (MEANF) {
    q.ub[0] = mean_field3(a.mc, a.varies, MC3_U, n, p);
    q.ub[1] = mean_field3(a.mc, a.varies, MC3_V, n, p);
    q.ub[2] = mean_field3(a.mc, a.varies, MC3_W, n, p);
    gp = mean_field3(a.mc, a.varies, MC3_GP, n, p);
    q.irb = mean_field3(a.mc, a.varies, MC3_IRB, n, p);
  } else {
    q.irb = 1.0 / a.rhob0;
  }
  q.c = gp * q.kap[IP];
  q.J = -a.jac[p];
  return q;
}

template <typename T>
__device__ __forceinline__ void adj_dir3(const AdjPoint3 &q, double m0, double m1, double m2, T (&F)[5]) {
  const double U = m0 * q.ub[0] + m1 * q.ub[1] + m2 * q.ub[2], m[3] = {m0, m1, m2};
  F[IS] = (T)(U * q.kap[IS] * q.J);
#pragma unroll
  for (int i = 0; i < 3; i++) F[IUX + i] = (T)((U * q.kap[IUX + i] + m[i] * q.c) * q.J);
  F[IP] = (T)((U * q.kap[IP] + (m0 * q.kap[IUX] + m1 * q.kap[IUY] + m2 * q.kap[IUZ]) * q.irb) * q.J);
}

// What bounds it: the wait for its operands (three quarters of a wave's time);
// a flux evaluation is some 75 FP64 operations.  Tiles of 32 x 8 points hold
// their own fluxes in registers from the plane that first needs them, so a
// point is evaluated once and its halo lanes (160 beside 256 points, one
// direction each) once: 1.2 evaluations a point.  A 64 x 4 tile that
// evaluated plane k with its whole halo again took 3.1.  Whole reverse step
// before, FP32 / FP64: 112 x 96 x 80 537 / 1039 -> 504 / 863 us, 144 x 120 x
// 112 1567 / 2935 -> 1284 / 2263, 256 x 200 x 256 7816 / 14353 -> 7102 / 12198.
template <typename T, bool MEANF, int KIND>
__global__ void __launch_bounds__(TPB) k_adj_stage3d(Adj3Args<T> a) {
  constexpr int H = ST_H;
  __shared__ T SX[5][A3_TY][A3_TX + 2 * H];  // xi fluxes of plane k with their halo columns
  __shared__ T SE[5][A3_TY + 2 * H][A3_TX];  // eta fluxes with their halo rows
  // XCD-banded tiles within each z chunk, as the forward stage
  const int ntl = a.ntx * a.nty;
  const int tile = xcd_tile(blockIdx.x, (ntl + 7) / 8);
  if (tile >= ntl) return;
  const int tx = threadIdx.x, ty = threadIdx.y, tid = ty * A3_TX + tx;
  const int i0 = (tile % a.ntx) * A3_TX, j0 = (tile / a.ntx) * A3_TY;
  const int k0 = blockIdx.y * a.zc, k1 = min(k0 + a.zc, a.nk);
  const int ni = a.ni, nj = a.nj, nk = a.nk;
  const size_t plane = (size_t)ni * nj, n = plane * nk;
  const int gi = i0 + tx, gj = j0 + ty;
  const bool own = gi < ni && gj < nj;
  const size_t col = own ? (size_t)gj * ni + gi : 0;
  const RowT5<T> rx = row_t5<T>(gi, ni), ry = row_t5<T>(gj, nj);
  const unsigned zmask = zones_meeting3(a.z, a.nz, i0, i0 + A3_TX - 1, j0, j0 + A3_TY - 1, k0, k1 - 1);
  // fluxes of the own column: zeta of planes k - 2 .. k + 2, xi and eta of
  // k .. k + 2 (each point of the tile is evaluated once per chunk)
  T wz[5][5], wx[5][3], we[5][3];
  auto column = [&](int kk, int q) {
    T f[3][5];
    if (kk >= 0 && kk < nk) {  // uniform
      const size_t p = (size_t)kk * plane + col;
      const AdjPoint3 pt = adj_point3<T, MEANF, KIND>(a, p, n);
#pragma unroll
      for (int l = 0; l < 3; l++)
        adj_dir3<T>(pt, a.met[(size_t)(3 * l) * n + p], a.met[(size_t)(3 * l + 1) * n + p],
                    a.met[(size_t)(3 * l + 2) * n + p], f[l]);
    }
    const bool ok = own && kk >= 0 && kk < nk;
#pragma unroll
    for (int v = 0; v < 5; v++) {
      wz[v][q] = ok ? f[2][v] : (T)0;
      if (q >= 2) {
        wx[v][q - 2] = ok ? f[0][v] : (T)0;
        we[v][q - 2] = ok ? f[1][v] : (T)0;
      }
    }
  };
#pragma unroll
  for (int q = 0; q < 4; q++) column(k0 - 2 + q, q);
  // the halo of a plane, a point and direction per lane: four rows beside the
  // tile (eta fluxes, waves 0 and 1) and four columns (xi, half of wave 2)
  static_assert(A3_TX == 32 && A3_TY == 8 && TPB == 256, "halo lanes");
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), hs = (tid >> 2) & 7, hq = wave < 2 ? tid >> 5 : tid & 3;
  const int hr = wave < 2 ? (hq < 2 ? hq : hq + A3_TY) : hs;       // row of SE or SX
  const int hc = wave < 2 ? tx : (hq < 2 ? hq : hq + A3_TX);       // and column
  const int hj = wave < 2 ? j0 - H + hr : j0 + hr, hi = wave < 2 ? i0 + hc : i0 - H + hc;
  const bool hon = tid < 160, hok = hj >= 0 && hj < nj && hi >= 0 && hi < ni;
  const size_t hp = (size_t)min(max(hj, 0), nj - 1) * ni + min(max(hi, 0), ni - 1);
  const double *hm = a.met + (wave < 2 ? (size_t)3 * n : 0);
  for (int k = k0; k < k1; k++) {
    column(k + 2, 4);
    if (hon) {
      const size_t p = (size_t)k * plane + hp;
      const AdjPoint3 pt = adj_point3<T, MEANF, KIND>(a, p, n);
      T f[5];
      adj_dir3<T>(pt, hm[p], hm[n + p], hm[2 * n + p], f);
#pragma unroll
      for (int v = 0; v < 5; v++) {
        T *to = wave < 2 ? &SE[v][hr][hc] : &SX[v][hr][hc];
        *to = hok ? f[v] : (T)0;
      }
    }
#pragma unroll
    for (int v = 0; v < 5; v++) {
      SX[v][ty][tx + H] = wx[v][0];
      SE[v][ty + H][tx] = we[v][0];
    }
    // the own point's operands, requested before the barrier
    const size_t p = (size_t)k * plane + col;
    T lacc[5], lin[5], lyin[5], mcv[MC3_COUNT];
#pragma unroll
    for (int v = 0; v < 5; v++) {
      lacc[v] = a.lacc[v * n + p];
      lin[v] = (KIND != STAGE_LAST && a.lin) ? a.lin[v * n + p] : (T)0;
      lyin[v] = KIND != STAGE_LAST && a.lyin ? a.lyin[v * n + p] : (T)0;
    }
    if (MEANF) {
#pragma unroll
      for (int f = 0; f < MC3_COUNT; f++)
        mcv[f] = f == MC3_GP || (KIND == STAGE_FIRST && f >= MC3_RP) ? (T)0 : mean_field3(a.mc, a.varies, f, n, p);
    }
    __syncthreads();
    if (own) {
      const RowT5<T> rz = row_t5<T>(k, nk);  // uniform
      T lam[5];
#pragma unroll
      for (int v = 0; v < 5; v++) {
        lam[v] = row_t5_sum<T>(rx, &SX[v][ty][tx + H], 1);
        lam[v] += row_t5_sum<T>(ry, &SE[v][ty + H][tx], A3_TX);
        lam[v] += row_t5_sum<T>(rz, &wz[v][2], 1);
      }
      T kap[5];
#pragma unroll
      for (int v = 0; v < 5; v++) {
        T kv = (T)a.hb * lacc[v];
        if (KIND != STAGE_LAST && a.lin) kv += (T)a.ha * lin[v];
        kap[v] = kv;
      }
      for (unsigned zm = zmask; zm; zm &= zm - 1) {
        const Zone3A<T> &zz = a.z[__builtin_ctz(zm)];
        if (gi >= zz.i0 && gi <= zz.i1 && gj >= zz.j0 && gj <= zz.j1 && k >= zz.k0 && k <= zz.k1) {
          const T sg = zz.sig[((size_t)(k - zz.k0) * zz.nzj + (gj - zz.j0)) * zz.nzi + (gi - zz.i0)];
#pragma unroll
          for (int v = 0; v < 5; v++) lam[v] += -sg * kap[v];
        }
      }
      T mur = 0;
      if (MEANF) {
        auto mc = [&](int f) { return mcv[f]; };
        auto G = [&](int v, int d) { return mc(MC3_G + 3 * v + d); };
        const T ub[3] = {mc(MC3_U), mc(MC3_V), mc(MC3_W)};
        const T g = (T)a.gamma, irb = mc(MC3_IRB);
#pragma unroll
        for (int d = 0; d < 3; d++) {
          T acc = G(IS, d) * kap[IS];
#pragma unroll
          for (int i = 0; i < 3; i++) acc += G(IUX + i, d) * kap[IUX + i];
          acc += G(IP, d) * kap[IP];
          lam[IUX + d] -= acc;
        }
        T div = 0;
#pragma unroll
        for (int d = 0; d < 3; d++) div += G(IUX + d, d);
        lam[IP] -= g * div * kap[IP];
        T mu = 0;
#pragma unroll
        for (int i = 0; i < 3; i++) {
          T s = 0;
#pragma unroll
          for (int d = 0; d < 3; d++) s += ub[d] * G(IUX + i, d);
          mu += s * kap[IUX + i];
        }
        mur = -(mu * irb);
        if (KIND != STAGE_FIRST) {
          lam[IS] += -(mc(MC3_RB) * mur);
          lam[IP] += mc(MC3_RP) * mur;
        }
      }
      if (a.grad) a.grad[p] += a.src * (double)kap[IP];
      if (KIND == STAGE_FIRST) {
#pragma unroll
        for (int v = 0; v < 5; v++) {
          T out = lam[v] + lacc[v] + lin[v];
          if (a.lyin) out += lyin[v];
          a.lout[v * n + p] = out;
        }
        if (MEANF) a.mu[p] = mur;
      } else {
#pragma unroll
        for (int v = 0; v < 5; v++) a.lout[v * n + p] = lam[v];
        if (a.lyout) {
#pragma unroll
          for (int v = 0; v < 5; v++) {
            T y = lin[v];
            if (a.lyin) y += lyin[v];
            a.lyout[v * n + p] = y;
          }
        }
      }
    }
    __syncthreads();
#pragma unroll
    for (int v = 0; v < 5; v++) {
#pragma unroll
      for (int q = 0; q < 4; q++) wz[v][q] = wz[v][q + 1];
#pragma unroll
      for (int q = 0; q < 2; q++) {
        wx[v][q] = wx[v][q + 1];
        we[v][q] = we[v][q + 1];
      }
    }
  }
}

// zeta^T column pass: tmp = F_zeta^T lam.
template <typename T, int ORDER>
__global__ void __launch_bounds__(TPB) k_adj_filter3d_z(const T *__restrict__ lam, T *__restrict__ tmp, int ni,
                                                        int nj, int nk, int zc) {
  constexpr int H = ORDER / 2;
  const size_t plane = (size_t)ni * nj, n = plane * nk;
  const size_t col = (size_t)blockIdx.x * TPB + threadIdx.x;
  if (col >= plane) return;
  const int k0 = blockIdx.y * zc, k1 = min(k0 + zc, nk);
  T w[5][2 * H + 1];
#pragma unroll
  for (int q = 0; q < 2 * H; q++) {
    const int kk = k0 - H + q;
    const bool ok = kk >= 0 && kk < nk;
#pragma unroll
    for (int v = 0; v < 5; v++) w[v][q] = ok ? lam[v * n + (size_t)kk * plane + col] : (T)0;
  }
  // four planes per pass, their window planes requested together (clamped
  // plane index, zeros selected afterwards)
  auto plane_out = [&](int k, const T (&wn)[5]) {
#pragma unroll
    for (int v = 0; v < 5; v++) w[v][2 * H] = wn[v];
    if (k >= 2 * H && k <= nk - 1 - 2 * H) {  // uniform; symmetric interior rows: F^T = F
#pragma unroll
      for (int v = 0; v < 5; v++) tmp[v * n + (size_t)k * plane + col] = filter_row<T, ORDER>(&w[v][H], 1, CODE_INTERIOR);
    } else {
      const FltRowT<T, ORDER> r = flt_row_t<T, ORDER>(k, nk);
#pragma unroll
      for (int v = 0; v < 5; v++) tmp[v * n + (size_t)k * plane + col] = flt_row_t_sum<T, ORDER>(r, &w[v][H], 1);
    }
#pragma unroll
    for (int v = 0; v < 5; v++)
#pragma unroll
      for (int q = 0; q < 2 * H; q++) w[v][q] = w[v][q + 1];
  };
  int k = k0;
  for (; k + 4 <= k1; k += 4) {
    T wn[4][5];
#pragma unroll
    for (int u = 0; u < 4; u++) {
      const int kk = k + u + H;
      const size_t pc = (size_t)min(kk, nk - 1) * plane + col;
#pragma unroll
      for (int v = 0; v < 5; v++) {
        const T t = lam[v * n + pc];
        wn[u][v] = kk < nk ? t : (T)0;
      }
    }
#pragma unroll
    for (int u = 0; u < 4; u++) plane_out(k + u, wn[u]);
  }
  for (; k < k1; k++) {
    const int kk = k + H;
    T wn[5];
#pragma unroll
    for (int v = 0; v < 5; v++) wn[v] = kk < nk ? lam[v * n + (size_t)kk * plane + col] : (T)0;
    plane_out(k, wn);
  }
}

template <typename T>
struct AdjF3Args {
  int ni, nj, nk, ntx, nty, ntiles;
  const T *tmp;    // zeta^T-filtered adjoint
  const T *orig;   // adjoint of the filtered state
  T *dst;
  const T *mu;     // null: none
  const T *mc;
  T rem, blend;
};

// eta^T then xi^T sweeps of plane blockIdx.y, blend and R^T mu; region,
// middle sweep and closure rows as in the 2-D form (k_adj_filter).
// 112 x 96 x 80 FP32: 66 -> 19 us.
template <typename T, int ORDER, int TY>
__global__ void __launch_bounds__(TPB) k_adj_filter3d_plane(AdjF3Args<T> a) {
  constexpr int NR = TY + 2 * FL_H, NC = FL_TX + 2 * FL_H;
  __shared__ T in[5][NR][NC];
  __shared__ T mid[5][TY][NC];
  const int tile = xcd_tile(blockIdx.x, (a.ntiles + 7) / 8);  // XCD-banded tiles of each plane
  if (tile >= a.ntiles) return;
  const int k = blockIdx.y;
  const int tx = threadIdx.x, ty = threadIdx.y, tid = ty * 64 + tx;
  const int i0 = (tile % a.ntx) * FL_TX, j0 = (tile / a.ntx) * TY;
  const int ni = a.ni, nj = a.nj;
  const size_t plane = (size_t)ni * nj, n = plane * a.nk, off = (size_t)k * plane;
  const bool inx = i0 >= 2 * FL_H && i0 + FL_TX + 2 * FL_H <= ni;
  const bool iny = j0 >= 2 * FL_H && j0 + TY + 2 * FL_H <= nj;
  // points outside the block read the nearest one inside and store 0
  auto load = [&](int idx) {
    const int r = idx / NC, c = idx - r * NC;
    const int gj = j0 - FL_H + r, gi = i0 - FL_H + c;
    const size_t p = off + (size_t)min(max(gj, 0), nj - 1) * ni + min(max(gi, 0), ni - 1);
    const bool ok = gj >= 0 && gj < nj && gi >= 0 && gi < ni;
#pragma unroll
    for (int v = 0; v < 5; v++) {
      const T x = a.tmp[v * n + p];
      in[v][r][c] = ok ? x : (T)0;
    }
  };
#pragma unroll
  for (int q = 0; q < NR * NC / TPB; q++) load(tid + q * TPB);
  if (tid + NR * NC / TPB * TPB < NR * NC) load(tid + NR * NC / TPB * TPB);
  // the points' own operands, requested before the barriers
  const int gi = i0 + tx;
  T orig[TY / 4][5], mu[TY / 4], mrb[TY / 4], mrp[TY / 4];
#pragma unroll
  for (int kr = 0; kr < TY / 4; kr++) {
    const size_t p = off + (size_t)min(j0 + ty + 4 * kr, nj - 1) * ni + min(gi, ni - 1);
#pragma unroll
    for (int v = 0; v < 5; v++) orig[kr][v] = a.orig[v * n + p];
    mu[kr] = a.mu ? a.mu[p] : (T)0;
    mrb[kr] = a.mu ? a.mc[MC3_RB * n + p] : (T)0;
    mrp[kr] = a.mu ? a.mc[MC3_RP * n + p] : (T)0;
  }
  __syncthreads();
  auto eta = [&](int idx) {
    const int r = idx / NC, c = idx - r * NC;
    if (iny) {
#pragma unroll
      for (int v = 0; v < 5; v++) mid[v][r][c] = filter_row<T, ORDER>(&in[v][r + FL_H][c], NC, CODE_INTERIOR);
    } else {
      const FltRowT<T, ORDER> w = flt_row_t<T, ORDER>(j0 + r, nj);
#pragma unroll
      for (int v = 0; v < 5; v++) mid[v][r][c] = flt_row_t_sum<T, ORDER>(w, &in[v][r + FL_H][c], NC);
    }
  };
#pragma unroll
  for (int q = 0; q < TY * NC / TPB; q++) eta(tid + q * TPB);
  if (tid + TY * NC / TPB * TPB < TY * NC) eta(tid + TY * NC / TPB * TPB);
  __syncthreads();
  FltRowT<T, ORDER> wx{};
  if (!inx) wx = flt_row_t<T, ORDER>(gi, ni);
#pragma unroll
  for (int kr = 0; kr < TY / 4; kr++) {
    const int r = ty + 4 * kr;
    const int gj = j0 + r;
    if (gi >= ni || gj >= nj) continue;
    const size_t p = off + (size_t)gj * ni + gi;
    T out[5];
#pragma unroll
    for (int v = 0; v < 5; v++) {
      const T *m = &mid[v][r][tx + FL_H];
      const T f = inx ? filter_row<T, ORDER>(m, 1, CODE_INTERIOR) : flt_row_t_sum<T, ORDER>(wx, m, 1);
      out[v] = a.rem * orig[kr][v] + a.blend * f;
    }
    if (a.mu) {
      out[IS] += -(mrb[kr] * mu[kr]);
      out[IP] += mrp[kr] * mu[kr];
    }
#pragma unroll
    for (int v = 0; v < 5; v++) a.dst[v * n + p] = out[v];
  }
}

template <typename T>
__global__ void __launch_bounds__(TPB) k_add_rt_mu3(T *__restrict__ lam, const T *__restrict__ mu,
                                                    const T *__restrict__ mc, size_t n) {
  const size_t p = (size_t)blockIdx.x * TPB + threadIdx.x;
  if (p >= n) return;
  const T m = mu[p];
  lam[IS * n + p] += -(mc[MC3_RB * n + p] * m);
  lam[IP * n + p] += mc[MC3_RP * n + p] * m;
}

}  // namespace

// ------------------------------------------------------------- launchers

template <typename T>
static hipError_t adj_stage3d_t(hipStream_t s, lee_handle *h, Block &b, const AdjStage &st) {
  Adj3Args<T> a{};
  a.ni = b.ni;
  a.nj = b.nj;
  a.nk = b.nk;
  a.ntx = (b.ni + A3_TX - 1) / A3_TX;
  a.nty = (b.nj + A3_TY - 1) / A3_TY;
  // resident workgroups a CU: what the registers of the instances leave (197 to
  // 244 in 64 bits, 130 to 140 and, with a uniform mean, 117 to 125 in 32); a
  // compiler that takes others changes the chunk, and so the time, not the result
  a.zc = z_chunk_rounds((a.ntx * a.nty + 7) / 8 * 8, b.nk, b.cus * (sizeof(T) == 8 ? 2 : b.uniform_mean ? 4 : 3),
                        ADJ_Z_START, ADJ_Z_CHUNK);
  a.nzc = (b.nk + a.zc - 1) / a.zc;
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
  a.mc = sizeof(T) == 8 ? (const T *)b.mc64 : (const T *)b.mc32;
  a.varies = b.mc_varies;
  a.u0 = b.umean[IUX];
  a.v0 = b.umean[IUY];
  a.w0 = b.umean[IUZ];
  a.gamma = h->cfg.gamma;
  a.gp0 = h->cfg.gamma * b.umean[IP];
  a.rhob0 = std::pow(h->cfg.gamma * b.umean[IP], 1.0 / h->cfg.gamma) * std::exp(-b.umean[IS]);
  a.nz = 0;
  for (const auto &z : b.zones) {
    if (a.nz >= MAX_ZONES) break;
    Zone3A<T> &q = a.z[a.nz++];
    q.i0 = z.is[0];
    q.i1 = z.ie[0];
    q.j0 = z.is[1];
    q.j1 = z.ie[1];
    q.k0 = z.is[2];
    q.k1 = z.ie[2];
    q.nzi = z.nz[0];
    q.nzj = z.nz[1];
    q.sig = sizeof(T) == 8 ? (const T *)z.sigma64 : (const T *)z.sigma32;
  }
  a.hb = st.hb;
  a.ha = st.ha;
  a.src = st.src;
  const dim3 grid((a.ntx * a.nty + 7) / 8 * 8, a.nzc), block(A3_TX, A3_TY);
  const bool mf = !b.uniform_mean;
#define LEE_A3(MF)                                                                                            \
  do {                                                                                                        \
    if (st.kind == STAGE_FIRST) hipLaunchKernelGGL((k_adj_stage3d<T, MF, STAGE_FIRST>), grid, block, 0, s, a); \
    else if (st.kind == STAGE_MID) hipLaunchKernelGGL((k_adj_stage3d<T, MF, STAGE_MID>), grid, block, 0, s, a); \
    else hipLaunchKernelGGL((k_adj_stage3d<T, MF, STAGE_LAST>), grid, block, 0, s, a);                         \
  } while (0)
  if (mf) LEE_A3(true);
  else LEE_A3(false);
#undef LEE_A3
  return hipGetLastError();
}

hipError_t adjoint_stage3d(hipStream_t s, lee_handle *h, Block &b, const AdjStage &st) {
  if (h->cfg.precision == LEE_FP32) return adj_stage3d_t<float>(s, h, b, st);
  return adj_stage3d_t<double>(s, h, b, st);
}

// dst = rem src + blend F_xi^T F_eta^T F_zeta^T src (+ R^T mu); scratch
// holds the zeta^T pass (all buffers index Block::A).
template <typename T>
static hipError_t adj_filter3d_t(hipStream_t s, lee_handle *h, Block &b, int src, int dst, int scratch,
                                 bool with_mu) {
  T *const *L = sizeof(T) == 8 ? (T *const *)b.A64 : (T *const *)b.A32;
  const size_t plane = (size_t)b.ni * b.nj;
  const bool o8 = h->cfg.filter_order == 8;
  const int zc = std::max(4, z_chunk((int)nba(plane), b.nk, A3_ZC, b.cus));
  const dim3 gz(nba(plane), (b.nk + zc - 1) / zc);
  if (o8) hipLaunchKernelGGL((k_adj_filter3d_z<T, 8>), gz, dim3(TPB), 0, s, L[src], L[scratch], b.ni, b.nj, b.nk, zc);
  else hipLaunchKernelGGL((k_adj_filter3d_z<T, 4>), gz, dim3(TPB), 0, s, L[src], L[scratch], b.ni, b.nj, b.nk, zc);
  constexpr int TY = 4;
  AdjF3Args<T> a{};
  a.ni = b.ni;
  a.nj = b.nj;
  a.nk = b.nk;
  a.ntx = (b.ni + FL_TX - 1) / FL_TX;
  a.nty = (b.nj + TY - 1) / TY;
  a.ntiles = a.ntx * a.nty;
  a.tmp = L[scratch];
  a.orig = L[src];
  a.dst = L[dst];
  a.mu = with_mu ? (sizeof(T) == 8 ? (const T *)b.amu64 : (const T *)b.amu32) : nullptr;
  a.mc = sizeof(T) == 8 ? (const T *)b.mc64 : (const T *)b.mc32;
  const double blend = h->cfg.filter_order > 0 ? h->cfg.filter_blend : 0.0;
  a.blend = (T)blend;
  a.rem = (T)(1.0 - blend);
  const dim3 grid((a.ntiles + 7) / 8 * 8, b.nk), block(64, 4);
  if (o8) hipLaunchKernelGGL((k_adj_filter3d_plane<T, 8, TY>), grid, block, 0, s, a);
  else hipLaunchKernelGGL((k_adj_filter3d_plane<T, 4, TY>), grid, block, 0, s, a);
  return hipGetLastError();
}

hipError_t adjoint_filter3d(hipStream_t s, lee_handle *h, Block &b, int src, int dst, int scratch, bool with_mu) {
  if (h->cfg.precision == LEE_FP32) return adj_filter3d_t<float>(s, h, b, src, dst, scratch, with_mu);
  return adj_filter3d_t<double>(s, h, b, src, dst, scratch, with_mu);
}

hipError_t adjoint_add_rt_mu3(hipStream_t s, lee_handle *h, Block &b, int buf) {
  if (h->cfg.precision == LEE_FP32)
    hipLaunchKernelGGL(k_add_rt_mu3<float>, dim3(nba(b.n)), dim3(TPB), 0, s, b.A32[buf], b.amu32, b.mc32, (size_t)b.n);
  else
    hipLaunchKernelGGL(k_add_rt_mu3<double>, dim3(nba(b.n)), dim3(TPB), 0, s, b.A64[buf], b.amu64, b.mc64,
                       (size_t)b.n);
  return hipGetLastError();
}

}  // namespace lee
