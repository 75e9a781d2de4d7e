// The plain FP64 path of the LEE time advance for gfx950: floating-point
// contraction off and the reference's operation order at every point, so the
// GPU result equals the CPU reference bit for bit.  It is the drop-in FP64
// path and the yardstick of the fused path.
//
// An RK stage is one launch and the filter two.  Every operator of the
// reference writes its result to memory and the next one reads it back; a
// point's operations only ever combine its own operands, the row values of
// its neighbours and its own running sums, so one thread can carry a point
// through all of them in the reference's order and round every step alike.
// All global indices are bounds-checked against the block extents.
#include <hip/hip_runtime.h>

#include "lee_device.h"
#include "lee_internal.h"

namespace lee {

namespace {

// One row of the reference operator at point p (coordinate c along a line of
// length len, memory stride st), every coefficient included, left to right.
__device__ double plain_row(const OpTable &op, const double *f, int p, int c, int len, int st, int code) {
#pragma clang fp contract(off)
  double acc = 0.0;
  if (code == CODE_INTERIOR) {
    for (int s = -op.half; s <= op.half; s++) {
      const int q = c + s;
      if (q >= 0 && q < len) acc += op.st[s + op.half] * f[p + s * st];
    }
  } else if (code == CODE_ZERO) {
    acc = 0.0;
  } else if (code < CODE_LEFT + op.nb) {
    const int k = code - CODE_LEFT;
    for (int s = 0; s < op.sb; s++) {
      const int q = c - k + s;
      if (q >= 0 && q < len) acc += op.bnd[k][s] * f[p + (s - k) * st];
    }
  } else {
    const int k = code - CODE_LEFT - op.nb;
    for (int s = 0; s < op.sb; s++) {
      const int q = c + k - s;
      if (q >= 0 && q < len) acc += op.sign_right * op.bnd[k][s] * f[p + (k - s) * st];
    }
  }
  return acc;
}

// plain_row unrolled for the scheme at hand (HALF = op.half, 2 HALF - 1 =
// op.sb), every value of a row requested before the sums: a closure row read
// entry by entry exposes one memory latency per entry, and the edge tiles'
// chain of them set the time of a small block (filter sweeps 16 -> 5 us each
// at 201 x 201).  Interior rows lie at least nb >= half
// points from both ends of the line (plan_codes, default_code), so they need
// no range check; entries of a closure row outside the line are skipped.
template <int HALF>
__device__ __forceinline__ double plain_row_h(const OpTable &op, const double *f, int p, int c, int len, int st,
                                              int code) {
#pragma clang fp contract(off)
  double acc = 0.0;
  if (code == CODE_INTERIOR) {
    double v[2 * HALF + 1];
#pragma unroll
    for (int s = 0; s <= 2 * HALF; s++) v[s] = f[p + (s - HALF) * st];
#pragma unroll
    for (int s = 0; s <= 2 * HALF; s++) acc += op.st[s] * v[s];
  } else if (code != CODE_ZERO) {
    constexpr int SB = 2 * HALF - 1;
    const bool left = code < CODE_LEFT + op.nb;
    const int k = code - CODE_LEFT - (left ? 0 : op.nb), dir = left ? 1 : -1;
    const double sign = left ? 1.0 : op.sign_right;
    double v[SB], w[SB];
#pragma unroll
    for (int s = 0; s < SB; s++) {
      const int o = dir * (s - k);
      v[s] = f[p + (c + o >= 0 && c + o < len ? o : 0) * st];
      w[s] = sign * op.bnd[k][s];
    }
#pragma unroll
    for (int s = 0; s < SB; s++) {
      const int q = c + dir * (s - k);
      const double t = acc + w[s] * v[s];
      acc = q >= 0 && q < len ? t : acc;
    }
  }
  return acc;
}

__global__ void __launch_bounds__(TPB) k_plain_op_dir(const double *__restrict__ f, double *__restrict__ df,
                                                      const int8_t *__restrict__ codes, int ni, int nj, int dir,
                                                      OpTable op) {
  const int p = blockIdx.x * TPB + threadIdx.x;
  const int n = ni * nj;
  if (p >= n) return;
  const int i = p % ni, j = p / ni;
  const int c = dir == 0 ? i : j, len = dir == 0 ? ni : nj, st = dir == 0 ? 1 : ni;
  const int code = codes ? (int)codes[p] : default_code(c, len, op.nb);
  df[p] = plain_row(op, f, p, c, len, st, code);
}

// StandardCentral::take_derivative_xyz (spatial:1802-1826):
// out = (0 + m[xi][d] d/dxi + m[eta][d] d/deta) * J
__global__ void __launch_bounds__(TPB) k_plain_deriv_xyz(const double *__restrict__ f, double *__restrict__ out,
                                                         const double *__restrict__ met,
                                                         const double *__restrict__ jac,
                                                         const int8_t *__restrict__ codes, int ni, int nj, int dxyz,
                                                         OpTable op) {
#pragma clang fp contract(off)
  const int p = blockIdx.x * TPB + threadIdx.x;
  const int n = ni * nj;
  if (p >= n) return;
  const int i = p % ni, j = p / ni;
  const int c0 = codes ? (int)codes[p] : default_code(i, ni, op.nb);
  const int c1 = codes ? (int)codes[n + p] : default_code(j, nj, op.nb);
  const double d0 = plain_row(op, f, p, i, ni, 1, c0);
  const double d1 = plain_row(op, f, p, j, nj, ni, c1);
  double sum = 0.0;
  sum += met[(size_t)(0 + dxyz) * n + p] * d0;
  sum += met[(size_t)(2 + dxyz) * n + p] * d1;
  out[p] = sum * jac[p];
}

// metrics::compute_ThomasLombard_2D + compute_Jacobian (metrics.cpp:107-129,
// 255-328).  xx = {x_xi, x_eta, y_xi, y_eta}.
__global__ void __launch_bounds__(TPB) k_metrics2d(const double *__restrict__ xx, double *__restrict__ met,
                                                   double *__restrict__ jac, int n) {
#pragma clang fp contract(off)
  const int p = blockIdx.x * TPB + threadIdx.x;
  if (p >= n) return;
  const double x_xi = xx[p], x_eta = xx[(size_t)n + p], y_xi = xx[(size_t)2 * n + p], y_eta = xx[(size_t)3 * n + p];
  met[p] = y_eta;
  met[(size_t)n + p] = -x_eta;
  met[(size_t)2 * n + p] = -y_xi;
  met[(size_t)3 * n + p] = x_xi;
  const double inv = x_xi * y_eta - x_eta * y_xi;
  jac[p] = 1.0 / inv;
}

// compute_auxiliary_variables_linear_Euler (state.cpp:701-736), rho' only:
// rho' = (p' gamma^-1 p_bar^-1 - s') rho_bar
__global__ void __launch_bounds__(TPB) k_aux_rho(const double *__restrict__ y, const double *__restrict__ mean,
                                                 const double *__restrict__ rhob, double *__restrict__ rho,
                                                 double gi, int n) {
#pragma clang fp contract(off)
  const int p = blockIdx.x * TPB + threadIdx.x;
  if (p >= n) return;
  const double pbi = 1.0 / mean[(size_t)IP * n + p];
  double r = y[(size_t)IP * n + p] * gi * pbi - y[(size_t)IS * n + p];
  r *= rhob[p];
  rho[p] = r;
}

// temporal::iblank_correction (temporal:380-393): holes -> sol_ref = 0
__global__ void __launch_bounds__(TPB) k_iblank_reset(double *__restrict__ y, const int8_t *__restrict__ iblank,
                                                      int n, int nv) {
  const int p = blockIdx.x * TPB + threadIdx.x;
  if (p >= n || iblank[p] != BLANKED) return;
  for (int v = 0; v < nv; v++) y[(size_t)v * n + p] = 0.0;
}


// Operands of one plain RK stage (KIND) or of the right-hand side alone.
constexpr int STAGE_RHS = 3;
struct PlainStageArgs {
  int ni, nj, ntx, nty, nv;
  const double *yin, *yn;           // stage input; y_n
  double *acc, *out;                // y_{n+1} accumulator; next stage input (STAGE_RHS: the right-hand side)
  const double *met, *jac, *mean, *mgrad, *rhob;
  const double *rho;                // carried aux density (null: that of yin)
  const int8_t *iblank, *codes;     // blocks with holes
  const double *r;                  // axisymmetric runs: the radius
  double gam, gi;
  int nz;
  ZoneT<double> z[MAX_ZONES];
  int si0, si1, sj0, sj1;
  const double *g;
  double s1, s2, he;
  double h, bi, a;
};

// spatial::compute_RHS + compute_RHS_linearized_Euler + add_RHSSourceTerms
// (spatial:1963-1990, 2053-2158; source.cpp:10-320) and RungeKutta::integrate's
// update loop (temporal:208-230) at one point, in the reference's order:
//   d/dx_d = (0 + m[xi][d] d/dxi + m[eta][d] d/deta) * J  (spatial:1802-1826)
//   rhs -= a * b ;  rhs -= (u' + rho'/rho_bar * u_bar) * grad  (spatial:2089-2092)
//   rhs -= gamma (pbar u_r' + p' ubar_r) / (r + 1e-99)  (axisymmetric, spatial:2119-2126)
//   rhs_p += (s1 * g) * s2 ;  rhs += -sigma (y - target) zone by zone
//   rhs *= h ;  y_next += b_i rhs ;  next input = y_n + a rhs ;  holes 0
// The aux density of a stage after the first is that of its input at the
// same point (state.cpp:701-736), so it is formed here from the two values
// it needs instead of being stored and read.
//
// What bounds it: at small blocks the latency of one workgroup, at large ones
// the arrays of 8 bytes a stage reads and writes (32 a point in the middle
// ones).  The tile with its halo goes through LDS and every other operand of
// the point is requested before the barrier, so a workgroup waits on memory
// once; reading the rows from L1 instead waited row by row, and a sponge's
// strength read once per variable five times (middle stage at 201 x 201
// 13.6 us, 12.1 us with the tile, 9.0 us with one strength read).  One launch
// per operator moved every intermediate through memory and made about 230
// launches a step: a step of 201 x 201 took 655 us and one of 461 x 307 with
// two walls 790 us; these stages and two filter launches take 49 and 111.
template <int HALF>
constexpr int plain_halo() { return HALF == 2 ? 2 : 8; }  // what a closure row of 2 HALF - 1 entries reaches

template <int HALF, int KIND>
__global__ void __launch_bounds__(TPB) k_plain_stage(PlainStageArgs a, OpTable op) {
#pragma clang fp contract(off)
  constexpr int H = plain_halo<HALF>(), RS = 64 + 2 * H, NR = 4 + 2 * H;
  __shared__ double s[4][NR][RS];
  const int tile = xcd_tile(blockIdx.x, (a.ntx * a.nty + 7) / 8);
  if (tile >= a.ntx * a.nty) return;
  const int tx = threadIdx.x, ty = threadIdx.y;
  const int i0 = (tile % a.ntx) * 64, j0 = (tile / a.ntx) * 4;
  const int i = i0 + tx, j = j0 + ty;
  const int ni = a.ni, nj = a.nj, n = ni * nj;
  constexpr int VAR[4] = {IS, IUX, IUY, IP};
  // the tile and its halo (0 outside the block, where no row reads)
  double ta[4][NR / 4], tb[4][NR / 4];
#pragma unroll
  for (int k = 0; k < NR / 4; k++) {
    const int gj = j0 - H + ty + 4 * k, ga = i0 - H + tx, gb = ga + 64;
    const bool row = gj >= 0 && gj < nj, oka = row && ga >= 0 && ga < ni, okb = tx < 2 * H && row && gb < ni;
#pragma unroll
    for (int v = 0; v < 4; v++) {
      const double *f = a.yin + (size_t)VAR[v] * n;
      ta[v][k] = oka ? f[gj * ni + ga] : 0.0;
      tb[v][k] = okb ? f[gj * ni + gb] : 0.0;
    }
  }
  // the point's own operands (those of the last point for lanes outside)
  const bool own = i < ni && j < nj;
  const int p = own ? j * ni + i : n - 1;
  const bool hole = KIND != STAGE_RHS && a.iblank && a.iblank[p] == BLANKED;
  const int c0 = a.codes ? (int)a.codes[p] : default_code(i, ni, op.nb);
  const int c1 = a.codes ? (int)a.codes[n + p] : default_code(j, nj, op.nb);
  const double m[2][2] = {{a.met[p], a.met[(size_t)n + p]}, {a.met[(size_t)2 * n + p], a.met[(size_t)3 * n + p]}};
  const double J = a.jac[p];
  const double ub[2] = {a.mean[(size_t)IUX * n + p], a.mean[(size_t)IUY * n + p]};
  const double rhob = a.rhob[p], pbar = a.mean[(size_t)IP * n + p];
  const double rho_in = a.rho ? a.rho[p] : 0.0, rad = a.r ? a.r[p] : 0.0;
  double g[NV][2], acc[NV], yn[NV];
#pragma unroll
  for (int v = 0; v < NV; v++) {
#pragma unroll
    for (int d = 0; d < 2; d++) g[v][d] = v == IUZ ? 0.0 : a.mgrad[(size_t)(2 * v + d) * n + p];
    acc[v] = KIND == STAGE_MID || KIND == STAGE_LAST ? a.acc[(size_t)v * n + p] : 0.0;
    yn[v] = KIND == STAGE_MID ? a.yn[(size_t)v * n + p] : 0.0;
  }
  const double w = a.yin[(size_t)IUZ * n + p];
#pragma unroll
  for (int k = 0; k < NR / 4; k++)
#pragma unroll
    for (int v = 0; v < 4; v++) {
      s[v][ty + 4 * k][tx] = ta[v][k];
      if (tx < 2 * H) s[v][ty + 4 * k][64 + tx] = tb[v][k];
    }
  __syncthreads();
  if (!own) return;
  if (hole) {
    for (int v = 0; v < a.nv; v++) {
      a.acc[(size_t)v * n + p] = 0.0;
      if (KIND != STAGE_LAST) a.out[(size_t)v * n + p] = 0.0;
    }
    return;
  }
  // chain rule from the two rows
  auto chain = [&](double d0, double d1, double (&out)[2]) {
#pragma unroll
    for (int d = 0; d < 2; d++) {
      double sum = 0.0;
      sum += m[0][d] * d0;
      sum += m[1][d] * d1;
      out[d] = sum * J;
    }
  };
  auto deriv = [&](int v, double (&out)[2]) {
    const double *f = &s[v][ty + H][tx + H];
    chain(plain_row_h<HALF>(op, f, 0, i, ni, 1, c0), plain_row_h<HALF>(op, f, 0, j, nj, RS, c1), out);
  };
  // the sponges, zone by zone, on nv variables whose other terms give r and
  // whose stage inputs are y (nothing relaxes towards a wave but s')
  auto sponges = [&](const double *y, double *r, auto nvar, bool entropy) {
#pragma unroll 1
    for (int q = 0; q < a.nz; q++) {
      const ZoneT<double> &z = a.z[q];
      if (i < z.i0 || i > z.i1 || j < z.j0 || j > z.j1) continue;
      const int zp = (j - z.j0) * z.nzi + (i - z.i0);
      const double sig = z.sig[zp];
      // a harmonic zone (apply_bufferZone_Freund_harmonicWave, source.cpp:264-320)
      // relaxes s' to the entropy wave he * hg and the other variables to 0
      const double wave = entropy && z.harm ? (z.hg ? a.he * z.hg[zp] : a.he) : 0.0;
#pragma unroll
      for (int v = 0; v < nvar.value; v++) {
        const double relax = -sig * (y[v] - (v == IS ? wave : 0.0));
        r[v] += relax;
      }
    }
  };
  auto update = [&](int v, double y, double r, double accv, double ynv) {
    const size_t q = (size_t)v * n + p;
    if (KIND == STAGE_RHS) {
      a.out[q] = r;
      return;
    }
    r *= a.h;
    double next = KIND == STAGE_FIRST ? y : accv;
    next += a.bi * r;
    a.acc[q] = next;
    if (KIND != STAGE_LAST) a.out[q] = (KIND == STAGE_FIRST ? y : ynv) + a.a * r;
  };
  const double yc[4] = {s[0][ty + H][tx + H], s[1][ty + H][tx + H], s[2][ty + H][tx + H], s[3][ty + H][tx + H]};
  const double up[2] = {yc[1], yc[2]}, pp = yc[3];
  double rho = rho_in;
  if (!a.rho) {
    const double pbi = 1.0 / pbar;
    rho = pp * a.gi * pbi - yc[0];
    rho *= rhob;
  }
  double ds[2], du[2][2], dp[2];
  deriv(0, ds);
  deriv(1, du[0]);
  deriv(2, du[1]);
  deriv(3, dp);
  double r[NV] = {0.0, 0.0, 0.0, 0.0, 0.0};
#pragma unroll
  for (int d = 0; d < 2; d++) {
    r[IS] -= ub[d] * ds[d];
    r[IS] -= up[d] * g[IS][d];
  }
#pragma unroll
  for (int vel = 0; vel < 2; vel++) {
#pragma unroll
    for (int d = 0; d < 2; d++) {
      r[IUX + vel] -= ub[d] * du[vel][d];
      r[IUX + vel] -= (up[d] + rho / rhob * ub[d]) * g[IUX + vel][d];
    }
    r[IUX + vel] -= dp[vel] / rhob;
  }
#pragma unroll
  for (int d = 0; d < 2; d++) {
    r[IP] -= ub[d] * dp[d];
    r[IP] -= up[d] * g[IP][d];
    r[IP] -= a.gam * pbar * du[d][d];
    r[IP] -= a.gam * pp * g[IUX + d][d];
  }
  if (a.r) {
    const double DUMMY_SMALL = 1e-99;
    r[IP] -= a.gam * (pbar * up[1] + pp * ub[1]) / (rad + DUMMY_SMALL);
  }
  if (i >= a.si0 && i <= a.si1 && j >= a.sj0 && j <= a.sj1)
    r[IP] += a.s1 * a.g[(j - a.sj0) * (a.si1 - a.si0 + 1) + (i - a.si0)] * a.s2;
  const double y5[NV] = {yc[0], up[0], up[1], w, pp};
  sponges(y5, r, std::integral_constant<int, NV>{}, true);
#pragma unroll
  for (int v = 0; v < NV; v++) update(v, y5[v], r[v], acc[v], yn[v]);
  // passive scalars, compute_RHS_linearized_Euler_scalar (spatial:2134-2158),
  // their rows read in place
  for (int v = NV; v < a.nv; v++) {
    const double *f = a.yin + (size_t)v * n;
    const size_t q = (size_t)v * n + p;
    double dz[2], rz = 0.0;
    chain(plain_row_h<HALF>(op, f, p, i, ni, 1, c0), plain_row_h<HALF>(op, f, p, j, nj, ni, c1), dz);
#pragma unroll
    for (int d = 0; d < 2; d++) {
      rz -= ub[d] * dz[d];
      rz -= up[d] * a.mgrad[(size_t)(2 * v + d) * n + p];
    }
    const double y = f[p];
    sponges(&y, &rz, std::integral_constant<int, 1>{}, false);
    update(v, y, rz, KIND == STAGE_MID || KIND == STAGE_LAST ? a.acc[q] : 0.0, KIND == STAGE_MID ? a.yn[q] : 0.0);
  }
}

// spatial::apply_filter (spatial:2191-2246), first launch: tmp = F_xi y of
// variable blockIdx.y (one thread a variable and point: five variables in
// turn were five latencies), and the aux density of the unfiltered y (rho null: not
// wanted), which the next step's first stage takes.
template <int HALF>
__global__ void __launch_bounds__(TPB) k_plain_filter_xi(const double *__restrict__ y, double *__restrict__ tmp,
                                                         const int8_t *__restrict__ codes, int ni, int nj, OpTable op,
                                                         const double *__restrict__ mean,
                                                         const double *__restrict__ rhob, double *__restrict__ rho,
                                                         double gi) {
#pragma clang fp contract(off)
  const int n = ni * nj, p = blockIdx.x * TPB + threadIdx.x;
  if (p >= n) return;
  const int i = p % ni, v = blockIdx.y, code = codes ? (int)codes[p] : default_code(i, ni, op.nb);
  tmp[(size_t)v * n + p] = plain_row_h<HALF>(op, y + (size_t)v * n, p, i, ni, 1, code);
  if (rho && v == 0) {
    const double pbi = 1.0 / mean[(size_t)IP * n + p];
    double r = y[(size_t)IP * n + p] * gi * pbi - y[(size_t)IS * n + p];
    r *= rhob[p];
    rho[p] = r;
  }
}

// Second launch: y = (1 - blend) y + blend F_eta tmp, holes reset to 0 when
// iblank is given (temporal::iblank_correction).
template <int HALF>
__global__ void __launch_bounds__(TPB) k_plain_filter_eta(double *__restrict__ y, const double *__restrict__ tmp,
                                                          const int8_t *__restrict__ codes,
                                                          const int8_t *__restrict__ iblank, int ni, int nj,
                                                          OpTable op, double rem, double blend) {
#pragma clang fp contract(off)
  const int n = ni * nj, p = blockIdx.x * TPB + threadIdx.x;
  if (p >= n) return;
  const int j = p / ni, code = codes ? (int)codes[n + p] : default_code(j, nj, op.nb);
  const bool hole = iblank && iblank[p] == BLANKED;
  const size_t vo = (size_t)blockIdx.y * n;
  const double f = plain_row_h<HALF>(op, tmp + vo, p, j, nj, ni, code);
  const double out = rem * y[vo + p] + blend * f;
  y[vo + p] = hole ? 0.0 : out;
}

inline unsigned nblocks(size_t n) { return (unsigned)((n + TPB - 1) / TPB); }

}  // namespace

// ------------------------------------------------------------- launchers

hipError_t metrics2d(hipStream_t s, Block &b, const OpTable &fd) {
  // x_xi, x_eta, y_xi, y_eta by the FD operator with no holes (metrics are
  // computed before overset marks any, simulation.cpp:207-217)
  double *xx = nullptr;
  hipError_t e = hipMalloc((void **)&xx, sizeof(double) * 4 * (size_t)b.n);
  if (e != hipSuccess) return e;
  for (int ph = 0; ph < 2; ph++)
    for (int cp = 0; cp < 2; cp++) {
      hipLaunchKernelGGL(k_plain_op_dir, dim3(nblocks(b.n)), dim3(TPB), 0, s, b.xyz + (size_t)ph * b.n,
                         xx + (size_t)(2 * ph + cp) * b.n, (const int8_t *)nullptr, b.ni, b.nj, cp, fd);
    }
  hipLaunchKernelGGL(k_metrics2d, dim3(nblocks(b.n)), dim3(TPB), 0, s, xx, b.met, b.jac, b.n);
  e = hipGetLastError();
  hipError_t e2 = hipStreamSynchronize(s);
  (void)hipFree(xx);
  return e != hipSuccess ? e : e2;
}

hipError_t plain_take_derivative_xyz(hipStream_t s, const Block &b, const OpTable &op, const double *f,
                                     int dir_xyz) {
  hipLaunchKernelGGL(k_plain_deriv_xyz, dim3(nblocks(b.n)), dim3(TPB), 0, s, f, b.dflux, b.met, b.jac,
                     b.has_holes ? b.code_fd : nullptr, b.ni, b.nj, dir_xyz, op);
  return hipGetLastError();
}

hipError_t aux_density(hipStream_t s, const Block &b, double gamma, const double *y, double *rho) {
  hipLaunchKernelGGL(k_aux_rho, dim3(nblocks(b.n)), dim3(TPB), 0, s, y, b.mean, b.rhobar, rho, 1.0 / gamma, b.n);
  return hipGetLastError();
}

hipError_t plain_stage(hipStream_t s, lee_handle *h, const Block &b, int stage, const StageScalars &sc,
                       const double *rho) {
  PlainStageArgs a{};
  a.ni = b.ni;
  a.nj = b.nj;
  a.ntx = (b.ni + 63) / 64;
  a.nty = (b.nj + 3) / 4;
  a.nv = nvars(h);
  // the buffers of the fused stages (make_stage_args); stage < 0: the
  // right-hand side of Y[2] into Y[3]
  const int in_idx = stage == 0 ? 0 : (stage % 2 == 1 || stage < 0 ? 2 : 3);
  a.yin = b.Y64[in_idx];
  a.yn = b.Y64[0];
  a.acc = b.Y64[1];
  a.out = b.Y64[stage < 0 ? 3 : (stage % 2 == 0 ? 2 : 3)];
  a.met = b.met;
  a.jac = b.jac;
  a.mean = b.mean;
  a.mgrad = b.mgrad;
  a.rhob = b.rhobar;
  a.rho = rho;
  a.iblank = b.has_holes ? b.iblank : nullptr;
  a.codes = b.has_holes ? b.code_fd : nullptr;
  a.r = h->cfg.axisym ? b.xyz + b.n : nullptr;
  a.gam = h->cfg.gamma;
  a.gi = 1.0 / h->cfg.gamma;
  for (const auto &z : b.zones) {
    if (a.nz >= MAX_ZONES) break;
    a.z[a.nz++] = {z.is[0], z.ie[0], z.is[1], z.ie[1], z.nz[0], z.sigma64, z.harmonic ? 1 : 0, z.hg};
  }
  a.si0 = b.src.i0;
  a.si1 = b.src.i1;
  a.sj0 = b.src.j0;
  a.sj1 = b.src.j1;
  a.g = b.src.g;
  a.s1 = sc.s1;
  a.s2 = sc.s2;
  a.he = sc.he;
  a.h = sc.h;
  a.bi = sc.b;
  a.a = sc.a;
  const dim3 grid((a.ntx * a.nty + 7) / 8 * 8), block(64, 4);
  const int last = h->cfg.rk_stages - 1;
#define LEE_PS(HALF)                                                                                         \
  do {                                                                                                       \
    if (stage < 0) hipLaunchKernelGGL((k_plain_stage<HALF, STAGE_RHS>), grid, block, 0, s, a, h->fd);        \
    else if (stage == 0) hipLaunchKernelGGL((k_plain_stage<HALF, STAGE_FIRST>), grid, block, 0, s, a, h->fd); \
    else if (stage < last) hipLaunchKernelGGL((k_plain_stage<HALF, STAGE_MID>), grid, block, 0, s, a, h->fd); \
    else hipLaunchKernelGGL((k_plain_stage<HALF, STAGE_LAST>), grid, block, 0, s, a, h->fd);                 \
  } while (0)
  if (h->fd.half == 2) LEE_PS(2);
  else LEE_PS(5);
#undef LEE_PS
  return hipGetLastError();
}

hipError_t plain_filter(hipStream_t s, lee_handle *h, const Block &b, double *y, double *tmp, double *rho,
                        bool reset_holes) {
  const dim3 g(nblocks(b.n), nvars(h)), t(TPB);
  const int8_t *cx = b.has_holes ? b.code_flt : nullptr, *ib = b.has_holes && reset_holes ? b.iblank : nullptr;
  const double blend = h->cfg.filter_blend, rem = 1.0 - blend, gi = 1.0 / h->cfg.gamma;
#define LEE_PF(HALF)                                                                                              \
  do {                                                                                                            \
    hipLaunchKernelGGL((k_plain_filter_xi<HALF>), g, t, 0, s, y, tmp, cx, b.ni, b.nj, h->flt, b.mean, b.rhobar,   \
                       rho, gi);                                                                                  \
    hipLaunchKernelGGL((k_plain_filter_eta<HALF>), g, t, 0, s, y, tmp, cx, ib, b.ni, b.nj, h->flt, rem, blend);   \
  } while (0)
  if (h->flt.half == 2) LEE_PF(2);
  else if (h->flt.half == 4) LEE_PF(4);
  else LEE_PF(5);
#undef LEE_PF
  return hipGetLastError();
}

hipError_t plain_iblank_reset(hipStream_t s, const Block &b, double *y, int nv) {
  if (!b.has_holes) return hipSuccess;
  hipLaunchKernelGGL(k_iblank_reset, dim3(nblocks(b.n)), dim3(TPB), 0, s, y, b.iblank, b.n, nv);
  return hipGetLastError();
}

}  // namespace lee
