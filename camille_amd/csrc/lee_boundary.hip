// Boundary phase of the 2-D paths: the faces' conditions
// (boundary_condition.cpp) and the overset interpolation (overset.cpp).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <type_traits>

#include "lee_args.h"

namespace lee {

namespace {

// ------------------------------------------------------ boundary conditions

// Stores and loads that other workgroups of the same launch see: past the
// caches that each XCD has to itself.
template <typename T>
__device__ __forceinline__ void put(T *p, T x) {
  __hip_atomic_store(p, x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <typename T>
__device__ __forceinline__ T get(const T *p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// One point of a BC face in global memory.  SHARED: other workgroups of the
// launch read or overwrite it.  NS: as bc_neumann_value's (OA4 faces read two
// points inward, not eight).
template <typename T, int NS, bool SHARED>
__device__ __forceinline__ void bc_face_point(T *__restrict__ y, const double *__restrict__ met,
                                              const double *__restrict__ jac, const int8_t *__restrict__ iblank,
                                              const BcArgs &a, T *__restrict__ rho, const double *__restrict__ mean,
                                              const double *__restrict__ rhob, double gi, int q) {
#pragma clang fp contract(off)
  const int fw = a.i1 - a.i0 + 1;
  const int i = a.i0 + q % fw, j = a.j0 + q / fw;
  const int n = a.ni * a.nj;
  const int p = j * a.ni + i;
  if (iblank && iblank[p] == BLANKED) return;
  const int c = a.dir == 0 ? i : j, len = a.dir == 0 ? a.ni : a.nj, sg = a.end == 0 ? 1 : -1;
  const int mf = a.dir == 0 ? 1 : a.ni;
  // the block point s points inward (clamped to the face point)
  auto at = [&](int s) {
    const int cs = c + sg * s;
    return p + sg * mf * (cs >= 0 && cs < len ? s : 0);
  };
  auto set = [](T *to, double x) {
    if constexpr (SHARED) put(to, (T)x);
    else *to = (T)x;
  };
  double data[NV];
  bc_face_data<T, NS>(a, q, p, c, len, met, jac, [&](int v, int s) { return y[(size_t)v * n + at(s)]; }, data);
  // passive scalars: Neumann data at Neumann, wall-slip (its non-velocity
  // variables, boundary_condition.cpp:122-136) and centerline faces; 0 at
  // dirichlet_allzero and harmonic-wave faces, whose data start at 0
  for (int z = 0; z < a.nsc; z++) {
    const size_t vo = (size_t)(NV + z) * n;
    double d = 0.0;
    if (bc_is_neumann(a)) {
      T nbz[NS];
#pragma unroll
      for (int s = 1; s <= NS; s++) nbz[s - 1] = y[vo + at(NS == 2 || s < a.sb ? s : 0)];
      d = bc_neumann_value<T, NS>(a, c, len, nbz);
    }
    set(&y[vo + p], d);
  }
  for (int v = 0; v < NV; v++) set(&y[(size_t)v * n + p], data[v]);
  if (rho) {
    const double pbi = 1.0 / mean[(size_t)IP * n + p];
    double r = data[IP] * gi * pbi - data[IS];
    r *= rhob[p];
    set(&rho[p], r);
  }
}

// Faces of one block that neither read nor write a point another one of them
// writes, in one launch: workgroups start[k] .. start[k + 1] - 1 take face k.
// A launch of one face is all latency (4 us for 700 points), so faces that
// may share one do (a channel's two walls: 8 launches a step -> 4).
constexpr int BC_BATCH = 4;
struct BcBatch {
  int nf;
  int start[BC_BATCH + 1];
  BcArgs f[BC_BATCH];
};

template <typename T, int NS>
__global__ void __launch_bounds__(TPB) k_bc_faces(T *__restrict__ y, const double *__restrict__ met,
                                                  const double *__restrict__ jac,
                                                  const int8_t *__restrict__ iblank, BcBatch b,
                                                  T *__restrict__ rho, const double *__restrict__ mean,
                                                  const double *__restrict__ rhob, double gi) {
  int k = 0;
  while (k + 1 < b.nf && (int)blockIdx.x >= b.start[k + 1]) k++;
  const BcArgs &a = b.f[k];
  const int q = ((int)blockIdx.x - b.start[k]) * TPB + threadIdx.x;
  if (q >= (a.i1 - a.i0 + 1) * (a.j1 - a.j0 + 1)) return;
  bc_face_point<T, NS, false>(y, met, jac, iblank, a, rho, mean, rhob, gi, q);
}

// ---------------------------------------------------------------- overset

template <typename T>
struct OvTables {
  int nv;  // variables per point (NV and the passive scalars)
  T *y[MAX_OV_BLOCKS];
  int ni[MAX_OV_BLOCKS], nn[MAX_OV_BLOCKS];
  T *rho[MAX_OV_BLOCKS];
  const double *mean[MAX_OV_BLOCKS];
  const double *rhob[MAX_OV_BLOCKS];
};

// compute_weighted_sum (overset.cpp:886-974): every receiver's weighted
// donor sum into buf before any receiver is written.
template <typename T>
__global__ void __launch_bounds__(TPB) k_ov_gather(OvTables<T> t, const int *__restrict__ db,
                                                   const int *__restrict__ dl, const int *__restrict__ w,
                                                   const double *__restrict__ coef, int stride,
                                                   double *__restrict__ buf, int nrecv) {
#pragma clang fp contract(off)
  const int r = blockIdx.x * TPB + threadIdx.x;
  if (r >= nrecv) return;
  const int b = db[r];
  const T *y = t.y[b];
  const int ni = t.ni[b], n = t.nn[b];
  const int w1 = w[3 * b], w2 = w[3 * b + 1];
  const double *c = coef + (size_t)r * stride;
  if (w1 == 5 && w2 == 5 && w[3 * b + 2] == 1) {
    // ORDER 4 in 2-D: the 25 donors of one variable are requested together
    // (clamped addresses, skipped donors masked), then summed in the
    // reference's order; one memory latency per variable instead of one
    // per donor
    const int d0 = dl[r];
    double cc[25];
    int li[25];
    bool ok[25];
#pragma unroll
    for (int q = 0; q < 25; q++) {
      const int l1 = d0 + (q % 5) + (q / 5) * ni;
      ok[q] = l1 >= 0 && l1 < n;
      li[q] = ok[q] ? l1 : 0;
      cc[q] = c[q];
    }
    for (int v = 0; v < t.nv; v++) {
      T yv[25];
#pragma unroll
      for (int q = 0; q < 25; q++) yv[q] = y[(size_t)v * n + li[q]];
      double a = 0.0;
#pragma unroll
      for (int q = 0; q < 25; q++) {
        const double t1 = a + cc[q] * (double)yv[q];
        a = ok[q] ? t1 : a;
      }
      buf[(size_t)r * t.nv + v] = a;
    }
    return;
  }
  double acc[MAXV];
  for (int v = 0; v < MAXV; v++) acc[v] = 0.0;
  int s = 0;
  for (int b2 = 0; b2 < w2; b2++)
    for (int b1 = 0; b1 < w1; b1++) {
      const int l1 = dl[r] + b1 + b2 * ni;
      if (l1 >= 0 && l1 < n)
        for (int v = 0; v < t.nv; v++) acc[v] += c[s] * (double)y[(size_t)v * n + l1];
      s++;
    }
  for (int v = 0; v < t.nv; v++) buf[(size_t)r * t.nv + v] = acc[v];
}

// compute_weighted_sum for 5 x 5 stencils (overset.cpp:886-974), receiver r
// and variable v: the 25 donor values and coefficients (receiver-minor, so
// coalesced across receivers) are requested together, then summed in the
// reference's order with the donors outside the block skipped.
template <typename T>
__device__ __forceinline__ double ov_sum5(const OvTables<T> &t, const int *__restrict__ db,
                                          const int *__restrict__ dl, const double *__restrict__ coef5, int nrecv,
                                          int r, int v) {
#pragma clang fp contract(off)
  const int b = db[r];
  const T *y = t.y[b] + (size_t)v * t.nn[b];
  const int ni = t.ni[b], n = t.nn[b], d0 = dl[r];
  double cc[25];
  T yv[25];
  bool ok[25];
#pragma unroll
  for (int q = 0; q < 25; q++) {
    const int l1 = d0 + (q % 5) + (q / 5) * ni;
    ok[q] = l1 >= 0 && l1 < n;
    cc[q] = coef5[(size_t)q * nrecv + r];
    yv[q] = y[ok[q] ? l1 : 0];
  }
  double a = 0.0;
#pragma unroll
  for (int q = 0; q < 25; q++) {
    const double t1 = a + cc[q] * (double)yv[q];
    a = ok[q] ? t1 : a;
  }
  return a;
}

// The gather of the two-phase update: one thread per (receiver, variable),
// every sum into buf before any receiver is written.
template <typename T>
__global__ void __launch_bounds__(TPB) k_ov_gather5(OvTables<T> t, const int *__restrict__ db,
                                                    const int *__restrict__ dl, const double *__restrict__ coef5,
                                                    double *__restrict__ buf, int nrecv) {
  const int gid = blockIdx.x * TPB + threadIdx.x;
  if (gid >= t.nv * nrecv) return;
  const int v = gid / nrecv, r = gid - v * nrecv;
  buf[(size_t)r * t.nv + v] = ov_sum5(t, db, dl, coef5, nrecv, r, v);
}

// update_each_grid (overset.cpp:1241-1278); optionally refreshes rho'.
template <typename T>
__device__ __forceinline__ void ov_scatter_one(const OvTables<T> &t, const int *__restrict__ rb,
                                               const int *__restrict__ rl, const double *__restrict__ buf,
                                               int with_rho, double gi, int r) {
#pragma clang fp contract(off)
  const int b = rb[r];
  const int n = t.nn[b], p = rl[r];
  if (p < 0 || p >= n) return;
  for (int v = 0; v < t.nv; v++) t.y[b][(size_t)v * n + p] = (T)buf[(size_t)r * t.nv + v];
  if (with_rho && t.rho[b]) {
    const double pbi = 1.0 / t.mean[b][(size_t)IP * n + p];
    double q = buf[(size_t)r * t.nv + IP] * gi * pbi - buf[(size_t)r * t.nv + IS];
    q *= t.rhob[b][p];
    t.rho[b][p] = (T)q;
  }
}

template <typename T>
__global__ void __launch_bounds__(TPB) k_ov_scatter(OvTables<T> t, const int *__restrict__ rb,
                                                    const int *__restrict__ rl, const double *__restrict__ buf,
                                                    int nrecv, int with_rho, double gi) {
  const int r = blockIdx.x * TPB + threadIdx.x;
  if (r >= nrecv) return;
  ov_scatter_one<T>(t, rb, rl, buf, with_rho, gi, r);
}

// The value of entry b of a per-block table in the kernel arguments: every
// entry is a scalar load issued at once, where indexing by lane would be a
// dependent load.
template <typename P>
__device__ __forceinline__ P of_block(const P (&t)[MAX_OV_BLOCKS], int b) {
  P r = t[0];
#pragma unroll
  for (int k = 1; k < MAX_OV_BLOCKS; k++) r = b == k ? t[k] : r;
  return r;
}

// Boundary phase of one stage in one launch: BC faces that may share a
// launch, of any block, and the interpolation of receivers ordered by
// plan_overset (lee_api.hip).
template <typename T>
struct BndFace {
  BcArgs a;
  T *y, *rho;
  const double *met, *jac, *mean, *rhob;
  const int8_t *iblank;
};
template <typename T>
struct BndArgs {
  OvTables<T> t;
  int nf, start[BC_BATCH + 1];  // faces; workgroups start[k] .. start[k + 1] - 1 take face k
  BndFace<T> f[BC_BATCH];
  const int *rb, *rl, *db, *dl;
  const double *coef5;
  double *buf;
  unsigned *done;               // workgroups that have ended their part; 0 between launches
  // receivers: nheld held ones, then those that read a held one (up to nuse),
  // others, and from nearly on those that read face points
  int nrecv, nheld, nuse, nearly, rpw, with_rho;
  double gi;
};

// Sum of receiver r, variable v (ov_sum5; the stencil lies in its block): its
// coefficients and the first donor's place, then the sum.  SHARED: some
// donors are points that other workgroups have written.
template <typename T>
struct OvSum {
  double c[25];
  const T *y;
  int ni;
};
template <typename T>
__device__ __forceinline__ OvSum<T> ov_stencil(const BndArgs<T> &a, int r, int v) {
  OvSum<T> s;
  const int b = a.db[r];
#pragma unroll
  for (int q = 0; q < 25; q++) s.c[q] = a.coef5[(size_t)q * a.nrecv + r];
  const int d0 = a.dl[r];
  s.ni = of_block(a.t.ni, b);
  s.y = of_block(a.t.y, b) + (size_t)v * of_block(a.t.nn, b) + d0;
  return s;
}
template <typename T, bool SHARED>
__device__ __forceinline__ double ov_sum(const OvSum<T> &o) {
#pragma clang fp contract(off)
  T yv[25];
#pragma unroll
  for (int q = 0; q < 25; q++) {
    const T *p = &o.y[(q % 5) + (q / 5) * o.ni];
    yv[q] = SHARED ? get(p) : *p;
  }
  double s = 0.0;
#pragma unroll
  for (int q = 0; q < 25; q++) s = s + o.c[q] * (double)yv[q];
  return s;
}

template <typename T>
__device__ __forceinline__ void ov_rho(const BndArgs<T> &a, int b, int p, double sp, double ss) {
#pragma clang fp contract(off)
  T *rho = of_block(a.t.rho, b);
  if (!rho) return;
  const double pbi = 1.0 / of_block(a.t.mean, b)[(size_t)IP * of_block(a.t.nn, b) + p];
  double q = sp * a.gi * pbi - ss;
  q *= of_block(a.t.rhob, b)[p];
  rho[p] = (T)q;
}

// All latency: three launches (faces, gather, scatter) took 4.6 + 8.0 + 4.1 us
// on a cylinder's 3858 receivers and 257 face points, for 2 MB; this one 10.7.  Here every
// workgroup takes face points or sums, and a sum is written at once where
// nobody reads its receiver.  The others' order: workgroups with face points,
// held sums or readers of held receivers count themselves when their part is
// done, and the one that counts last (none waits) forms the sums that read
// face points and writes what was held.  What it reads of the others' goes
// through put and get (a release fence at agent scope instead writes a whole
// L2 back per workgroup: 19 us).  Their order rests on the instruction set, not
// on the memory model, to which all of it is relaxed: gfx950 stores of agent
// scope are written through to where every XCD's loads of agent scope read, and
// s_waitcnt 0 ends only when they have been; the barrier after it puts the
// stores of every wave before the count, and the branch on the count puts the
// loads behind it.
// 128 threads: the lanes of a sum scatter over 25 rows, so the sums are
// spread over as many CUs as there are.
constexpr int OV_T = 128;

// What one workgroup may be left with: the receivers it writes at the end, in
// passes of OV_T.  A pass costs it 1 to 2 us (a float run that refreshes rho':
// 7.9 us for the launch with 2 held receivers, 10.3 with 256, 14.3 with 512,
// 21.7 with 1024, 52 with 3072), where the launches per face, gather and
// scatter take 12 to 18 whatever the receivers' kind.  The sums it forms first
// cost 2.5 to 3.5 us for one pass and as much for the next (14.1 us with 51
// receivers that read face points, 15.8 with 60, 363 with 4000; 12 to 18 us in
// launches of their own), so they have to fit one.
constexpr int OV_LAST_PASSES = 3;

template <typename T, int NS>
__global__ void __launch_bounds__(OV_T) k_boundary(BndArgs<T> a) {
  __shared__ double sums[OV_T];
  __shared__ bool last;
  const int tid = threadIdx.x, nbc = a.start[a.nf], nv = a.t.nv;
  if ((int)blockIdx.x < nbc) {
    int k = 0;
    while (k + 1 < a.nf && (int)blockIdx.x >= a.start[k + 1]) k++;
    const BndFace<T> &f = a.f[k];
    const int q = ((int)blockIdx.x - a.start[k]) * OV_T + tid;
    if (q < (f.a.i1 - f.a.i0 + 1) * (f.a.j1 - f.a.j0 + 1))
      bc_face_point<T, NS, true>(f.y, f.met, f.jac, f.iblank, f.a, f.rho, f.mean, f.rhob, a.gi, q);
  } else {
    const int v = tid / a.rpw, lr = tid - v * a.rpw, r = ((int)blockIdx.x - nbc) * a.rpw + lr;
    const bool on = v < nv && r < a.nearly;
    const int b = on ? a.rb[r] : 0, p = on ? a.rl[r] : 0;
    if (on) {
      const double s = ov_sum<T, false>(ov_stencil(a, r, v));
      if (r < a.nheld) put(&a.buf[(size_t)v * a.nrecv + r], s);
      else of_block(a.t.y, b)[(size_t)v * of_block(a.t.nn, b) + p] = (T)s;
      sums[tid] = s;
    }
    if (a.with_rho) {
      __syncthreads();
      if (on && v == 0 && r >= a.nheld) ov_rho(a, b, p, sums[IP * a.rpw + lr], sums[IS * a.rpw + lr]);
    }
  }
  if (a.nheld == 0 && a.nearly == a.nrecv) return;
  const int counted = nbc + max((a.nuse + a.rpw - 1) / a.rpw, 1);
  if ((int)blockIdx.x >= counted) return;
  // what the last part needs of the tables, requested before the count: each
  // read after it is one more latency on the launch
  const int nlate = (a.nrecv - a.nearly) * nv, nw = a.nheld + a.nrecv - a.nearly;
  auto late = [&](int q) { return ov_stencil(a, a.nearly + q / nv, q % nv); };
  auto written = [&](int q) { return q < a.nheld ? q : a.nearly + q - a.nheld; };
  OvSum<T> first{};
  if (tid < nlate) first = late(tid);
  int wb = 0, wp = 0;
  if (tid < nw) {
    wb = a.rb[written(tid)];
    wp = a.rl[written(tid)];
  }
  // this wave's loads have returned and its stores are complete
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
  __builtin_amdgcn_s_waitcnt(0);
  __syncthreads();
  if (tid == 0)
    last = __hip_atomic_fetch_add(a.done, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == (unsigned)counted - 1;
  __syncthreads();
  if (!last) return;
  for (int q = tid; q < nlate; q += OV_T) {
    if (q != tid) first = late(q);
    put(&a.buf[(size_t)(q % nv) * a.nrecv + a.nearly + q / nv], ov_sum<T, true>(first));
  }
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
  __builtin_amdgcn_s_waitcnt(0);
  __syncthreads();
  for (int q = tid; q < nw; q += OV_T) {
    const int r = written(q);
    if (q != tid) {
      wb = a.rb[r];
      wp = a.rl[r];
    }
    T *y = of_block(a.t.y, wb);
    const int n = of_block(a.t.nn, wb);
    double s[MAXV];
#pragma unroll
    for (int v = 0; v < MAXV; v++) s[v] = v < nv ? get(&a.buf[(size_t)v * a.nrecv + r]) : 0.0;
#pragma unroll
    for (int v = 0; v < MAXV; v++)
      if (v < nv) y[(size_t)v * n + wp] = (T)s[v];
    if (a.with_rho) ov_rho(a, wb, wp, s[IP], s[IS]);
  }
  if (tid == 0) __hip_atomic_store(a.done, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

inline unsigned nblocks(size_t n) { return (unsigned)((n + TPB - 1) / TPB); }

}  // namespace

// ------------------------------------------------------------- launchers

bool boundary_in_one_launch(int nv, int nheld, int nlate) {
  return nlate * nv <= OV_T && nheld + nlate <= OV_LAST_PASSES * OV_T;
}

hipError_t apply_bcs(hipStream_t s, lee_handle *h, const Block &b, double *y64, float *y32, bool fp32,
                     double *rho64, float *rho32, double he) {
  const int8_t *ib = b.has_holes ? b.iblank : nullptr;
  BcBatch t{};
  auto flush = [&]() {
    if (t.nf == 0) return;
    const dim3 grid(t.start[t.nf]);
    const bool oa4 = h->fd.sb == 3;
    auto launch = [&](auto kernel, auto *y, auto *rho) {
      hipLaunchKernelGGL(kernel, grid, dim3(TPB), 0, s, y, b.met, b.jac, ib, t, rho, b.mean, b.rhobar,
                         1.0 / h->cfg.gamma);
    };
    if (fp32) launch(oa4 ? k_bc_faces<float, 2> : k_bc_faces<float, 8>, y32, rho32);
    else launch(oa4 ? k_bc_faces<double, 2> : k_bc_faces<double, 8>, y64, rho64);
    t.nf = 0;
  };
  // in the order of the BC file; a face joins the launch before it unless
  // their reaches meet (faces that share a corner keep their order)
  for (const auto &f : b.faces) {
    const BcArgs a = make_bc_args(h, b, f, he);
    const BcReach r = bc_reach(a);
    bool apart = t.nf < BC_BATCH;
    for (int k = 0; k < t.nf; k++) apart &= bc_apart(r, bc_reach(t.f[k]));
    if (!apart) flush();
    t.f[t.nf] = a;
    t.start[t.nf + 1] = t.start[t.nf] + (int)nblocks((size_t)(a.i1 - a.i0 + 1) * (a.j1 - a.j0 + 1));
    t.nf++;
  }
  flush();
  return hipGetLastError();
}

template <typename T>
static OvTables<T> ov_tables(const lee_handle *h, T *const *ys, T *const *rhos) {
  OvTables<T> t{};
  t.nv = nvars(h);
  for (int ib = 0; ib < h->nblk; ib++) {
    t.y[ib] = ys[ib];
    t.ni[ib] = h->b[ib].ni;
    t.nn[ib] = h->b[ib].n;
    t.rho[ib] = rhos ? rhos[ib] : nullptr;
    t.mean[ib] = h->b[ib].mean;
    t.rhob[ib] = h->b[ib].rhobar;
  }
  return t;
}

// The two-phase form, for receivers without an order and for callers that
// bring their own buffer.
template <typename T>
static hipError_t overset_t(hipStream_t s, lee_handle *h, T *const *ys, T *const *rhos, bool with_rho, double *buf) {
  const OvTables<T> t = ov_tables<T>(h, ys, rhos);
  const Overset &o = h->ov;
  if (o.coef5)
    hipLaunchKernelGGL(k_ov_gather5<T>, dim3(nblocks((size_t)t.nv * o.nrecv)), dim3(TPB), 0, s, t, o.db, o.dl, o.coef5,
                       buf, o.nrecv);
  else
    hipLaunchKernelGGL(k_ov_gather<T>, dim3(nblocks(o.nrecv)), dim3(TPB), 0, s, t, o.db, o.dl, o.w, o.coef, o.stride,
                       buf, o.nrecv);
  hipLaunchKernelGGL(k_ov_scatter<T>, dim3(nblocks(o.nrecv)), dim3(TPB), 0, s, t, o.rb, o.rl, buf, o.nrecv,
                     with_rho ? 1 : 0, 1.0 / h->cfg.gamma);
  return hipGetLastError();
}

hipError_t overset_interpolate_arrays(hipStream_t s, lee_handle *h, double *const *ys, double *buf) {
  if (h->ov.nrecv == 0) return hipSuccess;
  return overset_t<double>(s, h, ys, nullptr, false, buf);
}

// Boundary phase of every block's state buffer: the faces, then the
// interpolation; rhos (or null) are refreshed at the points it sets.
template <typename T>
static hipError_t boundary_phase_t(hipStream_t s, lee_handle *h, T *const *ys, T *const *rhos, double he) {
  const Overset &o = h->ov;
  BndArgs<T> a{};
  bool one = o.ordered;  // the faces of all blocks in the launch of the interpolation
  for (int ib = 0; ib < h->nblk && one; ib++)
    for (const auto &f : h->b[ib].faces) {
      const Block &b = h->b[ib];
      BndFace<T> q{make_bc_args(h, b, f, he), ys[ib], rhos ? rhos[ib] : nullptr, b.met, b.jac, b.mean, b.rhobar,
                   b.has_holes ? b.iblank : nullptr};
      one = one && a.nf < BC_BATCH;
      for (int k = 0; k < a.nf && one; k++) one = a.f[k].y != q.y || bc_apart(bc_reach(a.f[k].a), bc_reach(q.a));
      if (!one) break;
      a.f[a.nf] = q;
      a.start[a.nf + 1] =
          a.start[a.nf] + (int)((size_t)(q.a.i1 - q.a.i0 + 1) * (q.a.j1 - q.a.j0 + 1) + OV_T - 1) / OV_T;
      a.nf++;
    }
  if (!one) {
    for (int ib = 0; ib < h->nblk; ib++) {
      const Block &b = h->b[ib];
      if (b.faces.empty()) continue;
      T *rho = rhos ? rhos[ib] : nullptr;
      hipError_t e;
      if constexpr (sizeof(T) == 8) e = apply_bcs(s, h, b, ys[ib], nullptr, false, rho, nullptr, he);
      else e = apply_bcs(s, h, b, nullptr, ys[ib], true, nullptr, rho, he);
      if (e != hipSuccess) return e;
    }
    a.nf = 0;
  }
  if (o.nrecv == 0) return hipSuccess;
  bool any_rho = false;
  for (int ib = 0; ib < h->nblk && rhos; ib++) any_rho |= rhos[ib] != nullptr;
  if (!o.ordered) return overset_t<T>(s, h, ys, rhos, any_rho, o.buf);
  a.t = ov_tables<T>(h, ys, rhos);
  a.rb = o.q_rb;
  a.rl = o.q_rl;
  a.db = o.q_db;
  a.dl = o.q_dl;
  a.coef5 = o.q_coef5;
  a.buf = o.buf;
  a.done = o.done;
  a.nrecv = o.nrecv;
  a.nheld = o.nheld;
  a.nuse = o.nuse;
  a.nearly = o.nearly;
  a.rpw = OV_T / a.t.nv;
  a.with_rho = any_rho ? 1 : 0;
  a.gi = 1.0 / h->cfg.gamma;
  const int wg = a.start[a.nf] + std::max((o.nearly + a.rpw - 1) / a.rpw, 1);
  if (h->fd.sb == 3) hipLaunchKernelGGL((k_boundary<T, 2>), dim3(wg), dim3(OV_T), 0, s, a);
  else hipLaunchKernelGGL((k_boundary<T, 8>), dim3(wg), dim3(OV_T), 0, s, a);
  return hipGetLastError();
}

// buf_index selects the state buffer (Y[k]) of every block.
hipError_t boundary_phase(hipStream_t s, lee_handle *h, bool fp32, int buf_index, bool with_rho, double he) {
  // the largest handles without receivers are batches: no table of blocks
  if (h->ov.nrecv == 0) {
    for (int ib = 0; ib < h->nblk; ib++) {
      Block &b = h->b[ib];
      if (b.faces.empty()) continue;
      const bool rho = with_rho && !b.uniform_mean;
      const hipError_t e = apply_bcs(s, h, b, b.Y64[buf_index], b.Y32[buf_index], fp32, rho ? b.rho64 : nullptr,
                                     rho ? b.rho32 : nullptr, he);
      if (e != hipSuccess) return e;
    }
    return hipSuccess;
  }
  auto run = [&](auto Y, auto rho) {
    std::remove_reference_t<decltype(Y(h->b[0]))> ys[MAX_OV_BLOCKS], rh[MAX_OV_BLOCKS];
    for (int ib = 0; ib < h->nblk; ib++) {
      ys[ib] = Y(h->b[ib]);
      rh[ib] = with_rho && !h->b[ib].uniform_mean ? rho(h->b[ib]) : nullptr;
    }
    return boundary_phase_t(s, h, ys, rh, he);
  };
  if (fp32)
    return run([&](Block &b) { return b.Y32[buf_index]; }, [](Block &b) { return b.rho32; });
  return run([&](Block &b) { return b.Y64[buf_index]; }, [](Block &b) { return b.rho64; });
}

}  // namespace lee
