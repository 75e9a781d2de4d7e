// HIP kernels of the LEE time advance for gfx950 (CDNA4).
//
// Fused path: one LDS-tiled kernel per RK stage (both directional
// derivatives of the four active variables, chain rule with FP64 metrics,
// LEE right-hand side, source, sponge, RK update, aux density) and one
// kernel per step for the two filter sweeps + blend + hole reset, templated
// on the bulk type (double or float); and batched ensembles of them.  The
// plain path is in lee_plain.hip, the boundary phase in lee_boundary.hip.
//
// All global indices are bounds-checked against the block extents.
#include <hip/hip_runtime.h>

#include <cmath>

#include "lee_args.h"
#include "lee_device.h"
#include "lee_internal.h"
#include "lee_stage.h"

namespace lee {

namespace {

// ------------------------------------------------------------------ fused

// INNER: the tile and its halo lie inside a block without holes (interior
// stencils only, no bounds tests); stage_tile below picks the instance.
// W: the derivative operator, OA4 (4, compile-time rows, halo 2) or FDO11P
// (11, rows from a.fdw, halo 6).
// The global loads of one stage tile, held in registers: the tile values
// with their halo (rows ty + 4k, k < KR; columns tx and, for tx < 2H,
// 64 + tx) and the per-point operands of rows ty + 4k (k < R).
template <typename T, int R, int W>
struct StageRegs {
  static constexpr int H = StageOp<W>::H, KR = (4 * R + 2 * H) / 4;
  T ta[4][KR], tb[4][KR];
  double pm[R][4], pj[R];
  T pacc[R][4], pyn[R][4];
};

// (1)-(2): the loads of a tile.  INNER: the tile and its halo lie inside the
// block (no bounds tests); the checked form reads the same values for such
// a tile.
template <typename T, int KIND, int R, bool INNER, int W = 4, typename AT>
__device__ __forceinline__ void stage_load(const AT &a, int tile, StageRegs<T, R, W> &g) {
  constexpr int TY = 4 * R;
  constexpr int H = StageOp<W>::H;
  constexpr int KR = StageRegs<T, R, W>::KR;
  static_assert(TY + 2 * H == 4 * KR, "tile rows and the halo come in fours");
  const int tx = threadIdx.x, ty = threadIdx.y;
  const int i0 = (tile % a.ntx) * ST_TX, j0 = (tile / a.ntx) * TY;
  const int ni = a.ni, nj = a.nj, n = ni * nj;
  const int VOFF[4] = {IS * n, IUX * n, IUY * n, IP * n};
  constexpr bool inner = INNER;
  const bool xtra = tx < 2 * H;
#pragma unroll
  for (int k = 0; k < KR; k++) {
    const int gj = j0 - H + ty + 4 * k;
    const bool rowok = inner || (gj >= 0 && gj < nj);
    const int gia = i0 - H + tx, gib = i0 - H + ST_TX + tx;
    const bool oka = inner || (rowok && gia >= 0 && gia < ni), okb = xtra && (inner || (rowok && gib < ni));
    const int qa = gj * ni + gia, qb = gj * ni + gib;
#pragma unroll
    for (int v = 0; v < 4; v++) {
      g.ta[v][k] = oka ? a.yin[VOFF[v] + qa] : (T)0;
      g.tb[v][k] = okb ? a.yin[VOFF[v] + qb] : (T)0;
    }
  }
  const int gi = i0 + tx;
#pragma unroll
  for (int k = 0; k < R; k++) {
    const int gj = j0 + ty + 4 * k;
    const bool ok = inner || (gi < ni && gj < nj);
    const int p = ok ? gj * ni + gi : 0;
#pragma unroll
    for (int q = 0; q < 4; q++) g.pm[k][q] = ok ? a.met[(size_t)q * n + p] : 0.0;
    g.pj[k] = ok ? a.jac[p] : 0.0;
#pragma unroll
    for (int v = 0; v < 4; v++) {
      g.pacc[k][v] = (KIND != STAGE_FIRST && ok) ? a.acc[VOFF[v] + p] : (T)0;
      g.pyn[k][v] = (KIND == STAGE_MID && ok) ? a.yn[VOFF[v] + p] : (T)0;
    }
  }
}

// (3)-(4): the tile's values through LDS, the derivatives, right-hand side,
// source, sponges and RK update of its points, from the loaded registers.
template <typename T, bool MEANF, bool HOLES, int KIND, int R, bool INNER, int W = 4, typename AT>
__device__ __forceinline__ void stage_finish(const AT &a, const StepT<T> &sc, int tile, const StageRegs<T, R, W> &g,
                                             StageLdsW<T, R, W> &s) {
  // every fusion is written out (fmx): the interior and edge instances of
  // this tile, and the batched kernels, round alike
#pragma clang fp contract(off)
  constexpr int TY = 4 * R;
  constexpr int H = StageOp<W>::H, NBC = StageOp<W>::NB;
  constexpr int KR = StageRegs<T, R, W>::KR;
  constexpr int RS = ST_TX + 2 * H;
  const int tx = threadIdx.x, ty = threadIdx.y;
  const int i0 = (tile % a.ntx) * ST_TX, j0 = (tile / a.ntx) * TY;
  const int ni = a.ni, nj = a.nj, n = ni * nj;
  const int VOFF[4] = {IS * n, IUX * n, IUY * n, IP * n};
  constexpr bool inner = INNER;
  const bool xtra = tx < 2 * H;
  const int gi = i0 + tx;
  const auto &ta = g.ta;
  const auto &tb = g.tb;
  const auto &pm = g.pm;
  const auto &pj = g.pj;
  const auto &pacc = g.pacc;
  const auto &pyn = g.pyn;
  // (3) tile to LDS
#pragma unroll
  for (int k = 0; k < KR; k++) {
    const int r = ty + 4 * k;
#pragma unroll
    for (int v = 0; v < 4; v++) {
      s[v][r][tx] = ta[v][k];
      if (xtra) s[v][r][ST_TX + tx] = tb[v][k];
    }
  }
  __syncthreads();

  // (4) the R points
#pragma unroll
  for (int k = 0; k < R; k++) {
    const int rr = ty + 4 * k;
    const int gj = j0 + rr;
    if (!inner && (gi >= ni || gj >= nj)) continue;
    const int p = gj * ni + gi;
    const int lj = rr + H, li = tx + H;
    int cx = CODE_INTERIOR, cy = CODE_INTERIOR;
    if (HOLES) {
      cx = a.code[p];
      cy = a.code[n + p];
    } else if (!inner) {
      cx = default_code(gi, ni, NBC);
      cy = default_code(gj, nj, NBC);
    }
    T dx[4], dy[4], yc[4];
#pragma unroll
    for (int v = 0; v < 4; v++) {
      const T *sp = &s[v][lj][li];
      yc[v] = sp[0];
      if constexpr (W == 4) {
        dx[v] = fd_row<T>(sp, 1, cx);
        dy[v] = fd_row<T>(sp, RS, cy);
      } else {
        dx[v] = wide_row<T>(sp, 1, cx, a.fdw);
        dy[v] = wide_row<T>(sp, RS, cy, a.fdw);
      }
    }
    T r[4];
    stage_rhs<T, MEANF, KIND == STAGE_FIRST>(a, sc.s1, sc.s2, a.he, gi, gj, p, n, pm[k], pj[k], yc, dx, dy, r);
    // RK stage update (temporal:208-230)
    const bool hole = HOLES && a.iblank[p] == BLANKED;
#pragma unroll
    for (int v = 0; v < 4; v++) {
      const size_t q = (size_t)VOFF[v] + p;
      T accv = 0, outv = 0;
      if (!hole) {
        const T rh = r[v] * sc.h;
        const T acc_in = KIND == STAGE_FIRST ? yc[v] : pacc[k][v];
        accv = fmx(sc.b, rh, acc_in);
        if (KIND != STAGE_LAST) {
          const T yn = KIND == STAGE_FIRST ? yc[v] : pyn[k][v];
          outv = fmx(sc.a, rh, yn);
        }
      }
      a.acc[q] = accv;
      if (KIND != STAGE_LAST) a.yout[q] = outv;
      r[v] = accv;
    }
    if (MEANF && KIND == STAGE_LAST) a.rho_out[p] = fmx(r[3], a.mc[MC_RP * n + p], -(r[0] * a.mc[MC_RB * n + p]));
  }
}

template <typename T, bool MEANF, bool HOLES, int KIND, int R, bool INNER, int W = 4, typename AT>
__device__ __forceinline__ void stage_tile_k(const AT &a, const StepT<T> &sc, int tile, StageLdsW<T, R, W> &s) {
  StageRegs<T, R, W> g;
  stage_load<T, KIND, R, INNER, W>(a, tile, g);
  stage_finish<T, MEANF, HOLES, KIND, R, INNER, W>(a, sc, tile, g, s);
}

template <typename T, bool MEANF, bool HOLES, int KIND, int R, int W = 4, typename AT>
__device__ __forceinline__ void stage_tile(const AT &a, const StepT<T> &sc, int tile, StageLdsW<T, R, W> &s) {
  constexpr int TY = 4 * R, H = StageOp<W>::H;
  const int i0 = (tile % a.ntx) * ST_TX, j0 = (tile / a.ntx) * TY;
  if constexpr (!HOLES) {
    if (i0 >= H && i0 + ST_TX + H <= a.ni && j0 >= H && j0 + TY + H <= a.nj) {
      stage_tile_k<T, MEANF, HOLES, KIND, R, true, W>(a, sc, tile, s);
      return;
    }
  } else {
    // a tile of a block with holes whose points all take the interior
    // stencil (no hole, no closure row) runs the interior instance
    if (a.clean && box_clean(a.clean, a.ni, a.nj, i0, i0 + ST_TX, j0, j0 + TY)) {
      stage_tile_k<T, MEANF, false, KIND, R, true, W>(a, sc, tile, s);
      return;
    }
  }
  stage_tile_k<T, MEANF, HOLES, KIND, R, false, W>(a, sc, tile, s);
}

template <typename T, bool MEANF, bool HOLES, int KIND, int R, int W = 4>
__global__ void __launch_bounds__(TPB) k_fused_stage(StageArgs<T> a) {
  __shared__ StageLdsW<T, R, W> s;
  const int tile = xcd_tile(blockIdx.x, a.chunk);
  if (tile >= a.ntiles) return;
  const StepT<T> sc{a.h, a.b, a.a, a.s1, a.s2};
  stage_tile<T, MEANF, HOLES, KIND, R, W>(a, sc, tile, s);
}

// Two blocks of one handle in one launch (an overset pair such as a
// background grid and a body grid): block 0's tiles, then block 1's, as one
// XCD-mapped list, each tile with its block's operands.  Every point runs
// the single-block arithmetic, so the results are those of two launches;
// the small block no longer costs a launch of its own.
template <typename T, bool MEANF, bool HOLES, int KIND, int R>
__global__ void __launch_bounds__(TPB) k_fused_stage_pair(StageArgs<T> a0, StageArgs<T> a1) {
  __shared__ StageLdsW<T, R, 4> s;
  const int total = a0.ntiles + a1.ntiles;
  const int tile = xcd_tile(blockIdx.x, (total + 7) / 8);
  if (tile >= total) return;
  const StepT<T> sc{a0.h, a0.b, a0.a, a0.s1, a0.s2};
  if (tile < a0.ntiles) stage_tile<T, MEANF, HOLES, KIND, R, 4>(a0, sc, tile, s);
  else stage_tile<T, MEANF, HOLES, KIND, R, 4>(a1, sc, tile - a0.ntiles, s);
}

// Batched ensemble: the tiles of all solves form one list; map[2t] is the
// solve of list entry t and map[2t + 1] its tile within the solve.  The
// list is split into eighths of `chunk` entries, one per XCD: workgroup
// (or virtual index) v maps to list position (v & 7) * chunk + (v >> 3),
// so with a grid that is a multiple of 8 each XCD works through one
// contiguous eighth of the list.  Per-solve operands come from `args`, the
// per-step scalars from `sched`, indexed by the step counter that the
// step's last kernel advances.
// The operand tables are read through the constant address space: they do
// not change during a launch, so their loads are scalar and the pointers
// loaded from them are known to address global memory (no flat accesses).
// One workgroup per list entry (the queue argument is unused: this kernel
// shares its signature with the persistent form below).
template <typename T, bool MEANF, int KIND, int R>
__global__ void __launch_bounds__(TPB)
    k_batch_stage(BatchStageArgs<T> ba, const LEE_CONST_AS StageArgs<T> *args, const LEE_CONST_AS int *map,
                  const LEE_CONST_AS BatchSched *sched, const int *__restrict__ counter, int *) {
  __shared__ StageLds<T, R> s;
  const int t = (blockIdx.x & 7) * ba.chunk + (blockIdx.x >> 3);
  if (t >= ba.total) return;
  // device-scope load: the counter was written by the previous step's filter launch
  const int step = __hip_atomic_load(counter, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  const int k = map[2 * t], local = map[2 * t + 1];
  const auto &q = sched[((size_t)step * ba.nsolve + k) * ba.nstage + ba.stage];
  const StepT<T> sc{(T)q.dt, ba.b, ba.a, q.s1, q.s2};
  stage_tile<T, MEANF, false, KIND, R>(args[k], sc, local, s);
}

// Persistent form of the batched stage (a grid smaller than the list).
// Workgroup b works on eighth b & 7 of the list (the hardware places
// workgroup b on XCD b mod 8, so each XCD keeps one contiguous eighth),
// one of the W = grid / 8 workgroups of that eighth.  The first S entries
// of the eighth (7/8 of them, whole rounds of W) are dealt out statically,
// entry w + k W to workgroup w; the rest are drawn QCH at a time from an
// atomic counter, so that the workgroups whose static share held cheap
// tiles (interior, outside sponges) take more of the remainder and the
// launch ends with the list instead of with the slowest fixed share.
// queue[QSTRIDE x] counts the draws from eighth x and queue[QSTRIDE x + 1]
// the workgroups of eighth x that have finished; the last of those resets
// both, so every launch starts from zero (each eighth has its own cache
// line).  A workgroup stops once its entry passes the eighth's end, and
// every draw advances the counter, so the loop ends.
constexpr int QCH = 2, QSTRIDE = 32;

template <typename T, bool MEANF, int KIND, int R>
__global__ void __launch_bounds__(TPB)
    k_batch_stage_q(BatchStageArgs<T> ba, const LEE_CONST_AS StageArgs<T> *args, const LEE_CONST_AS int *map,
                    const LEE_CONST_AS BatchSched *sched, const int *__restrict__ counter, int *__restrict__ queue) {
  __shared__ StageLds<T, R> s;
  __shared__ int drawn[2];
  const int step = __hip_atomic_load(counter, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  const int x = blockIdx.x & 7, lo = x * ba.chunk;
  const int n = min(ba.chunk, ba.total - lo);  // entries of this eighth (may be <= 0)
  const int W = (int)(gridDim.x >> 3), w = (int)(blockIdx.x >> 3);
  const int S = n > 0 ? (n * 7 / 8) / W * W : 0;
  int *const qx = queue + QSTRIDE * x;
  const bool lead = threadIdx.x == 0 && threadIdx.y == 0;
  // draw d goes through slot d & 1: every thread reads it right after draw
  // d's barrier, so before draw d + 1's barrier, and the lead thread writes
  // the slot again only at draw d + 2, after that barrier
  int nd = 0;
  auto draw = [&]() {
    const int slot = nd++ & 1;
    if (lead) drawn[slot] = __hip_atomic_fetch_add(qx, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __syncthreads();
    return S + QCH * drawn[slot];
  };
  auto advance = [&](int e) {
    if (e < S) return e + W < S ? e + W : draw();
    if ((e - S) % QCH != QCH - 1) return e + 1;
    return draw();
  };
  // the loads take the bounds-checked form, which reads the same values for
  // an interior tile; the finish takes the tile's own instance
  auto finish = [&](int e, const StageRegs<T, R, 4> &g) {
    const int t = lo + e;
    const int k = map[2 * t], local = map[2 * t + 1];
    const auto &q = sched[((size_t)step * ba.nsolve + k) * ba.nstage + ba.stage];
    const StepT<T> sc{(T)q.dt, ba.b, ba.a, q.s1, q.s2};
    const int i0 = (local % args[k].ntx) * ST_TX, j0 = (local / args[k].ntx) * (4 * R);
    if (i0 >= ST_H && i0 + ST_TX + ST_H <= args[k].ni && j0 >= ST_H && j0 + 4 * R + ST_H <= args[k].nj)
      stage_finish<T, MEANF, false, KIND, R, true>(args[k], sc, local, g, s);
    else
      stage_finish<T, MEANF, false, KIND, R, false>(args[k], sc, local, g, s);
  };
  int e = w < S ? w : draw();
  while (e < n) {
    const int t = lo + e;
    StageRegs<T, R, 4> g;
    stage_load<T, KIND, R, false>(args[map[2 * t]], map[2 * t + 1], g);
    finish(e, g);
    __syncthreads();  // the LDS tile is rewritten by the next entry
    e = advance(e);
  }
  if (lead) {
    const int done = __hip_atomic_fetch_add(qx + 1, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (done == W - 1) {
      __hip_atomic_store(qx, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      __hip_atomic_store(qx + 1, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
  }
}

template <typename T, bool HOLES, int ORDER, int NVAR, int TY>
__global__ void __launch_bounds__(TPB) k_fused_filter(FilterArgs<T> a) {
  __shared__ FilterLds<T, NVAR, TY, filter_halo<ORDER>()> L;
  const int tile = xcd_tile(blockIdx.x, a.chunk);
  if (tile >= a.ntiles) return;
  filter_tile<T, HOLES, ORDER, NVAR, TY>(a, tile, L);
}

// Persistent, software-pipelined form: a grid of G workgroups (G a
// multiple of 8, about one resident wave of workgroups) strides through
// the XCD-permuted tile list; each workgroup issues the global loads of its
// next tile before computing the current one, so the loads overlap the
// LDS sweeps instead of waiting for a new launch round.  Two tiles' values
// stay in registers: up to 256 VGPRs (two waves per SIMD) keep them out of
// scratch.
template <typename T, bool HOLES, int ORDER, int NVAR, int TY>
__global__ void __launch_bounds__(TPB) __attribute__((amdgpu_waves_per_eu(1, 2)))
k_fused_filter_p(FilterArgs<T> a) {
  __shared__ FilterLds<T, NVAR, TY> L;
  const int G = gridDim.x, total = 8 * a.chunk;
  auto tile_of = [&](int v) { return (v & 7) * a.chunk + (v >> 3); };
  auto live = [&](int v) { return v < total && tile_of(v) < a.ntiles; };
  // loads are issued for every slot (past the end: the last tile again) so
  // that no branch sits between a tile's loads and its use
  auto ld = [&](int v) { return min(tile_of(v), a.ntiles - 1); };
  // (the scheduling barrier keeps the compiler from sinking the prefetch
  // into the sweeps, where each load would be waited for at once; the copy
  // at the end of an iteration waits for loads that had the whole tile's
  // sweeps to arrive)
  FilterRegs<T, NVAR, TY> R;
  int v = blockIdx.x;
  filter_load<T, HOLES, NVAR, TY>(a, ld(v), R);
  for (; v < total; v += G) {
    FilterRegs<T, NVAR, TY> N;
    filter_load<T, HOLES, NVAR, TY>(a, ld(v + G), N);
    __builtin_amdgcn_sched_barrier(0);
    if (live(v)) filter_compute<T, HOLES, ORDER, NVAR, TY>(a, tile_of(v), L, R);
    __syncthreads();
    R = N;
  }
}

// Column-march form (blocks without holes): one wave per (variable, strip,
// row chunk), four waves per workgroup, no LDS (filter_march).
template <typename T, int ORDER, int L>
__global__ void __launch_bounds__(TPB) k_fused_filter_m(FilterArgs<T> a) {
  filter_march<T, ORDER, L>(a);
}

// Stacked column march (blocks without holes): NW waves per (variable,
// strip, stack of NW R rows), xi rows shared through LDS (filter_stack).
template <typename T, int ORDER, int NW, int R, bool HOLES>
__global__ void __launch_bounds__(64 * NW) k_fused_filter_s(FilterArgs<T> a) {
  __shared__ StackLds<T, NW, R> L;
  filter_stack<T, ORDER, NW, R, HOLES>(a, L);
}

// The stacked filter of two blocks in one launch (see k_fused_stage_pair).
template <typename T, int ORDER, int NW, int R, bool HOLES>
__global__ void __launch_bounds__(64 * NW) k_fused_filter_s_pair(FilterArgs<T> a0, FilterArgs<T> a1) {
  __shared__ StackLds<T, NW, R> L;
  const int total = a0.ntiles + a1.ntiles;
  const int t = xcd_tile(blockIdx.x, (total + 7) / 8);
  if (t >= total) return;
  if (t < a0.ntiles) stack_item<T, ORDER, NW, R, HOLES>(a0, t, L);
  else stack_item<T, ORDER, NW, R, HOLES>(a1, t - a0.ntiles, L);
}

template <typename T>
struct BatchFilterArgs {
  const FilterArgs<T> *args;     // nsolve entries
  const int *map;                // (solve, tile) per list entry
  int *counter;                  // advanced by one at the end of the step
  int nsolve, total, chunk;
};

// The batched filter is the last kernel of a step: one thread advances the
// step counter (no kernel of this launch reads it; the next step's stage
// kernels see the new value).
template <typename T, int ORDER, int TY>
__global__ void __launch_bounds__(TPB)
    k_batch_filter(BatchFilterArgs<T> ba, const LEE_CONST_AS FilterArgs<T> *args, const LEE_CONST_AS int *map) {
  __shared__ FilterLds<T, 4, TY> L;
  if (blockIdx.x == 0 && threadIdx.x == 0 && threadIdx.y == 0) {
    const int c = __hip_atomic_load(ba.counter, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __hip_atomic_store(ba.counter, c + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);  // vector store
  }
  for (int v = blockIdx.x; v < 8 * ba.chunk; v += gridDim.x) {
    const int t = (v & 7) * ba.chunk + (v >> 3);
    if (t >= ba.total) continue;
    filter_tile<T, false, ORDER, 4, TY>(args[map[2 * t]], map[2 * t + 1], L);
    __syncthreads();
  }
}


// Batched stacked column march (solves without holes): the list entries are
// (solve, stack) pairs; four waves of R rows per stack.
template <typename T, int ORDER, int R>
__global__ void __launch_bounds__(TPB)
    k_batch_filter_s(BatchFilterArgs<T> ba, const LEE_CONST_AS FilterArgs<T> *args, const LEE_CONST_AS int *map) {
  __shared__ StackLds<T, 4, R> L;
  if (blockIdx.x == 0 && threadIdx.x == 0 && threadIdx.y == 0) {
    const int c = __hip_atomic_load(ba.counter, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __hip_atomic_store(ba.counter, c + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);  // vector store
  }
  for (int v = blockIdx.x; v < 8 * ba.chunk; v += gridDim.x) {
    const int t = (v & 7) * ba.chunk + (v >> 3);
    if (t >= ba.total) continue;
    stack_item<T, ORDER, 4, R>(args[map[2 * t]], map[2 * t + 1], L);
    __syncthreads();  // the LDS rows are rewritten by the next stack
  }
}

// Passive w' in 2-D: only the sponge acts on it (the velocity loop of
// spatial:2077-2103 stops at num_dim), then the RK update.
template <typename T>
__global__ void __launch_bounds__(TPB) k_passive_w(StageArgs<T> a, int kind) {
  const int p = blockIdx.x * TPB + threadIdx.x;
  const int ni = a.ni, nj = a.nj, n = ni * nj;
  if (p >= n) return;
  const int gi = p % ni, gj = p / ni;
  const size_t q = (size_t)IUZ * n + p;
  const T w = a.yin[q];
  T r = 0;
  for (int z = 0; z < a.nz; z++) {
    const ZoneT<T> &zz = a.z[z];
    if (gi >= zz.i0 && gi <= zz.i1 && gj >= zz.j0 && gj <= zz.j1)
      r += -zz.sig[(gj - zz.j0) * zz.nzi + (gi - zz.i0)] * w;
  }
  if (a.iblank && a.iblank[p] == BLANKED) {
    a.acc[q] = 0;
    if (kind != STAGE_LAST) a.yout[q] = 0;
    return;
  }
  const T rh = r * a.h;
  const T acc_in = kind == STAGE_FIRST ? w : a.acc[q];
  a.acc[q] = acc_in + a.b * rh;
  if (kind != STAGE_LAST) {
    const T yn = kind == STAGE_FIRST ? w : a.yn[q];
    a.yout[q] = yn + a.a * rh;
  }
}

// One RK stage of the passive scalars of a LEE_SCALAR run, one thread per
// (scalar, point), after the stage kernel of the same buffers (it writes
// only the five LEE variables of acc and yout; this kernel only the
// scalars'): compute_RHS_linearized_Euler_scalar (spatial:2134-2158),
//   rhs_Z = -ubar dZ'/dx - u' dZbar/dx - vbar dZ'/dy - v' dZbar/dy
// in the reference's term order, the Freund sponges relaxing Z' to 0
// (source.cpp:174-201, 264-320), the RK update and the hole reset as in
// the stage kernel.  Derivative rows read the stage input in place (the
// closure rows stay inside the block); metrics, J, the mean velocity and
// the scalars' mean gradients are FP64.  W: OA4 (4) or FDO11P (11) rows.
template <typename T, int KIND, int W>
__global__ void __launch_bounds__(TPB) k_scalar_stage(StageArgs<T> a, int nsc) {
#pragma clang fp contract(off)
  const int ni = a.ni, nj = a.nj, n = ni * nj;
  const int t = blockIdx.x * TPB + threadIdx.x;
  if (t >= nsc * n) return;
  const int z = t / n, p = t - z * n;
  const int gi = p % ni, gj = p / ni;
  const size_t q = (size_t)(NV + z) * n + p;
  int cx, cy;
  if (a.code) {
    cx = a.code[p];
    cy = a.code[n + p];
  } else {
    cx = default_code(gi, ni, StageOp<W>::NB);
    cy = default_code(gj, nj, StageOp<W>::NB);
  }
  const T *sp = a.yin + q;
  T dx, dy;
  if constexpr (W == 4) {
    dx = fd_row<T>(sp, 1, cx);
    dy = fd_row<T>(sp, ni, cy);
  } else {
    dx = wide_row<T>(sp, 1, cx, a.fdw);
    dy = wide_row<T>(sp, ni, cy, a.fdw);
  }
  const double mxx = a.met[p], mxy = a.met[(size_t)n + p], myx = a.met[(size_t)2 * n + p],
               myy = a.met[(size_t)3 * n + p];
  const double J = a.jac[p];
  const T fx = (T)(fmx(mxx, (double)dx, myx * (double)dy) * J);
  const T fy = (T)(fmx(mxy, (double)dx, myy * (double)dy) * J);
  const T u0 = (T)a.mean[(size_t)IUX * n + p], v0 = (T)a.mean[(size_t)IUY * n + p];
  const T up = a.yin[(size_t)IUX * n + p], vp = a.yin[(size_t)IUY * n + p];
  const T gzx = (T)a.mgrad[(size_t)(2 * (NV + z)) * n + p], gzy = (T)a.mgrad[(size_t)(2 * (NV + z) + 1) * n + p];
  const T zc = sp[0];
  T r = -(u0 * fx);
  r = fmx(-up, gzx, r);
  r = fmx(-v0, fy, r);
  r = fmx(-vp, gzy, r);
  for (int k = 0; k < a.nz; k++) {
    const ZoneT<T> &zz = a.z[k];
    if (gi >= zz.i0 && gi <= zz.i1 && gj >= zz.j0 && gj <= zz.j1)
      r = fmx(-zz.sig[(gj - zz.j0) * zz.nzi + (gi - zz.i0)], zc, r);
  }
  T accv = 0, outv = 0;
  if (!(a.iblank && a.iblank[p] == BLANKED)) {
    const T rh = r * a.h;
    const T acc_in = KIND == STAGE_FIRST ? zc : a.acc[q];
    accv = fmx(a.b, rh, acc_in);
    if (KIND != STAGE_LAST) {
      const T yn = KIND == STAGE_FIRST ? zc : a.yn[q];
      outv = fmx(a.a, rh, yn);
    }
  }
  a.acc[q] = accv;
  if (KIND != STAGE_LAST) a.yout[q] = outv;
}

template <typename S, typename D>
__global__ void __launch_bounds__(TPB) k_cast(const S *__restrict__ a, D *__restrict__ b, size_t n) {
  const size_t p = (size_t)blockIdx.x * TPB + threadIdx.x;
  if (p < n) b[p] = (D)a[p];
}

inline unsigned nblocks(size_t n) { return (unsigned)((n + TPB - 1) / TPB); }

}  // namespace

// ------------------------------------------------------------- launchers

template <typename T>
static hipError_t fused_stage_t(hipStream_t s, lee_handle *h, Block &b, int stage, const StageScalars &sc, T *const *Y,
                                T *rho) {
  const int kind = stage_kind(h, stage);
  const bool wide = h->cfg.fd_order == 11;
  const int R = wide ? 1 : b.tune_r;  // the 11-point rows run on tiles of 4 rows
  const StageArgs<T> a = make_stage_args<T>(h, b, stage, Y, rho, R, sc);
  const dim3 grid(a.chunk * 8), block(64, 4);
  const bool mf = !b.uniform_mean, ho = b.has_holes;
#define LEE_LAUNCH(MF, HO, K)                                                                     \
  do {                                                                                            \
    if (wide) hipLaunchKernelGGL((k_fused_stage<T, MF, HO, K, 1, 11>), grid, block, 0, s, a);    \
    else if (R == 1) hipLaunchKernelGGL((k_fused_stage<T, MF, HO, K, 1>), grid, block, 0, s, a); \
    else if (R == 2) hipLaunchKernelGGL((k_fused_stage<T, MF, HO, K, 2>), grid, block, 0, s, a); \
    else hipLaunchKernelGGL((k_fused_stage<T, MF, HO, K, 4>), grid, block, 0, s, a);             \
  } while (0)
#define LEE_KINDS(MF, HO)                                      \
  do {                                                         \
    if (kind == STAGE_FIRST) LEE_LAUNCH(MF, HO, STAGE_FIRST);  \
    else if (kind == STAGE_MID) LEE_LAUNCH(MF, HO, STAGE_MID); \
    else LEE_LAUNCH(MF, HO, STAGE_LAST);                       \
  } while (0)
  if (mf && ho) LEE_KINDS(true, true);
  else if (mf) LEE_KINDS(true, false);
  else if (ho) LEE_KINDS(false, true);
  else LEE_KINDS(false, false);
#undef LEE_KINDS
#undef LEE_LAUNCH
  if (b.carry_w)
    hipLaunchKernelGGL(k_passive_w<T>, dim3(nblocks(b.n)), dim3(TPB), 0, s, a, kind);
  if (const int nsc = h->cfg.num_scalar) {
    const dim3 sg(nblocks((size_t)nsc * b.n));
#define LEE_SCALARS(K)                                                                              \
  do {                                                                                              \
    if (wide) hipLaunchKernelGGL((k_scalar_stage<T, K, 11>), sg, dim3(TPB), 0, s, a, nsc);          \
    else hipLaunchKernelGGL((k_scalar_stage<T, K, 4>), sg, dim3(TPB), 0, s, a, nsc);                \
  } while (0)
    if (kind == STAGE_FIRST) LEE_SCALARS(STAGE_FIRST);
    else if (kind == STAGE_MID) LEE_SCALARS(STAGE_MID);
    else LEE_SCALARS(STAGE_LAST);
#undef LEE_SCALARS
  }
  return hipGetLastError();
}

hipError_t fused_stage(hipStream_t s, lee_handle *h, Block &b, int stage, const StageScalars &sc) {
  if (h->cfg.precision == LEE_FP32) return fused_stage_t<float>(s, h, b, stage, sc, b.Y32, b.rho32);
  return fused_stage_t<double>(s, h, b, stage, sc, b.Y64, b.rho64);
}

// Whether a 2-D handle's two blocks can share one stage launch and one
// filter launch: the same kernel instance (holes, mean kind, operator) and
// the same tile height; the filter also needs both blocks in the same
// stacked column-march form.
bool pair_stage_ok(const lee_handle *h) {
  if (h->nblk != 2 || h->batch || h->cfg.num_dim != 2 || h->cfg.fd_order != 4 || h->cfg.path != LEE_PATH_FUSED)
    return false;
  const Block &b0 = h->b[0], &b1 = h->b[1];
  return b0.has_holes == b1.has_holes && b0.uniform_mean == b1.uniform_mean && b0.tune_r == b1.tune_r;
}

bool pair_filter_ok(const lee_handle *h) {
  if (!pair_stage_ok(h) || h->cfg.filter_order == 11 || h->cfg.filter_order == 0) return false;
  const Block &b0 = h->b[0], &b1 = h->b[1];
  return b0.tune_mc > 1 && b0.tune_mc == b1.tune_mc && b0.tune_ml == b1.tune_ml && !b0.carry_w && !b1.carry_w;
}

template <typename T>
static hipError_t fused_stage_pair_t(hipStream_t s, lee_handle *h, int stage, const StageScalars &sc) {
  Block &b0 = h->b[0], &b1 = h->b[1];
  const int kind = stage_kind(h, stage), R = b0.tune_r;
  T *const *Y0 = sizeof(T) == 8 ? (T *const *)b0.Y64 : (T *const *)b0.Y32;
  T *const *Y1 = sizeof(T) == 8 ? (T *const *)b1.Y64 : (T *const *)b1.Y32;
  T *r0 = sizeof(T) == 8 ? (T *)b0.rho64 : (T *)b0.rho32;
  T *r1 = sizeof(T) == 8 ? (T *)b1.rho64 : (T *)b1.rho32;
  const StageArgs<T> a0 = make_stage_args<T>(h, b0, stage, Y0, r0, R, sc);
  const StageArgs<T> a1 = make_stage_args<T>(h, b1, stage, Y1, r1, R, sc);
  const dim3 grid((a0.ntiles + a1.ntiles + 7) / 8 * 8), block(64, 4);
  const bool mf = !b0.uniform_mean, ho = b0.has_holes;
#define LEE_PL(MF, HO, K)                                                                              \
  do {                                                                                                 \
    if (R == 1) hipLaunchKernelGGL((k_fused_stage_pair<T, MF, HO, K, 1>), grid, block, 0, s, a0, a1); \
    else if (R == 2) hipLaunchKernelGGL((k_fused_stage_pair<T, MF, HO, K, 2>), grid, block, 0, s, a0, a1); \
    else hipLaunchKernelGGL((k_fused_stage_pair<T, MF, HO, K, 4>), grid, block, 0, s, a0, a1);         \
  } while (0)
#define LEE_PK(MF, HO)                                     \
  do {                                                     \
    if (kind == STAGE_FIRST) LEE_PL(MF, HO, STAGE_FIRST);  \
    else if (kind == STAGE_MID) LEE_PL(MF, HO, STAGE_MID); \
    else LEE_PL(MF, HO, STAGE_LAST);                       \
  } while (0)
  if (mf && ho) LEE_PK(true, true);
  else if (mf) LEE_PK(true, false);
  else if (ho) LEE_PK(false, true);
  else LEE_PK(false, false);
#undef LEE_PK
#undef LEE_PL
  // the per-block extras of fused_stage_t: a carried w' and the passive scalars
  for (int ib = 0; ib < 2; ib++) {
    Block &b = h->b[ib];
    const StageArgs<T> &a = ib == 0 ? a0 : a1;
    if (b.carry_w) hipLaunchKernelGGL(k_passive_w<T>, dim3(nblocks(b.n)), dim3(TPB), 0, s, a, kind);
    if (const int nsc = h->cfg.num_scalar) {
      const dim3 sg(nblocks((size_t)nsc * b.n));
      if (kind == STAGE_FIRST) hipLaunchKernelGGL((k_scalar_stage<T, STAGE_FIRST, 4>), sg, dim3(TPB), 0, s, a, nsc);
      else if (kind == STAGE_MID) hipLaunchKernelGGL((k_scalar_stage<T, STAGE_MID, 4>), sg, dim3(TPB), 0, s, a, nsc);
      else hipLaunchKernelGGL((k_scalar_stage<T, STAGE_LAST, 4>), sg, dim3(TPB), 0, s, a, nsc);
    }
  }
  return hipGetLastError();
}

hipError_t fused_stage_pair(hipStream_t s, lee_handle *h, int stage, const StageScalars &sc) {
  if (h->cfg.precision == LEE_FP32) return fused_stage_pair_t<float>(s, h, stage, sc);
  return fused_stage_pair_t<double>(s, h, stage, sc);
}

// Operands of the filter on block b with tile height TYF (four variables).
template <typename T>
static FilterArgs<T> make_filter_args(const lee_handle *h, const Block &b, T *const *Y, int src, int dst, int TYF) {
  FilterArgs<T> a{};
  a.ni = b.ni;
  a.nj = b.nj;
  a.ntx = (b.ni + FL_TX - 1) / FL_TX;
  a.nty = (b.nj + TYF - 1) / TYF;
  a.ntiles = a.ntx * a.nty;
  a.chunk = (a.ntiles + 7) / 8;
  a.src = Y[src];
  a.dst = Y[dst];
  a.iblank = b.iblank;
  a.code = b.code_flt;
  a.clean = b.clean_flt;
  a.blend = (T)h->cfg.filter_blend;
  a.rem = (T)(1.0 - h->cfg.filter_blend);
  a.vars[0] = IS;
  a.vars[1] = IUX;
  a.vars[2] = IUY;
  a.vars[3] = IP;
  a.flw = h->flw;
  return a;
}

template <typename T>
static hipError_t fused_filter_t(hipStream_t s, lee_handle *h, Block &b, T *const *Y, int src, int dst) {
  const int TYF = b.tune_fty;
  FilterArgs<T> a = make_filter_args<T>(h, b, Y, src, dst, TYF);
  const dim3 grid(a.chunk * 8), block(64, 4);
  // persistent pipelined form: tune_fgrid workgroups (a multiple of 8) stride over the tiles
  const bool pipe = b.tune_fgrid > 0;
  const dim3 pgrid(std::min(a.chunk * 8, (b.tune_fgrid + 7) / 8 * 8));
  const bool o8 = h->cfg.filter_order == 8;
  if (h->cfg.filter_order == 11) {  // SFO11P: the tile form, tiles of 4 or 8 rows, halo 6
    for (int pass = 0; pass < (b.carry_w ? 2 : 1); pass++) {
      const bool four = pass == 0;
      if (!four) a.vars[0] = IUZ;
#define LEE_FLW(HO, NVV)                                                                                  \
  do {                                                                                                    \
    if (TYF == 4) hipLaunchKernelGGL((k_fused_filter<T, HO, 11, NVV, 4>), grid, block, 0, s, a);          \
    else hipLaunchKernelGGL((k_fused_filter<T, HO, 11, NVV, 8>), grid, block, 0, s, a);                   \
  } while (0)
      if (b.has_holes) {
        if (four) LEE_FLW(true, 4);
        else LEE_FLW(true, 1);
      } else {
        if (four) LEE_FLW(false, 4);
        else LEE_FLW(false, 1);
      }
#undef LEE_FLW
    }
    return hipGetLastError();
  }
  if (b.tune_mc > 0 && (!b.has_holes || b.tune_mc > 1)) {
    // column-march forms: every carried variable in one launch
    const int nv = b.carry_w ? 5 : 4;
    a.vars[4] = IUZ;
    const int NW = b.tune_mc, L = b.tune_ml;
    a.ntx = (b.ni + March::STRIDE - 1) / March::STRIDE;
    a.nty = (b.nj + NW * L - 1) / (NW * L);
    a.ntiles = nv * a.ntx * a.nty;  // waves (single-wave form) or stacks
    a.chunk = NW == 1 ? ((a.ntiles + 3) / 4 + 7) / 8 : (a.ntiles + 7) / 8;
    const dim3 mgrid(a.chunk * 8), sblock(64, NW == 1 ? 4 : NW);
#define LEE_FLM(OR, LL) hipLaunchKernelGGL((k_fused_filter_m<T, OR, LL>), mgrid, sblock, 0, s, a)
#define LEE_FLS(OR, NWV, RR)                                                                              \
  do {                                                                                                    \
    if (b.has_holes) hipLaunchKernelGGL((k_fused_filter_s<T, OR, NWV, RR, true>), mgrid, sblock, 0, s, a); \
    else hipLaunchKernelGGL((k_fused_filter_s<T, OR, NWV, RR, false>), mgrid, sblock, 0, s, a);            \
  } while (0)
#define LEE_FLM_O(OR)                              \
  do {                                             \
    if (NW == 1 && L == 8) LEE_FLM(OR, 8);         \
    else if (NW == 1) LEE_FLM(OR, 16);             \
    else if (NW == 8) LEE_FLS(OR, 8, 8);           \
    else if (L == 4) LEE_FLS(OR, 4, 4);            \
    else if (L == 8) LEE_FLS(OR, 4, 8);            \
    else LEE_FLS(OR, 4, 16);                       \
  } while (0)
    if (o8) LEE_FLM_O(8);
    else LEE_FLM_O(4);
#undef LEE_FLM_O
#undef LEE_FLS
#undef LEE_FLM
    return hipGetLastError();
  }
  // the four active variables together, then w' alone when it is carried
  for (int pass = 0; pass < (b.carry_w ? 2 : 1); pass++) {
    const bool four = pass == 0;
    if (!four) a.vars[0] = IUZ;
#define LEE_FLT1(HO, OR, NVV, TYV)                                                                       \
  do {                                                                                                   \
    if (pipe) hipLaunchKernelGGL((k_fused_filter_p<T, HO, OR, NVV, TYV>), pgrid, block, 0, s, a);        \
    else hipLaunchKernelGGL((k_fused_filter<T, HO, OR, NVV, TYV>), grid, block, 0, s, a);                \
  } while (0)
#define LEE_FLT(HO, OR, NVV)            \
  do {                                  \
    if (TYF == 4) LEE_FLT1(HO, OR, NVV, 4);  \
    else if (TYF == 8) LEE_FLT1(HO, OR, NVV, 8); \
    else if (TYF == 12) LEE_FLT1(HO, OR, NVV, 12); \
    else LEE_FLT1(HO, OR, NVV, 16);      \
  } while (0)
#define LEE_FLT_NV(HO, OR)            \
  do {                                \
    if (four) LEE_FLT(HO, OR, 4);     \
    else LEE_FLT(HO, OR, 1);          \
  } while (0)
    if (b.has_holes) {
      if (o8) LEE_FLT_NV(true, 8);
      else LEE_FLT_NV(true, 4);
    } else {
      if (o8) LEE_FLT_NV(false, 8);
      else LEE_FLT_NV(false, 4);
    }
#undef LEE_FLT_NV
#undef LEE_FLT
#undef LEE_FLT1
  }
  return hipGetLastError();
}

// The passive scalars of a LEE_SCALAR run (apply_filter filters every
// solution variable, spatial:2191-2246): one tile-form launch of one
// variable each, tiles of 8 rows (every filter form computes each point
// with the same operations).
template <typename T>
static hipError_t scalar_filter_t(hipStream_t s, lee_handle *h, Block &b, T *const *Y, int src, int dst) {
  FilterArgs<T> a = make_filter_args<T>(h, b, Y, src, dst, 8);
  const dim3 grid(a.chunk * 8), block(64, 4);
  const int o = h->cfg.filter_order;
  for (int z = 0; z < h->cfg.num_scalar; z++) {
    a.vars[0] = NV + z;
#define LEE_FLZ(HO)                                                                       \
  do {                                                                                    \
    if (o == 11) hipLaunchKernelGGL((k_fused_filter<T, HO, 11, 1, 8>), grid, block, 0, s, a); \
    else if (o == 8) hipLaunchKernelGGL((k_fused_filter<T, HO, 8, 1, 8>), grid, block, 0, s, a); \
    else hipLaunchKernelGGL((k_fused_filter<T, HO, 4, 1, 8>), grid, block, 0, s, a);   \
  } while (0)
    if (b.has_holes) LEE_FLZ(true);
    else LEE_FLZ(false);
#undef LEE_FLZ
  }
  return hipGetLastError();
}

// Both blocks of a pair (pair_filter_ok) in one stacked column-march launch.
template <typename T>
static hipError_t fused_filter_pair_t(hipStream_t s, lee_handle *h, int src, int dst) {
  Block &b0 = h->b[0], &b1 = h->b[1];
  const int NW = b0.tune_mc, L = b0.tune_ml;
  FilterArgs<T> a[2];
  for (int ib = 0; ib < 2; ib++) {
    Block &b = h->b[ib];
    T *const *Y = sizeof(T) == 8 ? (T *const *)b.Y64 : (T *const *)b.Y32;
    a[ib] = make_filter_args<T>(h, b, Y, src, dst, b.tune_fty);
    a[ib].ntx = (b.ni + March::STRIDE - 1) / March::STRIDE;
    a[ib].nty = (b.nj + NW * L - 1) / (NW * L);
    a[ib].ntiles = 4 * a[ib].ntx * a[ib].nty;  // stacks of the four active variables
    a[ib].chunk = (a[ib].ntiles + 7) / 8;
  }
  const dim3 grid((a[0].ntiles + a[1].ntiles + 7) / 8 * 8), block(64, NW);
  const bool ho = b0.has_holes, o8 = h->cfg.filter_order == 8;
#define LEE_FP(OR, NWV, RR)                                                                                      \
  do {                                                                                                           \
    if (ho) hipLaunchKernelGGL((k_fused_filter_s_pair<T, OR, NWV, RR, true>), grid, block, 0, s, a[0], a[1]);   \
    else hipLaunchKernelGGL((k_fused_filter_s_pair<T, OR, NWV, RR, false>), grid, block, 0, s, a[0], a[1]);     \
  } while (0)
#define LEE_FP_O(OR)                    \
  do {                                  \
    if (NW == 8) LEE_FP(OR, 8, 8);      \
    else if (L == 4) LEE_FP(OR, 4, 4);  \
    else if (L == 8) LEE_FP(OR, 4, 8);  \
    else LEE_FP(OR, 4, 16);             \
  } while (0)
  if (o8) LEE_FP_O(8);
  else LEE_FP_O(4);
#undef LEE_FP_O
#undef LEE_FP
  hipError_t e = hipGetLastError();
  for (int ib = 0; ib < 2 && e == hipSuccess && h->cfg.num_scalar; ib++) {
    Block &b = h->b[ib];
    T *const *Y = sizeof(T) == 8 ? (T *const *)b.Y64 : (T *const *)b.Y32;
    e = scalar_filter_t<T>(s, h, b, Y, src, dst);
  }
  return e;
}

hipError_t fused_filter_pair(hipStream_t s, lee_handle *h, int src, int dst) {
  if (h->cfg.precision == LEE_FP32) return fused_filter_pair_t<float>(s, h, src, dst);
  return fused_filter_pair_t<double>(s, h, src, dst);
}

hipError_t fused_filter(hipStream_t s, lee_handle *h, Block &b, int src, int dst) {
  const bool f32 = h->cfg.precision == LEE_FP32;
  hipError_t e = f32 ? fused_filter_t<float>(s, h, b, b.Y32, src, dst) : fused_filter_t<double>(s, h, b, b.Y64, src, dst);
  if (e != hipSuccess || h->cfg.num_scalar == 0) return e;
  return f32 ? scalar_filter_t<float>(s, h, b, b.Y32, src, dst) : scalar_filter_t<double>(s, h, b, b.Y64, src, dst);
}

// ------------------------------------------------------------ batched ensemble

void batch_release(lee_handle *h) {
  BatchPlan &p = h->bp;
  if (p.exec) (void)hipGraphExecDestroy(p.exec);
  p.exec = nullptr;
  for (void *q : {p.stage_args, p.filter_args, p.pair_args, (void *)p.tile_map_stage, (void *)p.tile_map_filter,
                  (void *)p.tile_map_pair})
    if (q) (void)hipFree(q);
  p.stage_args = p.filter_args = p.pair_args = nullptr;
  p.tile_map_stage = p.tile_map_filter = p.tile_map_pair = nullptr;
  p.ready = false;
}

// Uploads the per-solve operand tables of every stage and of the filter for
// the current tile shape, and the tile prefix sums.  The schedule and the
// step counter are allocated by the caller.
// With p.tuning the tables describe runs on scratch buffers only (stages: Y2
// -> Y3 and Y1; filter: Y1 -> Y2), so the autotuner can time launches without
// touching the state in Y0.
template <typename T>
static void batch_resident_t(lee_handle *h);

template <typename T>
static hipError_t batch_prepare_t(hipStream_t s, lee_handle *h) {
  BatchPlan &p = h->bp;
  const int ns = h->nblk, S = h->cfg.rk_stages;
  std::vector<StageArgs<T>> sa((size_t)S * ns);
  std::vector<FilterArgs<T>> fa(ns);
  std::vector<int> ts, tf;
  const StageScalars zero{0.0, 0.0, 0.0, 0.0, 0.0};
  for (int k = 0; k < ns; k++) {
    Block &b = h->b[k];
    T *const *Y = sizeof(T) == 8 ? (T *const *)b.Y64 : (T *const *)b.Y32;
    T *rho = sizeof(T) == 8 ? (T *)b.rho64 : (T *)b.rho32;
    for (int st = 0; st < S; st++)
      sa[(size_t)st * ns + k] = make_stage_args<T>(h, b, p.tuning ? (st == 0 ? -2 : (st == S - 1 ? -3 : -1)) : st, Y, rho, p.R, zero);
    fa[k] = make_filter_args<T>(h, b, Y, 1, p.tuning ? 2 : 0, p.TY);
    if (p.stack) {  // stacks of four waves of p.stack rows, four variables
      fa[k].ntx = (b.ni + March::STRIDE - 1) / March::STRIDE;
      fa[k].nty = (b.nj + 4 * p.stack - 1) / (4 * p.stack);
      fa[k].ntiles = 4 * fa[k].ntx * fa[k].nty;
    }
    for (int t = 0; t < sa[k].ntiles; t++) {
      ts.push_back(k);
      ts.push_back(t);
    }
    for (int t = 0; t < fa[k].ntiles; t++) {
      tf.push_back(k);
      tf.push_back(t);
    }
  }
  p.total_stage = (int)(ts.size() / 2);
  p.total_filter = (int)(tf.size() / 2);
  hipError_t e;
  if ((e = hipMalloc(&p.stage_args, sizeof(StageArgs<T>) * sa.size())) != hipSuccess) return e;
  if ((e = hipMalloc(&p.filter_args, sizeof(FilterArgs<T>) * fa.size())) != hipSuccess) return e;
  if ((e = hipMalloc((void **)&p.tile_map_stage, sizeof(int) * ts.size())) != hipSuccess) return e;
  if ((e = hipMalloc((void **)&p.tile_map_filter, sizeof(int) * tf.size())) != hipSuccess) return e;
  if ((e = hipMemcpyAsync(p.stage_args, sa.data(), sizeof(StageArgs<T>) * sa.size(), hipMemcpyHostToDevice, s)))
    return e;
  if ((e = hipMemcpyAsync(p.filter_args, fa.data(), sizeof(FilterArgs<T>) * fa.size(), hipMemcpyHostToDevice, s)))
    return e;
  if ((e = hipMemcpyAsync(p.tile_map_stage, ts.data(), sizeof(int) * ts.size(), hipMemcpyHostToDevice, s)))
    return e;
  if ((e = hipMemcpyAsync(p.tile_map_filter, tf.data(), sizeof(int) * tf.size(), hipMemcpyHostToDevice, s)))
    return e;
  // the host vectors die here: wait for the copies
  if ((e = hipStreamSynchronize(s)) != hipSuccess) return e;
  batch_resident_t<T>(h);
  return hipSuccess;
}

hipError_t batch_prepare(hipStream_t s, lee_handle *h) {
  batch_release(h);
  hipError_t e = h->cfg.precision == LEE_FP32 ? batch_prepare_t<float>(s, h) : batch_prepare_t<double>(s, h);
  if (e == hipSuccess && h->bp.pair) e = batch_pair_prepare(s, h);
  // ready once every table that a launch reads is there: all of them or none
  if (e == hipSuccess) h->bp.ready = true;
  else batch_release(h);
  return e;
}

// Grid of a batch launch over `total` list entries: one workgroup per entry
// (setting 0, or a setting at least that large), a persistent grid of the
// given size rounded up to a multiple of 8, or (LEE_GRID_RESIDENT) the
// workgroups the device holds at once for that kernel.
static unsigned batch_grid(int total, int setting, int resident) {
  const int chunk = (total + 7) / 8;
  const int full = 8 * chunk;
  const int g = setting == LEE_GRID_RESIDENT ? resident : setting;
  if (g <= 0 || g >= full) return (unsigned)full;
  return (unsigned)((g + 7) / 8 * 8);
}

template <typename T>
using BatchStageFn = void (*)(BatchStageArgs<T>, const LEE_CONST_AS StageArgs<T> *, const LEE_CONST_AS int *,
                              const LEE_CONST_AS BatchSched *, const int *, int *);
template <typename T>
using BatchFilterFn = void (*)(BatchFilterArgs<T>, const LEE_CONST_AS FilterArgs<T> *, const LEE_CONST_AS int *);

// queued: the persistent work-queue kernel (a grid smaller than the list)
template <typename T, bool MF, int K>
static BatchStageFn<T> batch_stage_fn_r(int R, bool queued) {
  if (queued) {
    if (R == 1) return k_batch_stage_q<T, MF, K, 1>;
    if (R == 2) return k_batch_stage_q<T, MF, K, 2>;
    return k_batch_stage_q<T, MF, K, 4>;
  }
  if (R == 1) return k_batch_stage<T, MF, K, 1>;
  if (R == 2) return k_batch_stage<T, MF, K, 2>;
  return k_batch_stage<T, MF, K, 4>;
}

template <typename T, bool MF>
static BatchStageFn<T> batch_stage_fn_k(int kind, int R, bool queued) {
  if (kind == STAGE_FIRST) return batch_stage_fn_r<T, MF, STAGE_FIRST>(R, queued);
  if (kind == STAGE_MID) return batch_stage_fn_r<T, MF, STAGE_MID>(R, queued);
  return batch_stage_fn_r<T, MF, STAGE_LAST>(R, queued);
}

template <typename T>
static BatchStageFn<T> batch_stage_fn(const lee_handle *h, int kind, bool queued) {
  const int R = h->bp.R;
  return h->b[0].uniform_mean ? batch_stage_fn_k<T, false>(kind, R, queued)
                              : batch_stage_fn_k<T, true>(kind, R, queued);
}

template <typename T, int OR>
static BatchFilterFn<T> batch_filter_fn_o(const BatchPlan &p) {
  if (p.stack == 4) return k_batch_filter_s<T, OR, 4>;
  if (p.stack == 8) return k_batch_filter_s<T, OR, 8>;
  if (p.stack) return k_batch_filter_s<T, OR, 16>;
  if (p.TY == 4) return k_batch_filter<T, OR, 4>;
  if (p.TY == 8) return k_batch_filter<T, OR, 8>;
  if (p.TY == 12) return k_batch_filter<T, OR, 12>;
  return k_batch_filter<T, OR, 16>;
}

template <typename T>
static BatchFilterFn<T> batch_filter_fn(const lee_handle *h) {
  return h->cfg.filter_order == 8 ? batch_filter_fn_o<T, 8>(h->bp) : batch_filter_fn_o<T, 4>(h->bp);
}

// Workgroups of kernel f resident on the whole device at once (its
// occupancy per CU, from registers and LDS, times the CUs), a multiple of 8.
static int resident_workgroups(const void *f, int device) {
  int per = 0, cus = 0;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, f, TPB, 0) != hipSuccess || per < 1) per = 1;
  if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, device) != hipSuccess || cus < 1) cus = 8;
  return std::max(8, per * cus / 8 * 8);
}

template <typename T>
static void batch_resident_t(lee_handle *h) {
  BatchPlan &p = h->bp;
  int rs = 1 << 30;
  for (int kind : {STAGE_FIRST, STAGE_MID, STAGE_LAST})
    rs = std::min(rs, resident_workgroups(reinterpret_cast<const void *>(batch_stage_fn<T>(h, kind, true)), h->device));
  p.res_stage = rs;
  p.res_filter = resident_workgroups(reinterpret_cast<const void *>(batch_filter_fn<T>(h)), h->device);
}

template <typename T>
static hipError_t batch_stage_t(hipStream_t s, lee_handle *h, int stage) {
  BatchPlan &p = h->bp;
  const int ns = h->nblk;
  BatchStageArgs<T> ba{};
  ba.args = (const StageArgs<T> *)p.stage_args + (size_t)stage * ns;
  ba.map = p.tile_map_stage;
  ba.sched = p.sched;
  ba.counter = p.counter;
  ba.nsolve = ns;
  ba.nstage = h->cfg.rk_stages;
  ba.stage = stage;
  ba.total = p.total_stage;
  ba.chunk = (p.total_stage + 7) / 8;
  ba.b = (T)h->b_i[stage];
  ba.a = (T)h->a_next[stage];
  const int kind = stage_kind(h, stage);
  const unsigned g = batch_grid(p.total_stage, p.grid_stage, p.res_stage);
  const bool queued = g < 8u * (unsigned)ba.chunk;
  const dim3 grid(g), block(64, 4);
  hipLaunchKernelGGL(batch_stage_fn<T>(h, kind, queued), grid, block, 0, s, ba, CA(ba.args), CA(ba.map), CA(ba.sched),
                     ba.counter, p.counter + QSTRIDE);
  return hipGetLastError();
}

hipError_t batch_stage(hipStream_t s, lee_handle *h, int stage) {
  if (h->cfg.precision == LEE_FP32) return batch_stage_t<float>(s, h, stage);
  return batch_stage_t<double>(s, h, stage);
}

template <typename T>
static hipError_t batch_filter_t(hipStream_t s, lee_handle *h) {
  BatchPlan &p = h->bp;
  BatchFilterArgs<T> ba{};
  ba.args = (const FilterArgs<T> *)p.filter_args;
  ba.map = p.tile_map_filter;
  ba.counter = p.tuning ? p.counter + 1 : p.counter;  // tuning runs leave the step counter alone
  ba.nsolve = h->nblk;
  ba.total = p.total_filter;
  ba.chunk = (p.total_filter + 7) / 8;
  const dim3 grid(batch_grid(p.total_filter, p.grid_filter, p.res_filter)), block(64, 4);
  hipLaunchKernelGGL(batch_filter_fn<T>(h), grid, block, 0, s, ba, CA(ba.args), CA(ba.map));
  return hipGetLastError();
}

hipError_t batch_filter(hipStream_t s, lee_handle *h) {
  if (h->cfg.precision == LEE_FP32) return batch_filter_t<float>(s, h);
  return batch_filter_t<double>(s, h);
}

hipError_t cast_state(hipStream_t s, const Block &, int, const double *src, float *dst, size_t n) {
  hipLaunchKernelGGL((k_cast<double, float>), dim3(nblocks(n)), dim3(TPB), 0, s, src, dst, n);
  return hipGetLastError();
}

hipError_t cast_back(hipStream_t s, const Block &, int, const float *src, double *dst, size_t n) {
  hipLaunchKernelGGL((k_cast<float, double>), dim3(nblocks(n)), dim3(TPB), 0, s, src, dst, n);
  return hipGetLastError();
}

}  // namespace lee
