// Two RK stages of the fused 2-D time advance in one launch (gfx950).
//
// A stage reads its input, y_n, the accumulator and the FP64 geometry and
// writes the accumulator and the next input; the next launch reads all of it
// back.  Run in pairs, the stages of RK4 move 92 + 108 bytes a point in FP32
// (uniform mean) instead of 92 + 124 + 124 + 92, and two launches replace
// four; the price is the first stage of each pair on a halo of 2 points.
// Every point takes the operations of the one-stage kernels in the same
// order, so the results are bit-identical to theirs.
//
// Steps of RK4 with the 8th-order filter, one stage a launch -> paired (us):
//   97 x 81      FP32 30.1 -> 15.9   FP64 31.8 -> 17.1   (1 row a wave)
//   257 x 257    FP32 30.4 -> 17.1   FP64 35.7 -> 21.2   (1 row)
//   513 x 513    FP32 41.3 -> 27.8   FP64 54.2 -> 39.7   (2 rows, FP64 1)
//   1025 x 1025  FP32 89.7 -> 59.1   FP64 132  -> 83.5   (2 rows)
//   2311 x 1507  FP32 299  -> 179    FP64 549  -> 306    (2 rows)
//   701 x 467, sheared mean and two walls: FP32 67.0 -> 45.2, FP64 96.0 -> 67.2
// What bounds it: at small blocks one workgroup's chain of latencies (launch,
// operands, two stages), at large ones HBM (2311 x 1507 FP32: 200 bytes a
// point in 155 us, 4.5 TB/s where a large copy reaches 4.9; the counters of
// 1025 x 1025 give 97 + 105 MB for the 97 + 113 that the data take).
//
// A workgroup is 8 waves of RA rows: RA = 2 costs 16 / 12 rows of the first
// stage, RA = 1 8 / 4, but has the shortest chain.  Measured and not kept, at
// 1025 x 1025 FP32 against 61 us then: 4 waves of 3 rows 63 (2311 x 1507 the same,
// FP64 1.6 times slower for its registers), 16 of 1 row 74, 4 of 2 rows 68, 16
// of 2 and 8 of 3 rows slower still.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>

#include "lee_args.h"
#include "lee_bc.h"
#include "lee_device.h"
#include "lee_internal.h"
#include "lee_stage.h"

namespace lee {

namespace {

constexpr int P2_WAVES = 8;  // waves of a workgroup
constexpr int P2_FACES = 4;  // BC faces a paired launch applies itself
constexpr int P2_ZONES = 4;  // sponge zones of a block run in pairs
constexpr int PZ = 2;        // sponge zones that may share a point of a paired launch (zones_meet_thrice)

// The BC faces between the two stages, and on the input of the second pair
// (the update after the stage before it); dt and source factors of each
// stage, entropy factors of the harmonic wave.
template <typename T>
struct PairScalars {
  StepT<T> s[2];
  double he[2];              // at the two stages
  int harm;                  // some zone relaxes to the harmonic wave
  int nf_in, nf;             // faces applied to the input / between the stages
  double he_in, he_mid;      // their entropy factors
  BcArgs f[P2_FACES];
  const double *met, *jac;
};

// bc::apply_BC on the part of the LDS tile (rows [r0, r1), columns [c0, c1);
// tile point (r, c) is block point (gi0 + c, gj0 + r)) that lies on a face.
// Faces lie on the block's ends, so the points their rows read inward are in
// the tile; faces one after the other, in the order of the BC file.
template <typename T, int NR, int RS>
__device__ __forceinline__ void faces_lds(T (&s)[4][NR][RS], const PairScalars<T> &ps, int nf, double he, int gi0,
                                          int gj0, int r0, int r1, int c0, int c1) {
  const int tid = threadIdx.y * 64 + threadIdx.x;
  for (int k = 0; k < nf; k++) {
    const BcArgs &f = ps.f[k];
    const int i0 = max(f.i0, gi0 + c0), i1 = min(f.i1, gi0 + c1 - 1);
    const int j0 = max(f.j0, gj0 + r0), j1 = min(f.j1, gj0 + r1 - 1);
    if (i0 > i1 || j0 > j1) continue;  // uniform over the workgroup
    BcArgs a = f;
    a.he = he;
    const int w = i1 - i0 + 1, cnt = w * (j1 - j0 + 1), sg = a.end == 0 ? 1 : -1;
    for (int t = tid; t < cnt; t += 64 * (int)blockDim.y) {
      const int i = i0 + t % w, j = j0 + t / w;
      const int c = a.dir == 0 ? i : j, len = a.dir == 0 ? a.ni : a.nj;
      const int q = (j - a.j0) * (a.i1 - a.i0 + 1) + (i - a.i0);
      double data[NV];
      bc_face_data<T, 2>(
          a, q, j * a.ni + i, c, len, ps.met, ps.jac,
          [&](int v, int d) -> T {
            if (v == IUZ) return (T)0;  // blocks that carry w' run one stage a launch
            const int o = c + sg * d >= 0 && c + sg * d < len ? sg * d : 0;
            return s[v == IP ? 3 : v][j - gj0 + (a.dir == 1 ? o : 0)][i - gi0 + (a.dir == 0 ? o : 0)];
          },
          data);
      s[0][j - gj0][i - gi0] = (T)data[IS];
      s[1][j - gj0][i - gi0] = (T)data[IUX];
      s[2][j - gj0][i - gi0] = (T)data[IUY];
      s[3][j - gj0][i - gi0] = (T)data[IP];
    }
    __syncthreads();
  }
}

// Butcher coefficients of the two stages of a batched pair.
template <typename T>
struct BatchPairCoef {
  T b[2], a[2];
};

// The value `off` bytes behind a uniform address: a scalar base and one
// 32-bit vector offset, so that the loads of a row need no vector arithmetic.
template <typename U>
__device__ __forceinline__ U ld_off(const U *base, unsigned off) {
  return *(const U *)((const char *)base + off);
}
template <typename U>
__device__ __forceinline__ void st_off(U *base, unsigned off, U v) {
  *(U *)((char *)base + off) = v;
}

// The input tile with its halo of 4, and a row of zeros (Row4) per row of a
// wave: the zeros then lie as far from every one of its rows, and the rows'
// addresses differ by constants.
template <typename T, int RA>
using PairLds = T[4][P2_WAVES * RA + 4 + RA][68];

// Stages A and B of a pair on a tile of 60 x (4 RA - 4) points.  Lane l of
// wave w holds block column 60 tile_x - 2 + l and the RA rows from
// TYO tile_y - 2 + RA w: the tile and its halo of 2, on which A is computed.
// The input tile (halo 4) is in LDS; A's results replace it there once every
// wave has computed its rows; B runs on the rows and lanes inside the halo,
// in the same threads, which keep the metrics, A's accumulator and y_n in
// registers.  Everything a point needs from memory is requested before the
// first barrier (the mean coefficients one row ahead): with the requests left
// at their use each row waited for memory on its own.
template <typename T, bool MEANF, bool FIRST, int RA, bool INNER, bool FACES, typename AT>
__device__ __forceinline__ void pair_tile_k(const AT &a, const PairScalars<T> &ps, int tx0, int ty0,
                                            PairLds<T, RA> &s) {
#pragma clang fp contract(off)
  constexpr int NW = P2_WAVES, NR = NW * RA, TYO = NR - 4, RS = 68;  // rows of A and of the tile
  const int lane = threadIdx.x, w = __builtin_amdgcn_readfirstlane((int)threadIdx.y);
  const int ni = a.ni, nj = a.nj;
  const size_t n = (size_t)ni * nj, VOFF[4] = {IS * n, IUX * n, IUY * n, IP * n};
  const int i0 = tx0 * 60 - 4, j0 = ty0 * TYO - 4;  // block point of LDS (0, 0)
  const int gi = i0 + 2 + lane;
  const bool col = INNER || (gi >= 0 && gi < ni);
  auto row_of = [&](int k) { return w * RA + k + 2; };  // LDS row
  const int zeros = NR + 4 - row_of(0);                 // rows down to the zeros
  const Row4<T> rx = row4<T>(INNER ? CODE_INTERIOR : default_code(gi, ni, 2), zeros * RS);
  auto in_block = [&](int k) {
    const int gj = j0 + row_of(k);
    return INNER || (col && gj >= 0 && gj < nj);
  };
  // points outside the block read the nearest one of it: no row inside the
  // block uses their values.  Rows are uniform, so an address is a scalar row
  // and one of a few lane offsets.
  auto row_start = [&](int k) {
    const int gj = j0 + row_of(k);
    return (size_t)(INNER ? gj : min(max(gj, 0), nj - 1)) * ni;
  };
  const unsigned ci = (unsigned)(INNER ? gi : min(max(gi, 0), ni - 1));
  const unsigned oT = ci * (unsigned)sizeof(T), o8 = ci * 8u;
  // the input tile
  T ta[RA + 1][4], tb[RA + 1][4];
  const bool xtra = lane < 4;
  const unsigned oa = (unsigned)(INNER ? i0 + lane : min(max(i0 + lane, 0), ni - 1)) * (unsigned)sizeof(T);
  const unsigned ob = (unsigned)min(i0 + lane + 64, ni - 1) * (unsigned)sizeof(T);
  auto in_row = [&](int k) {
    const int gj = j0 + w + NW * k;
    return (size_t)(INNER ? gj : min(max(gj, 0), nj - 1)) * ni;
  };
#pragma unroll
  for (int k = 0; k <= RA; k++) {
    if (k == RA && w >= 4) break;  // NR + 4 rows
#pragma unroll
    for (int v = 0; v < 4; v++) ta[k][v] = ld_off(a.yin + VOFF[v] + in_row(k), oa);
  }
  if (xtra) {
#pragma unroll
    for (int k = 0; k <= RA; k++) {
      if (k == RA && w >= 4) break;
#pragma unroll
      for (int v = 0; v < 4; v++) tb[k][v] = ld_off(a.yin + VOFF[v] + in_row(k), ob);
    }
  }
  // the points' own operands
  double m[RA][4], J[RA];
  T yn[RA][4], acc[RA][4], rho0[RA];
#pragma unroll
  for (int k = 0; k < RA; k++) {
    const size_t r = row_start(k);
#pragma unroll
    for (int q = 0; q < 4; q++) m[k][q] = ld_off(a.met + q * n + r, o8);
    J[k] = ld_off(a.jac + r, o8);
#pragma unroll
    for (int v = 0; v < 4; v++) {
      yn[k][v] = FIRST ? (T)0 : ld_off(a.yn + VOFF[v] + r, oT);
      acc[k][v] = FIRST ? (T)0 : ld_off((const T *)a.acc + VOFF[v] + r, oT);
    }
    rho0[k] = MEANF && FIRST ? ld_off(a.rho_in + r, oT) : (T)0;
  }
  // the sponges of the tile (uniform), then each point's first and second:
  // their places are found first and both strengths requested together.  The
  // zones' boxes are read at fixed places, all at once (unused ones are empty).
  unsigned zmask = 0;
#pragma unroll
  for (int z = 0; z < P2_ZONES; z++)
    zmask |= a.z[z].i0 <= i0 + 65 && a.z[z].i1 >= i0 + 2 && a.z[z].j0 <= j0 + NR + 1 && a.z[z].j1 >= j0 + 2 ? 1u << z : 0;
  const bool sponged = zmask != 0;
  T sg[RA][PZ];
  int sz[RA][PZ];  // their zones (-1: none)
#pragma unroll
  for (int k = 0; k < RA; k++)
#pragma unroll
    for (int q = 0; q < PZ; q++) {
      sg[k][q] = (T)0;
      sz[k][q] = -1;
    }
  if (sponged) {
    const T *at[RA][PZ];
#pragma unroll
    for (int k = 0; k < RA; k++) {
      const int gj = j0 + row_of(k);
      at[k][0] = at[k][1] = nullptr;
#pragma unroll
      for (int z = 0; z < P2_ZONES; z++) {
        if (!(zmask >> z & 1)) continue;  // uniform
        const auto &zz = a.z[z];
        const bool in = gi >= zz.i0 && gi <= zz.i1 && gj >= zz.j0 && gj <= zz.j1;
        const T *sp = zz.sig + ((gj - zz.j0) * zz.nzi + (gi - zz.i0));
        const bool second = in && sz[k][0] >= 0;
        at[k][1] = second ? sp : at[k][1];
        sz[k][1] = second ? z : sz[k][1];
        at[k][0] = in && !second ? sp : at[k][0];
        sz[k][0] = in && !second ? z : sz[k][0];
      }
    }
#pragma unroll
    for (int k = 0; k < RA; k++)
#pragma unroll
      for (int q = 0; q < PZ; q++)
        if (sz[k][q] >= 0) sg[k][q] = *at[k][q];
  }
  const bool sourced = a.si0 <= i0 + 65 && a.si1 >= i0 + 2 && a.sj0 <= j0 + NR + 1 && a.sj1 >= j0 + 2;  // uniform
  T mc[2][MC_COUNT];
  // mean coefficients of row k (STALE: see stage_terms)
  auto mean_of = [&](auto stale, int k, T (&c)[MC_COUNT]) {
    const size_t r = row_start(k);
#pragma unroll
    for (int f = 0; f < MC_R; f++)
      c[f] = stale.value && (f == MC_RP || f == MC_RB) ? (T)0 : ld_off(a.mc + f * n + r, oT);
    c[MC_R] = a.axi ? ld_off(a.mc + MC_R * n + r, oT) : (T)0;
  };
  if (MEANF) mean_of(std::integral_constant<bool, FIRST>{}, 0, mc[0]);
  static_assert(P2_WAVES == 8 && RA <= 2, "a wave sets a variable's row of zeros");
  if (!INNER && w < 4 * RA) {
    s[w & 3][NR + 4 + (w >> 2)][lane] = (T)0;
    if (xtra) s[w & 3][NR + 4 + (w >> 2)][64 + lane] = (T)0;
  }
#pragma unroll
  for (int k = 0; k <= RA; k++)
#pragma unroll
    for (int v = 0; v < 4; v++) {
      if (k == RA && w >= 4) break;
      s[v][w + NW * k][lane] = ta[k][v];
      if (xtra) s[v][w + NW * k][64 + lane] = tb[k][v];
    }
  __syncthreads();
  if (FACES && !FIRST && ps.nf_in) faces_lds<T>(s, ps, ps.nf_in, ps.he_in, i0, j0, 0, NR + 4, 0, 68);
  // right-hand side of stage st at row k from the LDS tile
  auto rhs = [&](auto stale, int st, int k, const T *mck, const T (&yc)[4], T (&r)[4]) {
    const int row = row_of(k), gj = j0 + row;
    T dx[4], dy[4];
    if constexpr (INNER) {
#pragma unroll
      for (int v = 0; v < 4; v++) {
        const T *sp = &s[v][row][lane + 2];
        dx[v] = fd_row<T>(sp, 1, CODE_INTERIOR);
        dy[v] = fd_row<T>(sp, RS, CODE_INTERIOR);
      }
    } else {
      const Row4<T> ry = row4<T>(default_code(gj, nj, 2), zeros);  // uniform
#pragma unroll
      for (int v = 0; v < 4; v++) {
        const T *sp = &s[v][row][lane + 2];
        dx[v] = row4_sum<T>(rx, sp, 1);
        dy[v] = row4_sum<T>(ry, sp, RS);
      }
    }
    stage_terms<T, MEANF, stale.value>(a, m[k], J[k], [&](int f) { return mck[f]; }, [&]() { return rho0[k]; }, yc, dx,
                                       dy, r);
    if (sourced && gi >= a.si0 && gi <= a.si1 && gj >= a.sj0 && gj <= a.sj1) {
      const double gval = a.g[(gj - a.sj0) * (a.si1 - a.si0 + 1) + (gi - a.si0)];
      r[3] += (T)(ps.s[st].s1 * gval * ps.s[st].s2);
    }
    if (sponged) {
#pragma unroll
      for (int q = 0; q < PZ; q++) {
        if (sz[k][q] < 0) continue;
        T ds = yc[0];
        if (ps.harm) {  // uniform
          const auto &zz = a.z[sz[k][q]];
          const int zp = (gj - zz.j0) * zz.nzi + (gi - zz.i0);
          if (zz.harm) ds = yc[0] - (T)(zz.hg ? ps.he[st] * zz.hg[zp] : ps.he[st]);
        }
        sponge_relax(sg[k][q], ds, yc, r);
      }
    }
  };
  // stage A on the rows of this wave: u replaces the input in LDS afterwards
  T u[RA][4];
#pragma unroll
  for (int k = 0; k < RA; k++) {
    // the next row's mean coefficients (B's first row after A's last) are
    // requested before this row's are used
    if (MEANF) {
      if (k + 1 < RA) mean_of(std::integral_constant<bool, FIRST>{}, k + 1, mc[(k + 1) % 2]);
      else mean_of(std::false_type{}, 0, mc[RA % 2]);
    }
    const int row = row_of(k);
    T yc[4], r[4] = {(T)0, (T)0, (T)0, (T)0};
#pragma unroll
    for (int v = 0; v < 4; v++) {
      yc[v] = s[v][row][lane + 2];
      if (FIRST) yn[k][v] = acc[k][v] = yc[v];
    }
    if (in_block(k)) rhs(std::integral_constant<bool, FIRST>{}, 0, k, mc[k % 2], yc, r);
#pragma unroll
    for (int v = 0; v < 4; v++) {
      const T rh = r[v] * ps.s[0].h;
      acc[k][v] = fmx(ps.s[0].b, rh, acc[k][v]);
      u[k][v] = fmx(ps.s[0].a, rh, yn[k][v]);
    }
  }
  __syncthreads();
#pragma unroll
  for (int k = 0; k < RA; k++)
#pragma unroll
    for (int v = 0; v < 4; v++) s[v][row_of(k)][lane + 2] = u[k][v];
  __syncthreads();
  if (FACES && ps.nf) faces_lds<T>(s, ps, ps.nf, ps.he_mid, i0, j0, 2, NR + 2, 2, 66);
  // stage B inside the halo
  const bool out_lane = lane >= 2 && lane < 62 && col;
#pragma unroll
  for (int k = 0; k < RA; k++) {
    if (MEANF && k + 1 < RA) mean_of(std::false_type{}, k + 1, mc[(RA + k + 1) % 2]);
    const int row = row_of(k), gj = j0 + row;
    if (row < 4 || row >= NR || (!INNER && gj >= nj) || !out_lane) continue;
    const size_t rs = row_start(k);
    T yc[4], r[4];
#pragma unroll
    for (int v = 0; v < 4; v++) yc[v] = s[v][row][lane + 2];
    const T(&mck)[MC_COUNT] = mc[(RA + k) % 2];
    rhs(std::integral_constant<bool, false>{}, 1, k, mck, yc, r);
    T accv[4];
#pragma unroll
    for (int v = 0; v < 4; v++) {
      const T rh = r[v] * ps.s[1].h;
      accv[v] = fmx(ps.s[1].b, rh, acc[k][v]);
      st_off(a.acc + VOFF[v] + rs, oT, accv[v]);
      if (FIRST) st_off(a.yout + VOFF[v] + rs, oT, fmx(ps.s[1].a, rh, yn[k][v]));
    }
    if (MEANF && !FIRST) st_off(a.rho_out + rs, oT, fmx(accv[3], mck[MC_RP], -(accv[0] * mck[MC_RB])));
  }
}

template <typename T, bool MEANF, bool FIRST, int RA, bool FACES, typename AT>
__device__ __forceinline__ void pair_tile(const AT &a, const PairScalars<T> &ps, int tile, PairLds<T, RA> &s) {
  constexpr int NR = P2_WAVES * RA;
  const int tx0 = tile % a.ntx, ty0 = tile / a.ntx;
  const int i0 = tx0 * 60 - 4, j0 = ty0 * (NR - 4) - 4;
  // a tile whose input lies inside the block, and off its faces: those that
  // touch one take the other instance, so that this one has no faces in it
  // (701 x 467 FP32 between walls 46.5 -> 45.5 us a step)
  constexpr int OFF = FACES ? 1 : 0;
  if (i0 >= OFF && i0 + 68 <= a.ni - OFF && j0 >= OFF && j0 + NR + 4 <= a.nj - OFF)
    pair_tile_k<T, MEANF, FIRST, RA, true, false>(a, ps, tx0, ty0, s);
  else
    pair_tile_k<T, MEANF, FIRST, RA, false, FACES>(a, ps, tx0, ty0, s);
}

// Waves per SIMD the registers are held to: four (two workgroups a CU) with a
// uniform mean, where a few spilled values cost less than half the waves
// (1025 x 1025 FP64 91 us a step against 113 unconstrained); with the mean
// coefficients in registers it would spill hundreds of bytes (701 x 467 FP64
// 117 us against 67).
constexpr int pair_waves(bool meanf, int ra) { return meanf ? (ra == 2 ? 2 : 3) : 4; }

// FACES: the block has faces.  Instances without them keep 30 to 100 scalar
// registers fewer in vector lanes: 1025 x 1025 FP32 / FP64 61.1 / 87.3 us a step
// -> 59.0 / 86.0, 701 x 467 FP32 sheared, without walls, 39.1 -> 37.4.
template <typename T, bool MEANF, bool FIRST, int RA, bool FACES>
__global__ void __launch_bounds__(64 * P2_WAVES, pair_waves(MEANF, RA)) k_fused_pair(StageArgs<T> a,
                                                                                     PairScalars<T> ps) {
  __shared__ PairLds<T, RA> s;
  const int tile = xcd_tile(blockIdx.x, a.chunk);
  if (tile >= a.ntiles) return;
  pair_tile<T, MEANF, FIRST, RA, FACES>(a, ps, tile, s);
}

// The same for a batched ensemble: one workgroup per (solve, tile) entry of
// the list, its operands and scalars from the batch's tables (k_batch_stage).
template <typename T, bool MEANF, bool FIRST, int RA>
__global__ void __launch_bounds__(64 * P2_WAVES, pair_waves(MEANF, RA))
    k_batch_pair(BatchStageArgs<T> ba, const LEE_CONST_AS StageArgs<T> *args, const LEE_CONST_AS int *map,
                 const LEE_CONST_AS BatchSched *sched, const int *__restrict__ counter, BatchPairCoef<T> c) {
  __shared__ PairLds<T, RA> s;
  const int t = (blockIdx.x & 7) * ba.chunk + (blockIdx.x >> 3);
  if (t >= ba.total) return;
  const int step = __hip_atomic_load(counter, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  const int k = map[2 * t], local = map[2 * t + 1];
  const LEE_CONST_AS BatchSched *q = sched + ((size_t)step * ba.nsolve + k) * ba.nstage + ba.stage;
  PairScalars<T> ps;
#pragma unroll
  for (int i = 0; i < 2; i++) {
    ps.s[i] = StepT<T>{(T)q[i].dt, c.b[i], c.a[i], q[i].s1, q[i].s2};
    ps.he[i] = 0.0;
  }
  ps.harm = 0;
  pair_tile<T, MEANF, FIRST, RA, false>(args[k], ps, local, s);
}

// Tile counts of the paired form, unused zones empty.
template <typename T>
inline void pair_tiles(StageArgs<T> &a, int RA) {
  const int rows = P2_WAVES * RA - 4;
  a.ntx = (a.ni + 59) / 60;
  a.nty = (a.nj + rows - 1) / rows;
  a.ntiles = a.ntx * a.nty;
  a.chunk = (a.ntiles + 7) / 8;
  for (int z = a.nz; z < P2_ZONES; z++) a.z[z].i1 = -1;  // empty
}

template <typename T>
hipError_t fused_pair_t(hipStream_t s, lee_handle *h, Block &b, int first, const PairStep &st, T *const *Y, T *rho) {
  const int RA = b.tune_pair;
  const bool F = first == 0 || first == -2;
  // the second pair of RK4 reads Y2 and the accumulator, like stage 1
  StageArgs<T> a = make_stage_args<T>(h, b, first > 0 ? 1 : first, Y, rho, 1, st.sc[0]);
  pair_tiles(a, RA);
  PairScalars<T> ps{};
  for (int k = 0; k < 2; k++) {
    const StageScalars &sc = st.sc[k];
    ps.s[k] = {(T)sc.h, (T)sc.b, (T)sc.a, sc.s1, sc.s2};
    ps.he[k] = sc.he;
  }
  ps.nf = (int)b.faces.size();
  ps.nf_in = F ? 0 : ps.nf;
  for (int k = 0; k < ps.nf; k++) ps.f[k] = make_bc_args(h, b, b.faces[k], 0.0);
  ps.he_in = st.he_in;
  ps.he_mid = st.he_mid;
  for (const auto &z : b.zones) ps.harm |= z.harmonic;
  ps.met = b.met;
  ps.jac = b.jac;
  const dim3 grid(a.chunk * 8), block(64, P2_WAVES);
  const bool mf = !b.uniform_mean;
#define LEE_P2(MF, FF)                                                                                           \
  do {                                                                                                           \
    if (RA == 1 && ps.nf == 0) hipLaunchKernelGGL((k_fused_pair<T, MF, FF, 1, false>), grid, block, 0, s, a, ps); \
    else if (RA == 1) hipLaunchKernelGGL((k_fused_pair<T, MF, FF, 1, true>), grid, block, 0, s, a, ps);          \
    else if (ps.nf == 0) hipLaunchKernelGGL((k_fused_pair<T, MF, FF, 2, false>), grid, block, 0, s, a, ps);      \
    else hipLaunchKernelGGL((k_fused_pair<T, MF, FF, 2, true>), grid, block, 0, s, a, ps);                       \
  } while (0)
  if (mf && F) LEE_P2(true, true);
  else if (mf) LEE_P2(true, false);
  else if (F) LEE_P2(false, true);
  else LEE_P2(false, false);
#undef LEE_P2
  return hipGetLastError();
}

}  // namespace

// Whether three sponge zones share a point.
static bool zones_meet_thrice(const Block &b) {
  const size_t n = b.zones.size();
  for (size_t x = 0; x < n; x++)
    for (size_t y = x + 1; y < n; y++)
      for (size_t z = y + 1; z < n; z++) {
        bool meet = true;
        for (int d = 0; d < 2; d++) {
          const int lo = std::max({b.zones[x].is[d], b.zones[y].is[d], b.zones[z].is[d]});
          const int hi = std::min({b.zones[x].ie[d], b.zones[y].ie[d], b.zones[z].ie[d]});
          meet &= lo <= hi;
        }
        if (meet) return true;
      }
  return false;
}

bool paired_stages_ok(const lee_handle *h, const Block &b) {
  if (h->cfg.num_dim != 2 || h->cfg.path != LEE_PATH_FUSED || h->cfg.fd_order != 4 ||
      h->cfg.rk_stages != 4 || h->cfg.num_scalar ||
      h->ov.nrecv || b.has_holes || b.carry_w || (int)b.faces.size() > P2_FACES || (int)b.zones.size() > P2_ZONES)
    return false;
  if (zones_meet_thrice(b)) return false;
  if (h->batch) {  // no boundary launches between stages, no wave factors in the schedule
    if (!b.faces.empty()) return false;
    for (const auto &z : b.zones)
      if (z.harmonic) return false;
  }
  for (const auto &f : b.faces) {
    const int len = f.dir == 0 ? b.ni : b.nj;
    if (f.is[f.dir] != (f.end == 0 ? 0 : len - 1)) return false;
  }
  return true;
}

// Keeps the stream at a fixed number of short sleeps, some 100 us, on one wave.
namespace {
__global__ void k_hold(int naps) {
  for (int k = 0; k < naps; k++) __builtin_amdgcn_s_sleep(127);  // 127 x 64 cycles
}
}  // namespace

hipError_t hold_stream(hipStream_t s) {
  hipLaunchKernelGGL(k_hold, dim3(1), dim3(64), 0, s, 30);
  return hipGetLastError();
}

hipError_t fused_pair(hipStream_t s, lee_handle *h, Block &b, int first, const PairStep &st) {
  if (h->cfg.precision == LEE_FP32) return fused_pair_t<float>(s, h, b, first, st, b.Y32, b.rho32);
  return fused_pair_t<double>(s, h, b, first, st, b.Y64, b.rho64);
}

template <typename T>
static hipError_t batch_pair_t(hipStream_t s, lee_handle *h, int first) {
  BatchPlan &p = h->bp;
  BatchStageArgs<T> ba{};
  // tables of pair 0 (stages 0, 1), then of pair 1
  const StageArgs<T> *args = (const StageArgs<T> *)p.pair_args + (size_t)(first / 2) * h->nblk;
  ba.nsolve = h->nblk;
  ba.nstage = h->cfg.rk_stages;
  ba.stage = first;
  ba.total = p.total_pair;
  ba.chunk = (p.total_pair + 7) / 8;
  const BatchPairCoef<T> c{{(T)h->b_i[first], (T)h->b_i[first + 1]}, {(T)h->a_next[first], (T)h->a_next[first + 1]}};
  const dim3 grid(8 * ba.chunk), block(64, P2_WAVES);
  const bool mf = !h->b[0].uniform_mean, F = first == 0;
#define LEE_BP(MF, FF)                                                                                          \
  do {                                                                                                          \
    if (p.pair == 1)                                                                                            \
      hipLaunchKernelGGL((k_batch_pair<T, MF, FF, 1>), grid, block, 0, s, ba, CA(args), CA(p.tile_map_pair),    \
                         CA(p.sched), p.counter, c);                                                            \
    else                                                                                                        \
      hipLaunchKernelGGL((k_batch_pair<T, MF, FF, 2>), grid, block, 0, s, ba, CA(args), CA(p.tile_map_pair),    \
                         CA(p.sched), p.counter, c);                                                            \
  } while (0)
  if (mf && F) LEE_BP(true, true);
  else if (mf) LEE_BP(true, false);
  else if (F) LEE_BP(false, true);
  else LEE_BP(false, false);
#undef LEE_BP
  return hipGetLastError();
}

hipError_t batch_pair(hipStream_t s, lee_handle *h, int first) {
  if (h->cfg.precision == LEE_FP32) return batch_pair_t<float>(s, h, first);
  return batch_pair_t<double>(s, h, first);
}

// Operand tables and tile list of the paired batch launches (p.pair rows a
// wave); p.tuning: on scratch buffers, as batch_prepare's.
template <typename T>
static hipError_t batch_pair_prepare_t(hipStream_t s, lee_handle *h) {
  BatchPlan &p = h->bp;
  const int ns = h->nblk;
  std::vector<StageArgs<T>> pa((size_t)2 * ns);
  std::vector<int> map;
  const StageScalars zero{0.0, 0.0, 0.0, 0.0, 0.0};
  for (int k = 0; k < ns; k++) {
    Block &b = h->b[k];
    T *const *Y = sizeof(T) == 8 ? (T *const *)b.Y64 : (T *const *)b.Y32;
    T *rho = sizeof(T) == 8 ? (T *)b.rho64 : (T *)b.rho32;
    for (int q = 0; q < 2; q++) {  // the second pair reads Y2 and the accumulator, like stage 1
      StageArgs<T> &a = pa[(size_t)q * ns + k];
      a = make_stage_args<T>(h, b, p.tuning ? -2 - q : q, Y, rho, 1, zero);
      pair_tiles(a, p.pair);
    }
    for (int t = 0; t < pa[k].ntiles; t++) {
      map.push_back(k);
      map.push_back(t);
    }
  }
  p.total_pair = (int)(map.size() / 2);
  hipError_t e;
  if ((e = hipMalloc(&p.pair_args, sizeof(StageArgs<T>) * pa.size())) != hipSuccess) return e;
  if ((e = hipMalloc((void **)&p.tile_map_pair, sizeof(int) * map.size())) != hipSuccess) return e;
  if ((e = hipMemcpyAsync(p.pair_args, pa.data(), sizeof(StageArgs<T>) * pa.size(), hipMemcpyHostToDevice, s)))
    return e;
  if ((e = hipMemcpyAsync(p.tile_map_pair, map.data(), sizeof(int) * map.size(), hipMemcpyHostToDevice, s))) return e;
  return hipStreamSynchronize(s);  // the host vectors die here
}

hipError_t batch_pair_prepare(hipStream_t s, lee_handle *h) {
  if (h->cfg.precision == LEE_FP32) return batch_pair_prepare_t<float>(s, h);
  return batch_pair_prepare_t<double>(s, h);
}

}  // namespace lee
