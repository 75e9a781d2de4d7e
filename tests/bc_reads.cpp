// Which points the conditions of a BC face read, from the functions the
// kernels run, against the reach that decides what may share a launch.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdio>

using std::max;
using std::min;
static struct { int x, y, z; } threadIdx, blockIdx;  // of kernels that this program does not call

#include "lee_args.h"

using namespace lee;

template <int NS>
int beyond(int type, int dir, int end, int sb, int len) {
  BcArgs a{};
  a.type = type;
  a.dir = dir;
  a.end = end;
  a.ni = dir == 0 ? len : 12;
  a.nj = dir == 0 ? 12 : len;
  a.sb = sb;
  a.i1 = a.ni - 1;
  a.j1 = a.nj - 1;
  const int c = end == 0 ? 0 : len - 1;
  (dir == 0 ? a.i0 : a.j0) = (dir == 0 ? a.i1 : a.j1) = c;
  for (int q = 0; q < sb; q++) a.neu[q] = q == 0 ? -1.5 : 0.5;
  const BcReach r = bc_reach(a);
  double met[4 * 12 * 12] = {0}, jac[12 * 12] = {0}, data[NV];
  int bad = 0;
  bc_face_data<double, NS>(a, 0, 0, c, len, met, jac, [&](int, int s) {
    const int at = c + (end == 0 ? s : -s);
    bad += at < r.lo[dir] || at > r.hi[dir];
    return 1.0;
  }, data);
  return bad;
}

int main() {
  int bad = 0;
  for (int type : {LEE_BC_NEUMANN, LEE_BC_WALL_SLIP_KINEMATIC, LEE_BC_CENTERLINE_AXISYM, LEE_BC_DIRICHLET_ALLZERO})
    for (int dir : {0, 1})
      for (int end : {0, 1}) {
        bad += beyond<8>(type, dir, end, 3, 12) + beyond<8>(type, dir, end, 9, 12) + beyond<2>(type, dir, end, 3, 12);
      }
  printf("%d reads beyond the reach\n", bad);
  return bad != 0;
}
