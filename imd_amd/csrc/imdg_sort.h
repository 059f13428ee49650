// imdg_sort.h -- what the rebuild chain (imdg_build.hip) and the one-block
// sort of small systems (imdg_step.hip) share: wrapping and binning an atom,
// and moving it to its new slot.
#pragma once

#include "imdg_device.h"

namespace imdg {

// fix_cells / do_boundaries and cell_coord of slot i: wraps its position and
// returns its cell (src/imd_main_3d.c:1972-2065, src/imd_geom_3d.c:1054-1074).
__device__ __forceinline__ int wrap_and_bin(const RepDev& R, double4* pos,
                                            int i) {
#pragma clang fp contract(off)
  double4 p = pos[i];
  double x[3] = {p.x, p.y, p.z};
  for (int d = 0; d < 3; d++) {
    if (R.pbc[d] != 1) continue;
    double f = -floor(x[0] * R.tbox[d][0] + x[1] * R.tbox[d][1] +
                      x[2] * R.tbox[d][2]);
    x[0] += f * R.box[d][0];
    x[1] += f * R.box[d][1];
    x[2] += f * R.box[d][2];
  }
  pos[i] = make_double4(x[0], x[1], x[2], p.w);
  int c[3];
  for (int d = 0; d < 3; d++) {
    c[d] = (int)(R.gdim[d] * (x[0] * R.tbox[d][0] + x[1] * R.tbox[d][1] +
                              x[2] * R.tbox[d][2]));
    if (c[d] >= R.gdim[d])
      c[d] = R.gdim[d] - 1;
    else if (c[d] < 0)
      c[d] = 0;
  }
  return R.cell_off + (c[0] * R.gdim[1] + c[1]) * R.gdim[2] + c[2];
}

// Lanes of one cell in the sorts.
#define SORT_LANES 32

// The (u, type) records of the step being built for.
__device__ __forceinline__ void* build_records(const BuildArgs& a) {
  return a.pair_only ? pair_records(a.rec_a, a.rec_b, a.ctl->steps_done)
                     : a.rec_a;
}

__device__ __forceinline__ void move_atom(const BuildArgs& a, const RepDev& R,
                                          int pc, int rc, int from, int to,
                                          int key, int cell) {
  const double4 p = a.pos[pc][from];
  const double4 m = a.mom[rc][from];
  a.pos[pc ^ 1][to] = p;
  a.mom[rc ^ 1][to] = m;
  a.aid[rc ^ 1][to] = key;
  a.acell[to] = cell;
  a.atype[to] = (signed char)p.w;
  a.xnbl[to] = p;
  double c[3];
  cell_centre(R, cell, c);
  void* rec = build_records(a);
  if (a.mixed)
    reinterpret_cast<float4*>(rec)[to] =
        make_float4((float)(p.x - c[0]), (float)(p.y - c[1]),
                    (float)(p.z - c[2]), (float)p.w);
  else
    reinterpret_cast<double4*>(rec)[to] =
        make_double4(p.x - c[0], p.y - c[1], p.z - c[2], p.w);
}

}  // namespace imdg
