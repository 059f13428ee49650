// imdg_device.h -- device helpers shared by the rebuild kernels
// (imdg_build.hip) and the per-step kernels (imdg_step.hip): wavefront and
// compensated reductions, IMD's 3-point table access on knot pairs, the
// grouped neighbour-list layout, cell geometry.
#pragma once

#include <hip/hip_runtime.h>
#include <math.h>

#include "imdg_internal.h"

namespace imdg {

// One DPP move of a double (both halves); rows outside the mask keep `old`.
template <int CTRL, int ROWS>
__device__ __forceinline__ double dpp_d(double old, double v) {
  const int lo = __builtin_amdgcn_update_dpp(__double2loint(old),
                                             __double2loint(v), CTRL, ROWS,
                                             0xf, false);
  const int hi = __builtin_amdgcn_update_dpp(__double2hiint(old),
                                             __double2hiint(v), CTRL, ROWS,
                                             0xf, false);
  return __hiloint2double(hi, lo);
}
__device__ __forceinline__ double lane63_d(double v) {
  return __hiloint2double(
      __builtin_amdgcn_readlane(__double2hiint(v), 63),
      __builtin_amdgcn_readlane(__double2loint(v), 63));
}

// Sum and maximum over the 64 lanes (every lane active), in every lane, by
// DPP moves: quad permutes, row mirrors, and the broadcasts of lanes 15 and
// 31 to the next rows (lane 63 ends with the total).  A cross-lane shuffle is
// a trip through LDS (64 cycles and more, twice per double and level): the
// reductions at the end of a small launch were 1 us of it.
__device__ __forceinline__ double wave_sum(double v) {
  v += dpp_d<0xb1, 0xf>(0.0, v);
  v += dpp_d<0x4e, 0xf>(0.0, v);
  v += dpp_d<0x141, 0xf>(0.0, v);
  v += dpp_d<0x140, 0xf>(0.0, v);
  v += dpp_d<0x142, 0xa>(0.0, v);
  v += dpp_d<0x143, 0xc>(0.0, v);
  return lane63_d(v);
}

// Minimum over the 64 lanes (every lane active) through DPP
// moves (quad permutes, row mirrors, row broadcasts of lanes 15 and 31:
// VALU operations without a trip through LDS), read from lane 63.
#define IMDG_DPP_REDUCE(OP, v)                                                \
  do {                                                                        \
    v = OP(v, __builtin_amdgcn_update_dpp(v, v, 0xb1, 0xf, 0xf, false));      \
    v = OP(v, __builtin_amdgcn_update_dpp(v, v, 0x4e, 0xf, 0xf, false));      \
    v = OP(v, __builtin_amdgcn_update_dpp(v, v, 0x141, 0xf, 0xf, false));     \
    v = OP(v, __builtin_amdgcn_update_dpp(v, v, 0x140, 0xf, 0xf, false));     \
    v = OP(v, __builtin_amdgcn_update_dpp(v, v, 0x142, 0xa, 0xf, false));     \
    v = OP(v, __builtin_amdgcn_update_dpp(v, v, 0x143, 0xc, 0xf, false));     \
  } while (0)

__device__ __forceinline__ int wave_min_i(int v) {
  IMDG_DPP_REDUCE(min, v);
  return __builtin_amdgcn_readlane(v, 63);
}


__device__ __forceinline__ double wave_max(double v) {
  v = fmax(v, dpp_d<0xb1, 0xf>(v, v));
  v = fmax(v, dpp_d<0x4e, 0xf>(v, v));
  v = fmax(v, dpp_d<0x141, 0xf>(v, v));
  v = fmax(v, dpp_d<0x140, 0xf>(v, v));
  v = fmax(v, dpp_d<0x142, 0xa>(v, v));
  v = fmax(v, dpp_d<0x143, 0xc>(v, v));
  return lane63_d(v);
}

// Error-free sum of two doubles (Knuth TwoSum).
__device__ __forceinline__ void two_sum(double a, double b, double& s,
                                        double& e) {
#pragma clang fp contract(off)
  s = a + b;
  double bb = s - a;
  e = (a - (s - bb)) + (b - bb);
}

// Neumaier-compensated accumulation.
__device__ __forceinline__ void kahan_add(double& s, double& c, double x) {
#pragma clang fp contract(off)
  double t = s + x;
  if (fabs(s) >= fabs(x))
    c += (s - t) + x;
  else
    c += (x - t) + s;
  s = t;
}

// Compensated sum of (s, c) pairs over the 64 lanes in a fixed order
// (TwoSum keeps every rounding error); the total, error added, in every lane.
__device__ __forceinline__ double wave_sum_comp(double s, double c) {
#define IMDG_COMB(CTRL, ROWS)                     \
  do {                                            \
    const double so = dpp_d<CTRL, ROWS>(0.0, s);  \
    const double co = dpp_d<CTRL, ROWS>(0.0, c);  \
    double t, e;                                  \
    two_sum(s, so, t, e);                         \
    s = t;                                        \
    c = c + co + e;                               \
  } while (0)
  IMDG_COMB(0xb1, 0xf);
  IMDG_COMB(0x4e, 0xf);
  IMDG_COMB(0x141, 0xf);
  IMDG_COMB(0x140, 0xf);
  IMDG_COMB(0x142, 0xa);
  IMDG_COMB(0x143, 0xc);
#undef IMDG_COMB
  return lane63_d(s + c);
}

__device__ __forceinline__ float rmin(float a, float b) { return fminf(a, b); }
__device__ __forceinline__ double rmin(double a, double b) { return fmin(a, b); }
__device__ __forceinline__ float rmax0(float a) { return fmaxf(a, 0.0f); }
__device__ __forceinline__ double rmax0(double a) { return fmax(a, 0.0); }
__device__ __forceinline__ float rfract(float t) {
  return __builtin_amdgcn_fractf(t);
}
__device__ __forceinline__ double rfract(double t) {
  return __builtin_amdgcn_fract(t);
}

// Segment index and fraction of IMD's 3-point table access
// (src/potaccess.h:329-340): argument clamped to [begin, end], segment
// k = floor((x - begin) / step) capped at len - 1, fraction
// chi = t - floor(t) before the cap (t >= 0, so floor(t) = (int)t; the
// subtraction is exact).  A NaN argument clamps to segment 0.
template <typename R>
__device__ __forceinline__ int seg_locate(R x, R begin, R end, R invstep,
                                          int len, R& chi) {
  R t = rmax0(rmin(x, end) - begin) * invstep;
  int k = (int)t;
  chi = rfract(t);
  return k < len - 1 ? k : len - 1;
}

// IMD's 3-point interpolation on segment k from the knots (p0_k, dv_k) and
// (p0_k+1, dv_k+1), with dv_k = t[k+1] - t[k] and the second difference
// d2v = dv_k+1 - dv_k = t[k+2] - 2 t[k+1] + t[k] (src/potaccess.h:345-353):
// value p0 + chi (dv + (chi - 1)/2 d2v), and twice the derivative with
// respect to the tabulated argument, 2 istep (dv + (chi - 1/2) d2v).
template <typename R, typename R2>
__device__ __forceinline__ R knot_val(R2 a, R2 b, R chi) {
  R d2v = b.y - a.y;
  return a.x + chi * (a.y + (R)0.5 * (chi - (R)1) * d2v);
}
template <typename R, typename R2>
__device__ __forceinline__ R knot_grad(R2 a, R2 b, R chi, R twoistep) {
  R d2v = b.y - a.y;
  return twoistep * (a.y + (chi - (R)0.5) * d2v);
}

// The 4-point and spline interpolations (src/potaccess.h:365-457) are cubic
// in the fraction x of segment k; their tables hold two knots per segment,
// (c0, c1) and (c2, c3): value c0 + x (c1 + x (c2 + x c3)), twice the
// derivative 2 istep (c1 + x (2 c2 + 3 x c3)).  tab_* pick the segment's
// first knot and evaluate it in either form (CUB: cubic segments; else the
// 3-point knots k, k+1).
template <typename R, typename R2>
__device__ __forceinline__ R cub_val(R2 a, R2 b, R x) {
  return a.x + x * (a.y + x * (b.x + x * b.y));
}
template <typename R, typename R2>
__device__ __forceinline__ R cub_grad(R2 a, R2 b, R x, R twoistep) {
  return twoistep * (a.y + x * ((R)2 * b.x + (R)3 * x * b.y));
}
template <bool CUB>
__device__ __forceinline__ int tab_knot(int k) {
  return CUB ? 2 * k : k;
}
template <bool CUB, typename R, typename R2>
__device__ __forceinline__ R tab_val(R2 a, R2 b, R x) {
  if (CUB) return cub_val<R>(a, b, x);
  return knot_val<R>(a, b, x);
}
template <bool CUB, typename R, typename R2>
__device__ __forceinline__ R tab_grad(R2 a, R2 b, R x, R twoistep) {
  if (CUB) return cub_grad<R>(a, b, x, twoistep);
  return knot_grad<R>(a, b, x, twoistep);
}
// Entry m of slot i in the grouped list layout (4 entries per lane).
__device__ __forceinline__ size_t nbr_index(int i, int m, int kmax) {
  return (((size_t)(i >> 6) * (kmax >> 2) + (m >> 2)) * IMDG_WAVE + (i & 63)) *
             IMDG_GROUP +
         (m & 3);
}

// First uint4 of slot i's list; group g is at + g * IMDG_WAVE.
__device__ __forceinline__ const uint4* list_of(const uint32_t* nbr, int i,
                                                int kmax) {
  return reinterpret_cast<const uint4*>(nbr) +
         ((size_t)(i >> 6) * (kmax >> 2)) * IMDG_WAVE + (i & 63);
}

// Byte address of slot i's first 16-bit entry (group 0) in the 16-bit
// format; group g is at + g * 512 bytes, entry m % 4 at + 2 (m % 4).
__device__ __forceinline__ const char* list16_of(const uint32_t* nbr, int i,
                                                 int kmax) {
  return reinterpret_cast<const char*>(nbr) + (size_t)(i >> 6) * kmax * 256 +
         (size_t)(i & 63) * 8;
}

__device__ __forceinline__ void cell_coords(const RepDev& R, int cell,
                                            int& cx, int& cy, int& cz) {
  int lc = cell - R.cell_off;
  cz = lc % R.gdim[2];
  int q = lc / R.gdim[2];
  cy = q % R.gdim[1];
  cx = q / R.gdim[1];
}

// Centre of a cell: sum_d (c_d + 1/2) box_d / gdim_d.
__device__ __forceinline__ void cell_centre(const RepDev& R, int cell,
                                            double* c) {
  int cx, cy, cz;
  cell_coords(R, cell, cx, cy, cz);
  double fx = cx + 0.5, fy = cy + 0.5, fz = cz + 0.5;
#pragma unroll
  for (int e = 0; e < 3; e++)
    c[e] = fx * R.cvec[0][e] + fy * R.cvec[1][e] + fz * R.cvec[2][e];
}

// Squared displacement since the last list build (check_nblist's test,
// src/imd_forces_nbl.c:2016-2024), FP64 with separate roundings.
__device__ __forceinline__ double disp2(double4 a, double4 b) {
#pragma clang fp contract(off)
  double d0 = a.x - b.x, d1 = a.y - b.y, d2 = a.z - b.z;
  return d0 * d0 + d1 * d1 + d2 * d2;
}

// Pair-only systems: the records the step number `step` gathers, rec_a in
// even steps and rec_b in odd ones (the step's integration writes the other).
template <typename P>
__device__ __forceinline__ P* pair_records(P* rec_a, P* rec_b, long step) {
  return (step & 1) ? rec_b : rec_a;
}

// Make the LDS stores of this wavefront visible to its own later loads
// (no block barrier: the waves of a block run independent schedules).
__device__ __forceinline__ void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// End of a rebuild, by one block: the longest list; on an overflow (of the
// list or of a cell's bucket) freeze the state (the host enlarges what
// overflowed and runs the chain again from the old buffers), otherwise clear
// the rebuild flags and flip the buffers that k_sort filled.  red: two ints
// per wavefront.  In a step with EAM it runs in block 0 of the density loop:
// nothing else in that kernel reads what it writes, except frozen, and the
// outputs of a density loop that goes on are computed again.  (The force
// loop reads the flip, so a pair-only step ends its rebuild before it.)
__device__ inline void list_done(const ListEnd& e, int* red) {
  if (!e.ctl->any_rebuild || e.ctl->frozen) return;
  const int nw = blockDim.x / IMDG_WAVE, w = threadIdx.x / IMDG_WAVE;
  const int over = e.ctl->cell_over;
  int m = 0, fb = 0;
  if (!over)
    for (int b = threadIdx.x; b < e.nblk; b += blockDim.x)
      if (e.rst[e.blk_rep[b >> e.blk_shift]].need_rebuild) {
        const int v = e.blkmax[b];
        m = max(m, v & ~IMDG_BLK_FALLBACK);
        fb += v & IMDG_BLK_FALLBACK ? 1 : 0;
      }
  for (int o = 32; o > 0; o >>= 1) {
    m = max(m, __shfl_xor(m, o, IMDG_WAVE));
    fb += __shfl_xor(fb, o, IMDG_WAVE);
  }
  if ((threadIdx.x % IMDG_WAVE) == 0) {
    red[w] = m;
    red[nw + w] = fb;
  }
  __syncthreads();
  if (threadIdx.x >= IMDG_WAVE) return;
  for (int k = 1; k < nw; k++) {
    m = max(m, red[k]);
    fb += red[nw + k];
  }
  m = max(m, red[0]);
  const bool full = over || m > e.kmax;
  if (!full)
    for (int q = threadIdx.x; q < e.nrep; q += IMDG_WAVE)
      if (e.rst[q].need_rebuild) {
        e.rst[q].rebuilt = 1;
        e.rst[q].nbl_count += 1;
        e.rst[q].need_rebuild = 0;
      }
  if (threadIdx.x != 0) return;
  e.ctl->tiles_fallback += fb;
  if (m > e.ctl->kmax_seen) e.ctl->kmax_seen = m;
  if (full) {
    // keep the rebuild flags: the host grows the list and builds again
    e.ctl->overflow = 1;
    e.ctl->frozen = 1;
  } else {
    e.ctl->pos_cur ^= 1;
    e.ctl->rec_cur ^= 1;
    e.ctl->any_rebuild = 0;
  }
}

}  // namespace imdg
