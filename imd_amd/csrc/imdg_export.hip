// imdg_export.hip -- per-atom results in input order, converted to FP64 on
// the device, so that a download is one contiguous copy per array.
//
// The state lives in slot order (sorted by cell) and in the force
// precision; the caller wants input order and doubles.  Doing the
// permutation on the host reads every slot array back (216 B per atom with
// the padding of the float4 records), widens it and scatters it with one
// thread: 109 ms for 2,048,000 atoms.  Here one thread per slot reads its
// slot's records and stores the 12 doubles at the atom's input index; the
// stores are 8 and 24 B pieces in scattered order (about 0.4 ms at
// 2,048,000 atoms), and what is left is the 96 B per atom that the caller
// asked for, over PCIe into pages that the caller touches for the first
// time: about 28 ms.
#include "imdg_device.h"

namespace imdg {

// Arrays of the caller's order: x, p, f (3 per atom) and epot, rho, df (1
// per atom), each for the m atoms from in0 on; NULL where not wanted.
template <typename R>
__global__ void __launch_bounds__(IMDG_BLOCK)
    k_export(StepArgs<R> a, const int* aid0, const int* aid1, long natoms,
             long in0, long m, ExportDst d) {
  const int b = blockIdx.x;
  const RepDev& Rp = a.rep[a.blk_rep[b]];
  const int s = b * IMDG_BLOCK + threadIdx.x;
  if (s - Rp.atom_off >= Rp.natoms) return;
  long in = (a.ctl->rec_cur ? aid1 : aid0)[s];
  if (in < 0 || in >= natoms) {
    a.ctl->export_bad = 1;  // every writer stores the same value
    return;
  }
  in -= in0;
  if (in < 0 || in >= m) return;
  const int pc = a.ctl->pos_cur;
  if (d.x) {
    const double4 v = a.pos[pc][s];
    d.x[3 * in] = v.x;
    d.x[3 * in + 1] = v.y;
    d.x[3 * in + 2] = v.z;
  }
  if (d.p) {
    const double4 v = a.mom[pc][s];
    d.p[3 * in] = v.x;
    d.p[3 * in + 1] = v.y;
    d.p[3 * in + 2] = v.z;
  }
  if (d.f) {
    const typename V4<R>::T v = a.frc[s];
    d.f[3 * in] = (double)v.x;
    d.f[3 * in + 1] = (double)v.y;
    d.f[3 * in + 2] = (double)v.z;
  }
  if (d.epot) d.epot[in] = (double)a.epot[s];
  if (d.rho) d.rho[in] = a.has_eam ? (double)a.rho[s] : 0.0;
  if (d.df) d.df[in] = a.has_eam ? (double)a.rec_b[s].w : 0.0;
}

// ncomp doubles per slot to input order (the stress tensor), the m atoms from
// in0 on.
__global__ void __launch_bounds__(IMDG_BLOCK)
    k_unsort(const RepDev* rep, Ctl* ctl, const int* blk_rep, const int* aid0,
             const int* aid1, long natoms, long in0, long m,
             const double* src, int ncomp, double* dst) {
  const int b = blockIdx.x;
  const RepDev& Rp = rep[blk_rep[b]];
  const int s = b * IMDG_BLOCK + threadIdx.x;
  if (s - Rp.atom_off >= Rp.natoms) return;
  long in = (ctl->rec_cur ? aid1 : aid0)[s];
  if (in < 0 || in >= natoms) {
    ctl->export_bad = 1;
    return;
  }
  in -= in0;
  if (in < 0 || in >= m) return;
  for (int q = 0; q < ncomp; q++)
    dst[in * ncomp + q] = src[(size_t)s * ncomp + q];
}

template <typename R>
hipError_t launch_export(const StepArgs<R>& a, int* const aid[2], long natoms,
                         long in0, long m, const ExportDst& d, int nblk,
                         hipStream_t st) {
  hipLaunchKernelGGL((k_export<R>), dim3(nblk), dim3(IMDG_BLOCK), 0, st, a,
                     aid[0], aid[1], natoms, in0, m, d);
  return hipGetLastError();
}

hipError_t launch_unsort(const RepDev* rep, Ctl* ctl, const int* blk_rep,
                         int* const aid[2], long natoms, long in0, long m,
                         const double* src, int ncomp, double* dst, int nblk,
                         hipStream_t st) {
  hipLaunchKernelGGL(k_unsort, dim3(nblk), dim3(IMDG_BLOCK), 0, st, rep, ctl,
                     blk_rep, aid[0], aid[1], natoms, in0, m, src, ncomp, dst);
  return hipGetLastError();
}

template hipError_t launch_export<float>(const StepArgs<float>&,
                                         int* const[2], long, long, long,
                                         const ExportDst&, int, hipStream_t);
template hipError_t launch_export<double>(const StepArgs<double>&,
                                          int* const[2], long, long, long,
                                          const ExportDst&, int, hipStream_t);

}  // namespace imdg
