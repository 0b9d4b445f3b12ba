// The dense AO two-electron tensor (ij|kl) on the GPU, for the quarter
// transform out[i][j][k][p] = sum_l (ij|kl) C[l][p] that the reference's
// ERI::quarter_trans computes (libint2_direct.cpp:913-1141) for the MO
// transforms of scf/src/eri/moeri.cpp.  The tensor is N^4 doubles, so this
// path is for small systems (N of a few hundred at most; 288 GB of HBM holds
// N = 400 with room to spare).  engine.cpp applies C with rocBLAS GEMMs.
//
// The tensor holds every quartet, so its shell-pair tables are made here
// without the J/K engine's cuts; the class kernels are in eri_dense_coop.hpp.
#include <hip/hip_runtime.h>

#include "eri_dense.hpp"

namespace qfe {

__global__ __launch_bounds__(256) void k_dense_pairs(DFBasisView b, const int2* __restrict__ pairs,
                                                     const int* __restrict__ prim0, int npair,
                                                     PairHdr* __restrict__ hdr, double4* __restrict__ ppos,
                                                     double* __restrict__ pk) {
  // one wave per pair, a lane per primitive pair
  const int i = (int)((blockIdx.x * blockDim.x + threadIdx.x) >> 6), lane = (int)(threadIdx.x & 63);
  if (i >= npair) return;
  const int sa = pairs[i].x, sb = pairs[i].y;
  const int na = b.po[sa + 1] - b.po[sa], nb = b.po[sb + 1] - b.po[sb];
  double A[3], B[3], AB2 = 0.0;
  for (int d = 0; d < 3; ++d) {
    A[d] = b.cen[3 * sa + d];
    B[d] = b.cen[3 * sb + d];
    AB2 += (A[d] - B[d]) * (A[d] - B[d]);
  }
  const int p0 = prim0[i];
  for (int k = lane; k < na * nb; k += 64) {
    const int ia = b.po[sa] + k / nb, ib = b.po[sb] + k % nb;
    const double x = b.exps[ia], y = b.exps[ib], p = x + y;
    ppos[p0 + k] = make_double4(p, (x * A[0] + y * B[0]) / p, (x * A[1] + y * B[1]) / p, (x * A[2] + y * B[2]) / p);
    pk[p0 + k] = b.coefs[ia] * b.coefs[ib] * exp(-x * y / p * AB2) / p;
  }
  if (lane == 0) {
    PairHdr h;
    for (int d = 0; d < 3; ++d) {
      h.A[d] = A[d];
      h.B[d] = B[d];
    }
    h.prim0 = p0;
    h.nprim = na * nb;
    h.sa = sa;
    h.sb = sb;
    h.bfa = b.bf0[sa];
    h.bfb = b.bf0[sb];
    h.cls = b.l[sa] * (b.l[sa] + 1) / 2 + b.l[sb];
    h.pstride = 1;
    hdr[i] = h;
  }
}

void launch_dense_pairs(const DFBasisView& b, const int2* pairs, const int* prim0, int npair, PairHdr* hdr,
                        double4* ppos, double* pk, hipStream_t s) {
  if (npair <= 0) return;
  hipLaunchKernelGGL(k_dense_pairs, dim3((npair + 3) / 4), dim3(256), 0, s, b, pairs, prim0, npair, hdr, ppos, pk);
}

}  // namespace qfe
