// The dense AO two-electron tensor for the quarter and MO transforms
// (pair tables in eri_dense.hip, class kernels in eri_dense_coop.hpp).
#pragma once

#include <hip/hip_runtime.h>

#include "dfj.hpp"
#include "eri_core.hpp"

namespace qfe {

// Headers and primitive tables of the shell pairs pairs[0, npair) (the higher
// l first), every primitive pair kept: pair i has the entries [prim0[i],
// prim0[i] + products of the contraction lengths) of ppos and pk
void launch_dense_pairs(const DFBasisView& b, const int2* pairs, const int* prim0, int npair, PairHdr* hdr,
                        double4* ppos, double* pk, hipStream_t s);

// One class of the tensor: every quartet of a bra pair and a ket pair (tri:
// bra and ket are the same list, each unordered pair of them once), stored at
// its eight permutation-equivalent places of eri (nbf^4, row-major)
struct DenseLaunch {
  const PairHdr* bra;
  int nbra;
  const PairHdr* ket;
  int nket;
  bool tri;
  const double4* ppos;
  const double* pk;
  int nbf;
  double* eri;
};
// bra class cb >= ket class ck, shells up to d, solid harmonics
void launch_dense(int cb, int ck, const DenseLaunch& a, const RysArgs& ra, hipStream_t s);

}  // namespace qfe
