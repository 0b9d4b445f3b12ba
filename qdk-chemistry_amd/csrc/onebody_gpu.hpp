// One-electron integrals on the GPU (kernels in onebody_gpu.hip).
#pragma once

#include <hip/hip_runtime.h>

#include "eri_core.hpp"

namespace qfe {

// Device view of a basis: per shell l, atom, centre (3 doubles), primitive
// range [po[s], po[s+1]) into exps/coefs (normalised contraction
// coefficients), first output function bf0[s]; per atom the nuclear charge
// seen by the electrons Z and the position R (3 doubles); the solid-harmonic
// table sph[l][m][c] (5 x 9 x 15 doubles); per shell the norm of x^l times its
// radial part, and the sum of the charges' magnitudes zsum (the scales of the
// cut on primitive pairs).  Shells up to l = 3; by_l holds the
// shell indices by angular momentum, those of l in [nl[l], nl[l + 1]).
struct OneBodyView {
  const int* l;
  const int* atom;
  const int* po;
  const int* bf0;
  const double* cen;
  const double* exps;
  const double* coefs;
  const double* Z;
  const double* R;
  const double* sph;
  const double* norm;
  double zsum;
  const int* by_l;
  int nl[5];
  int nsh, natoms, nbf, pure;
};

// op 0 = S, 1 = T, 2 = V into out (nbf x nbf, row-major, device)
void launch_one_body(const OneBodyView& b, const RysArgs& ra, int op, double* out, hipStream_t s);
// sum_mn W_mn dO_mn/dR added to ncopy copies of grad[natoms][3] (device, 3
// natoms apart, zeroed by the caller, a power of two of them)
void launch_one_body_grad(const OneBodyView& b, const RysArgs& ra, int op, const double* W, double* grad, int ncopy,
                          hipStream_t s);

}  // namespace qfe
