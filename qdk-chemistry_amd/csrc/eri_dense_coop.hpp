// Dense AO tensor, one block per canonical shell quartet of a class: the
// solid-harmonic block (eri_jk_coop.hpp's coop_quartet) stored at its eight
// permutation-equivalent places.
//
// The bound is the store of nbf^4 doubles; a thread per quartet with runtime
// angular momenta kept its block and tables in 21 KB of scratch a lane and
// took 29 ms for the 85 million elements of (H2O)4/cc-pVDZ (23 GB/s); the 21
// class kernels take 3.0 ms (230 GB/s), 0.3-0.5 ms each for the classes of s
// and p shells, whose many small quartets cost a block's latency each.
#pragma once

#include "eri_dense.hpp"
#include "eri_jk_coop.hpp"

namespace qfe {

template <class G>
__global__ __launch_bounds__(G::BLK) void k_eri_dense(DenseLaunch a, RysArgs ra) {
  extern __shared__ double lds[];
  const int tid = (int)threadIdx.x;
  const CoopOffsets<G> of(tid);
  const size_t n = (size_t)a.nbf, nn = n * n;
  const long long ntask = a.tri ? (long long)a.nbra * (a.nbra + 1) / 2 : (long long)a.nbra * a.nket;
  constexpr int MA = G::MA, MB = G::MB, MC = G::MC, MD = G::MD;
  for (long long t = blockIdx.x; t < ntask; t += gridDim.x) {
    int p, q;
    if (a.tri) {  // row p >= column q of the lower triangle
      p = (int)((sqrt(8.0 * (double)t + 1.0) - 1.0) / 2.0);
      while ((long long)p * (p + 1) / 2 > t) --p;
      while ((long long)(p + 1) * (p + 2) / 2 <= t) ++p;
      q = (int)(t - (long long)p * (p + 1) / 2);
    } else {
      p = (int)(t / a.nket);
      q = (int)(t % a.nket);
    }
    const PairHdr bra = a.bra[p], ket = a.ket[q];
    __syncthreads();  // the last quartet's block has been read
    const double* V = coop_quartet<G>(bra, ket, a.ppos, a.pk, nullptr, ra, 0.0, of, lds);
    const size_t fa = bra.bfa, fb = bra.bfb, fc = ket.bfa, fd = ket.bfb;
    // each pair of images with the index that is contiguous in memory
    // fastest; where shells coincide two stores hit one element with one value
    for (int e = tid; e < MA * MB * MC * MD; e += G::BLK) {
      {  // d fastest: (ab|cd) and (ba|cd)
        const int i = e / (MD * MC * MB), j = e / (MD * MC) % MB, k = e / MD % MC, l = e % MD;
        const double v = V[e];
        const size_t cd = (fc + k) * n + fd + l;
        a.eri[((fa + i) * n + fb + j) * nn + cd] = v;
        a.eri[((fb + j) * n + fa + i) * nn + cd] = v;
      }
      {  // c fastest: (ab|dc) and (ba|dc)
        const int i = e / (MC * MD * MB), j = e / (MC * MD) % MB, l = e / MC % MD, k = e % MC;
        const double v = V[((i * MB + j) * MC + k) * MD + l];
        const size_t dc = (fd + l) * n + fc + k;
        a.eri[((fa + i) * n + fb + j) * nn + dc] = v;
        a.eri[((fb + j) * n + fa + i) * nn + dc] = v;
      }
      {  // b fastest: (cd|ab) and (dc|ab)
        const int k = e / (MB * MA * MD), l = e / (MB * MA) % MD, i = e / MB % MA, j = e % MB;
        const double v = V[((i * MB + j) * MC + k) * MD + l];
        const size_t ab = (fa + i) * n + fb + j;
        a.eri[((fc + k) * n + fd + l) * nn + ab] = v;
        a.eri[((fd + l) * n + fc + k) * nn + ab] = v;
      }
      {  // a fastest: (cd|ba) and (dc|ba)
        const int k = e / (MA * MB * MD), l = e / (MA * MB) % MD, j = e / MA % MB, i = e % MA;
        const double v = V[((i * MB + j) * MC + k) * MD + l];
        const size_t ba = (fb + j) * n + fa + i;
        a.eri[((fc + k) * n + fd + l) * nn + ba] = v;
        a.eri[((fd + l) * n + fc + k) * nn + ba] = v;
      }
    }
  }
}

template <int LA, int LB, int LC, int LD>
void dense_coop(const DenseLaunch& a, const RysArgs& ra, hipStream_t s) {
  using G = JKCoop<LA, LB, LC, LD>;
  const long long ntask = a.tri ? (long long)a.nbra * (a.nbra + 1) / 2 : (long long)a.nbra * a.nket;
  if (ntask <= 0) return;
  auto kern = k_eri_dense<G>;
  constexpr int bytes = G::WORK * (int)sizeof(double);
  coop_lds(kern, bytes);
  hipLaunchKernelGGL(kern, dim3((unsigned)std::min(ntask, 1LL << 20)), dim3(G::BLK), bytes, s, a, ra);
}

}  // namespace qfe
