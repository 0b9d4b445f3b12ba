// Cooperative nuclear-gradient kernel: one block per canonical shell quartet
// (the contraction of eri_grad.hpp, ERI::get_gradients,
// libint2_direct.cpp:646-890).
//
// For every (primitive quartet, root) combination of a batch, three lanes
// build the 1-D integrals with one extra unit on A, B and C in LDS.  Each
// cartesian component then sums its nine derivatives (centres A, B, C) over
// the batch and applies its Coulomb and exchange weights once: the weights
// do not depend on the combination.
//
// Why a block per quartet: one thread per quartet with runtime angular
// momenta kept its tables in 30 KB of scratch a lane, and every launch of
// such a kernel waited for the runtime to set that scratch up (about 55 ms a
// class): 1861 ms for one water molecule in def2-TZVP, 46 ms with this
// kernel.  The component phase is bound by its LDS reads (21 a component and
// combination for about 45 FP64 operations).
#pragma once

#include "eri_coop.hpp"
#include "eri_grad.hpp"

namespace qfe {

template <int LA_, int LB_, int LC_, int LD_>
struct GradCoop {
  static constexpr int LA = LA_, LB = LB_, LC = LC_, LD = LD_;
  static constexpr int L = LA + LB + LC + LD;
  static constexpr int NR = (L + 1) / 2 + 1;
  static constexpr int NA = ncart(LA), NB = ncart(LB), NC = ncart(LC), ND = ncart(LD);
  static constexpr int NCOMP = NA * NB * NC * ND;
  // strides of the 1-D tables, and their size (odd, so that the lanes of the
  // first phase store to different banks)
  static constexpr int SD = 1, SC = LD + 1, SB = (LC + 2) * SC, SA = (LB + 2) * SB;
  static constexpr int NI = ((LA + 2) * SA) | 1;
  // one wave per quartet; four for the largest blocks
  static constexpr int BLK = NCOMP >= 1000 ? 256 : 64;
  // combinations per batch: three lanes each, at most 32 KB of tables
  static constexpr int CM_LDS = 4096 / (3 * NI) < 1 ? 1 : 4096 / (3 * NI);
  static constexpr int CM = BLK / 3 < CM_LDS ? BLK / 3 : CM_LDS;
  // density blocks: ab, cd, then ac, bd, ad, bc per spin
  static constexpr int NX = NA * NC + NB * ND + NA * ND + NB * NC;
  static constexpr int NDEN = NA * NB + NC * ND + 2 * NX;
  static constexpr int LDS = CM * 3 * NI + CM * 3 + NDEN;  // doubles
  // threads of the component phase: NSL slices of the batch's combinations
  static constexpr int NSL = NCOMP >= BLK ? 1 : BLK / NCOMP;
};

template <class G>
__global__ __launch_bounds__(G::BLK) void k_eri_grad_coop(
    const int2* __restrict__ tasks, long long ntask, const PairHdr* __restrict__ pairs,
    const double4* __restrict__ ppos, const double* __restrict__ pk, const double* __restrict__ pa, RysArgs ra,
    const double* __restrict__ sph, const double* __restrict__ P, const double* __restrict__ Pk,
    const double* __restrict__ Pk2, int nbf, const int* __restrict__ sh_atom, int natoms, double kscale,
    int ncopy, double* __restrict__ gJ, double* __restrict__ gK) {
  gJ += (size_t)(blockIdx.x & (unsigned)(ncopy - 1)) * 6 * natoms;
  gK += (size_t)(blockIdx.x & (unsigned)(ncopy - 1)) * 6 * natoms;
  constexpr double TWO_PI_52 = 34.98683665524972;
  __shared__ double tab[G::CM * 3 * G::NI];
  __shared__ double par[G::CM * 3];
  __shared__ double den[G::NDEN];
  __shared__ double red[18];
  double* const dab = den;
  double* const dcd = den + G::NA * G::NB;
  const int tid = (int)threadIdx.x;
  for (long long t = blockIdx.x; t < ntask; t += gridDim.x) {
    const int2 tk = tasks[t];
    const PairHdr bra = pairs[tk.x], ket = pairs[tk.y];
    const int nspin = Pk2 ? 2 : 1;
    __syncthreads();  // the last task's readers are done
    if (tid < 18) red[tid] = 0.0;
    for (int i = tid; i < G::NA * G::NB; i += G::BLK)
      dab[i] = coop_cart_density<G::LA, G::LB>(P, nbf, sph, bra.bfa, bra.bfb, i / G::NB, i % G::NB);
    for (int i = tid; i < G::NC * G::ND; i += G::BLK)
      dcd[i] = coop_cart_density<G::LC, G::LD>(P, nbf, sph, ket.bfa, ket.bfb, i / G::ND, i % G::ND);
    for (int sp = 0; sp < nspin; ++sp) {
      const double* D = sp ? Pk2 : Pk;
      double* x = dcd + G::NC * G::ND + sp * G::NX;
      for (int i = tid; i < G::NA * G::NC; i += G::BLK)
        x[i] = coop_cart_density<G::LA, G::LC>(D, nbf, sph, bra.bfa, ket.bfa, i / G::NC, i % G::NC);
      x += G::NA * G::NC;
      for (int i = tid; i < G::NB * G::ND; i += G::BLK)
        x[i] = coop_cart_density<G::LB, G::LD>(D, nbf, sph, bra.bfb, ket.bfb, i / G::ND, i % G::ND);
      x += G::NB * G::ND;
      for (int i = tid; i < G::NA * G::ND; i += G::BLK)
        x[i] = coop_cart_density<G::LA, G::LD>(D, nbf, sph, bra.bfa, ket.bfb, i / G::ND, i % G::ND);
      x += G::NA * G::ND;
      for (int i = tid; i < G::NB * G::NC; i += G::BLK)
        x[i] = coop_cart_density<G::LB, G::LC>(D, nbf, sph, bra.bfb, ket.bfa, i / G::NC, i % G::NC);
    }
    const double deg =
        (bra.sa == bra.sb ? 1.0 : 2.0) * (ket.sa == ket.sb ? 1.0 : 2.0) * (tk.x == tk.y ? 1.0 : 2.0);
    const double wj = 0.5 * deg, wk = (Pk2 ? -0.25 : -0.125) * kscale * deg;
    double gj[9], gk[9];
    sfor<9>([&](auto i) { gj[i] = gk[i] = 0.0; });
    const int ncomb = bra.nprim * ket.nprim * G::NR;
    for (int g0 = 0; g0 < ncomb; g0 += G::CM) {
      const int nc = ncomb - g0 < G::CM ? ncomb - g0 : G::CM;
      // phase 1: lane (combination, direction)
      if (tid < 3 * nc) {
        const int i = tid / 3, x = tid % 3;
        const int pr = (g0 + i) / G::NR, r = (g0 + i) % G::NR;
        const int ib = bra.prim0 + pr % bra.nprim * bra.pstride, ik = ket.prim0 + pr / bra.nprim * ket.pstride;
        const double4 Pp = ppos[ib], Q = ppos[ik];
        const double p = Pp.x, q = Q.x;
        const double PQx = Pp.y - Q.y, PQy = Pp.z - Q.z, PQz = Pp.w - Q.w;
        const double rs = frsq(p + q), rpq = rs * rs;
        const double T = p * q * rpq * (PQx * PQx + PQy * PQy + PQz * PQz);
        double ur, wr;
        rys_root_one<G::NR>(T, ra, r, ur, wr);
        const double PQ = x == 0 ? PQx : (x == 1 ? PQy : PQz);
        const double Pc = x == 0 ? Pp.y : (x == 1 ? Pp.z : Pp.w), Qc = x == 0 ? Q.y : (x == 1 ? Q.z : Q.w);
        const double Ac = x == 0 ? bra.A[0] : (x == 1 ? bra.A[1] : bra.A[2]);
        const double Bc = x == 0 ? bra.B[0] : (x == 1 ? bra.B[1] : bra.B[2]);
        const double Cc = x == 0 ? ket.A[0] : (x == 1 ? ket.A[1] : ket.A[2]);
        const double Dc = x == 0 ? ket.B[0] : (x == 1 ? ket.B[1] : ket.B[2]);
        const double h2p = 0.5 * frcp(p), h2q = 0.5 * frcp(q);
        const double xa = q * rpq * ur, xc = p * rpq * ur;
        const double s = x == 2 ? wr * (TWO_PI_52 * pk[ib] * pk[ik] * rs) : 1.0;
        rys_1d_store<G::LA + G::LB + 1, G::LC + G::LD + 1, G::LA + 1, G::LB + 1, G::LC + 1, G::LD>(
            s, (Pc - Ac) - xa * PQ, (Qc - Cc) + xc * PQ, 0.5 * rpq * ur, h2p - h2p * xa, h2q - h2q * xc, Ac - Bc,
            Cc - Dc, tab + (i * 3 + x) * G::NI);
        if (x == 0) {
          par[3 * i] = 2.0 * pa[ib];
          par[3 * i + 1] = 2.0 * (p - pa[ib]);
          par[3 * i + 2] = 2.0 * pa[ik];
        }
      }
      __syncthreads();
      // phase 2: thread (slice, component)
      for (int c0 = tid; c0 < G::NCOMP * G::NSL; c0 += G::BLK) {
        const int sl = c0 / G::NCOMP, cm = c0 % G::NCOMP;
        const int cd = cm % G::ND, cc = cm / G::ND % G::NC, cb = cm / (G::ND * G::NC) % G::NB,
                  ca = cm / (G::ND * G::NC * G::NB);
        int ea[3], eb[3], ec[3], ed[3];
        coop_xyz<G::LA>(ca, ea[0], ea[1], ea[2]);
        coop_xyz<G::LB>(cb, eb[0], eb[1], eb[2]);
        coop_xyz<G::LC>(cc, ec[0], ec[1], ec[2]);
        coop_xyz<G::LD>(cd, ed[0], ed[1], ed[2]);
        int o[3], dA[3], dB[3], dC[3];
        double fa[3], fb[3], fc[3];
        sfor<3>([&](auto x) {
          o[x] = ea[x] * G::SA + eb[x] * G::SB + ec[x] * G::SC + ed[x];
          // the lowered entry (any valid one where its factor is zero)
          dA[x] = ea[x] ? G::SA : 0;
          dB[x] = eb[x] ? G::SB : 0;
          dC[x] = ec[x] ? G::SC : 0;
          fa[x] = (double)ea[x];
          fb[x] = (double)eb[x];
          fc[x] = (double)ec[x];
        });
        double S[9];
        sfor<9>([&](auto i) { S[i] = 0.0; });
        for (int i = sl; i < nc; i += G::NSL) {
          const double* tb = tab + i * 3 * G::NI;
          const double ta = par[3 * i], tbb = par[3 * i + 1], tg = par[3 * i + 2];
          double v[3];
          sfor<3>([&](auto x) { v[x] = tb[x * G::NI + o[x]]; });
          sfor<3>([&](auto x) {
            const double* e = tb + x * G::NI + o[x];
            const double ot = v[(x + 1) % 3] * v[(x + 2) % 3];
            double a = ta * e[G::SA], b = tbb * e[G::SB], c = tg * e[G::SC];
            if constexpr (G::LA > 0) a = fma(-fa[x], e[-dA[x]], a);
            if constexpr (G::LB > 0) b = fma(-fb[x], e[-dB[x]], b);
            if constexpr (G::LC > 0) c = fma(-fc[x], e[-dC[x]], c);
            S[x] = fma(a, ot, S[x]);
            S[3 + x] = fma(b, ot, S[3 + x]);
            S[6 + x] = fma(c, ot, S[6 + x]);
          });
        }
        const double wJ = wj * dab[ca * G::NB + cb] * dcd[cc * G::ND + cd];
        double wK = 0.0;
        for (int sp = 0; sp < nspin; ++sp) {
          const double* xac = dcd + G::NC * G::ND + sp * G::NX;
          const double* xbd = xac + G::NA * G::NC;
          const double* xad = xbd + G::NB * G::ND;
          const double* xbc = xad + G::NA * G::ND;
          wK = fma(xac[ca * G::NC + cc], xbd[cb * G::ND + cd], wK);
          wK = fma(xad[ca * G::ND + cd], xbc[cb * G::NC + cc], wK);
        }
        wK *= wk;
        sfor<9>([&](auto i) {
          gj[i] = fma(wJ, S[i], gj[i]);
          gk[i] = fma(wK, S[i], gk[i]);
        });
      }
      __syncthreads();
    }
    // nine sums each over the block; D by translation invariance
    sfor<9>([&](auto i) {
      gj[i] = wave_sum(gj[i]);
      gk[i] = wave_sum(gk[i]);
    });
    if constexpr (G::BLK > 64) {
      if ((tid & 63) == 0)
        sfor<9>([&](auto i) {
          atomicAdd(&red[i], gj[i]);
          atomicAdd(&red[9 + i], gk[i]);
        });
    } else if (tid == 0) {
      sfor<9>([&](auto i) {
        red[i] = gj[i];
        red[9 + i] = gk[i];
      });
    }
    __syncthreads();
    if (tid < 24) {  // (J or K, centre, direction)
      const int k = tid / 12, c = tid / 3 % 4, x = tid % 3;
      const double* r = red + 9 * k;
      const double v = c < 3 ? r[3 * c + x] : -(r[x] + r[3 + x] + r[6 + x]);
      const int sh = c == 0 ? bra.sa : (c == 1 ? bra.sb : (c == 2 ? ket.sa : ket.sb));
      unsafeAtomicAdd((k ? gK : gJ) + sh_atom[sh] + x * natoms, v);
    }
  }
}

template <int LA, int LB, int LC, int LD>
void grad_coop(const GradLaunch& a, hipStream_t s) {
  using G = GradCoop<LA, LB, LC, LD>;
  if (a.ntask <= 0) return;
  if (a.sph == nullptr) throw std::runtime_error("solid-harmonic table missing for the cooperative gradient kernel");
  const long long grid = std::min(a.ntask, 65536LL);
  hipLaunchKernelGGL((k_eri_grad_coop<G>), dim3((unsigned)grid), dim3(G::BLK), 0, s, a.tasks, a.ntask, a.pairs, a.ppos,
                     a.pk, a.pa, *a.ra, a.sph, a.P, a.Pk, a.Pk2, a.nbf, a.sh_atom, a.natoms, a.kscale,
                     a.ncopy, a.gJ, a.gK);
}

}  // namespace qfe
