// One-electron integrals on the GPU for the SCF: overlap S, kinetic T,
// nuclear attraction V over all shell pairs, and the density-contracted
// nuclear derivatives sum_mn W_mn dO_mn/dR.  The reference evaluates these
// with Libint2 in scf/src/util/int1e.cpp (S :518, T and V and their
// derivatives :473-977).  The recursions are those of the host path
// (onebody.cpp): Obara-Saika 1-D overlaps for S and T (T from the
// second-derivative identity), Rys quadrature for V with the engine's root
// tables (roots of the Boys measure at T = p |PC|^2, C00 = PA - u PC,
// B10 = (1 - u)/2p, horizontal transfer to the second centre).
//
// One wave per shell pair of a class (la lb), angular momenta known at compile
// time: the significant primitive pairs are listed in LDS, and the lanes take
// the (primitive pair, nucleus) combinations in turn, each summing its own
// cartesian block (V) or its nucleus's forces (the V gradient) in registers.
// The kernels are bound by the FP64 work of those combinations; a thread per
// pair with runtime angular momenta kept its tables in 4-6 KB of scratch a
// lane: V took 13 ms and its gradient 14.6 ms at (H2O)24/cc-pVDZ, 0.15 and
// 0.37 ms now.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "eri_core.hpp"
#include "onebody_gpu.hpp"

namespace qfe {

namespace {

constexpr double kPi1 = 3.14159265358979323846;
// A primitive pair is dropped when no element of its S, T, V or derivative
// block can reach this times the norms of its two shells (ob_bound).  The
// prefactor |c_a c_b| exp(-ab/p |AB|^2) alone does not tell: for two f shells
// of exponent 0.05 at 34 bohr it is 1e-18 and S is 1e-9.  A block sums at most
// 4096 primitive pairs, so what is dropped stays ten digits below the rounding
// of an element of order one.  At (H2O)64/cc-pVDZ the cut keeps 29-33 % of the
// primitive pairs (73 % have a prefactor above the FP64 underflow).
constexpr double kPairThr = 1e-30;

// shells of pair t of class (LA LB): every ordered combination for LA > LB,
// the lower triangle for LA == LB
template <int LA, int LB>
__device__ void ob_pair(const OneBodyView& b, long long t, int& s1, int& s2) {
  const int n2 = b.nl[LB + 1] - b.nl[LB];
  int i, j;
  if constexpr (LA == LB) {
    i = (int)((sqrt(8.0 * (double)t + 1.0) - 1.0) / 2.0);
    while ((long long)i * (i + 1) / 2 > t) --i;
    while ((long long)(i + 1) * (i + 2) / 2 <= t) ++i;
    j = (int)(t - (long long)i * (i + 1) / 2);
  } else {
    i = (int)(t / n2);
    j = (int)(t % n2);
  }
  s1 = b.by_l[b.nl[LA] + i];
  s2 = b.by_l[b.nl[LB] + j];
}

template <int LA, int LB>
long long ob_npairs(const OneBodyView& b) {
  const long long n1 = b.nl[LA + 1] - b.nl[LA], n2 = b.nl[LB + 1] - b.nl[LB];
  return LA == LB ? n1 * (n1 + 1) / 2 : n1 * n2;
}

// one primitive pair: exponent sum, P - A, prefactor and the two exponents.
// P - A is formed as -b/p (A - B): the difference of the rounded centres loses
// |A| / |P - A| digits, and the derivatives multiply it by 2a (1e4 and more).
struct ObPrim {
  double p, PA[3], K, a, b;
};

// What an element of a primitive pair's cartesian block of operator op (0 = S,
// 1 = T, 2 = V summed over the nuclei), or of its derivative by a centre, is
// bounded by.  With r the distance from P a polynomial about A or B is at most
// (D + r)^l, D = max(|PA|, |PB|), and the n-th moment of D + r over
// exp(-p r^2), n <= 9, at most (D + 1.75 / sqrt(p))^n = m^n (Minkowski; the
// ninth root of the ninth moment of r is 1.73 / sqrt(p)); 1/|r - C| is largest
// for C = P, where the moments are smaller.  The kinetic energy multiplies the
// second polynomial by lb (lb - 1) / (2 r^2), b (2 lb + 3) and 2 b^2 r^2, a
// derivative the first by 2a r and la / r, the second by 2b r and lb / r.
template <int LA, int LB, int op, bool GRAD>
__device__ double ob_bound(double a, double bb, double AB2, double K, double zsum) {
  constexpr double lb = LB;
  const double p = a + bb, m = ((a > bb ? a : bb) * sqrt(AB2) + 1.75 * sqrt(p)) / p, m2 = m * m;
  double v = fabs(K) * (op == 2 ? 2.0 * kPi1 / p * zsum : kPi1 / p * sqrt(kPi1 / p));
  for (int i = 0; i < LA + LB; ++i) v *= m;
  if constexpr (op == 1) v *= 0.5 * lb * (lb - 1.0) / m2 + bb * (2.0 * lb + 3.0) + 2.0 * bb * bb * m2;
  if constexpr (GRAD) v *= 2.0 * p * m + (LA + LB) / m;
  return v;
}

// The significant ones of the primitive pairs [i0, i0 + 64) of (s1, s2),
// packed into list (64 entries of LDS); returns their number.  Called by the
// whole one-wave block.
template <int LA, int LB, int op, bool GRAD>
__device__ int ob_prims(const OneBodyView& b, int s1, int s2, int i0, int np, ObPrim* list) {
  const int lane = (int)threadIdx.x, i = i0 + lane;
  ObPrim q;
  bool keep = false;
  if (i < np) {
    const int n2 = b.po[s2 + 1] - b.po[s2];
    const int ia = b.po[s1] + i / n2, ib = b.po[s2] + i % n2;
    const double* A = b.cen + 3 * s1;
    const double* B = b.cen + 3 * s2;
    double AB2 = 0.0;
    for (int d = 0; d < 3; ++d) AB2 += (A[d] - B[d]) * (A[d] - B[d]);
    q.a = b.exps[ia];
    q.b = b.exps[ib];
    q.p = q.a + q.b;
    for (int d = 0; d < 3; ++d) q.PA[d] = -q.b / q.p * (A[d] - B[d]);
    q.K = exp(-q.a * q.b / q.p * AB2) * (b.coefs[ia] * b.coefs[ib]);
    // a NaN is kept
    keep = q.K != 0.0 && !(ob_bound<LA, LB, op, GRAD>(q.a, q.b, AB2, q.K, b.zsum) < kPairThr * b.norm[s1] * b.norm[s2]);
  }
  const unsigned long long m = __ballot(keep);
  __syncthreads();  // the last list has been read
  if (keep) list[__popcll(m & ((1ull << lane) - 1ull))] = q;
  __syncthreads();
  return __popcll(m);
}

// 1-D overlaps S[i][j] without the (pi/p)^(1/2) prefactor
template <int I, int J>
__device__ void ob_os1d(double PA, double PB, double o2p, double (&S)[I + 1][J + 1]) {
  sfor<I + 1>([&](auto ii) {
    constexpr int i = ii;
    sfor<J + 1>([&](auto jj) {
      constexpr int j = jj;
      if constexpr (i == 0 && j == 0) {
        S[0][0] = 1.0;
      } else if constexpr (j == 0) {
        double v = PA * S[i - 1][0];
        if constexpr (i >= 2) v += (i - 1) * o2p * S[i - 2][0];
        S[i][0] = v;
      } else {
        double v = PB * S[i][j - 1];
        if constexpr (i >= 1) v += i * o2p * S[i - 1][j - 1];
        if constexpr (j >= 2) v += (j - 1) * o2p * S[i][j - 2];
        S[i][j] = v;
      }
    });
  });
}

// 1-D kinetic integral T(i, j) from the overlaps (ket exponent b)
template <int i, int j, int I, int J>
__device__ double ob_t1(const double (&S)[I][J], double b) {
  double t = -2.0 * b * (2 * j + 1) * S[i][j] + 4.0 * b * b * S[i][j + 2];
  if constexpr (j >= 2) t += j * (j - 1) * S[i][j - 2];
  return -0.5 * t;
}

// 1-D nuclear-attraction integrals I(a, b) of one root, a <= AM, b <= BM,
// a + b <= L
template <int L, int AM, int BM>
__device__ void ob_1d(double s, double C00, double B10, double AB, double (&I)[AM + 1][BM + 1]) {
  double g[L + 1];
  g[0] = s;
  if constexpr (L >= 1) g[1] = C00 * s;
  sfor<(L >= 2 ? L - 1 : 0)>([&](auto ii) {
    constexpr int i = ii + 1;
    g[i + 1] = C00 * g[i] + i * B10 * g[i - 1];
  });
  sfor<BM + 1>([&](auto bb) {
    constexpr int b = bb;
    if constexpr (b > 0) sfor<L + 1 - b>([&](auto i) { g[i] = g[i + 1] + AB * g[i]; });
    sfor<AM + 1>([&](auto a) {
      if constexpr (a + b <= L) I[a][b] = g[a];
    });
  });
}

// Between the components (and roots) of the larger classes: without it the
// scheduler hoists every component's loads and products at once and spills.
template <int LA, int LB>
__device__ __forceinline__ void ob_fence() {
  if constexpr (LA + LB >= 3) {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
  }
}

__device__ double ob_wave_sum(double v) {
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
  return v;
}

// output function m of a shell of momentum l as a sum over cartesians: its
// coefficient of component c
__device__ double ob_coef(const OneBodyView& b, int l, int m, int c) {
  return (b.pure && l >= 2) ? b.sph[(l * 9 + m) * 15 + c] : (m == c ? 1.0 : 0.0);
}
__device__ int ob_nfun(const OneBodyView& b, int l) { return (b.pure && l >= 2) ? 2 * l + 1 : ncart(l); }

}  // namespace

// S, T or V of one shell pair per block (one wave): pair blockIdx.y gridDim.x +
// blockIdx.x of the class's npair
template <int LA, int LB, int op>
__global__ __launch_bounds__(64) void k_one_body(OneBodyView b, RysArgs ra, long long npair,
                                                 double* __restrict__ out) {
  constexpr int NA = ncart(LA), NB = ncart(LB), L = LA + LB, NR = L / 2 + 1;
  __shared__ ObPrim list[64];
  __shared__ double blk[NA * NB];
  const int lane = (int)threadIdx.x;
  const long long t = (long long)blockIdx.y * gridDim.x + blockIdx.x;
  if (t >= npair) return;
  int s1, s2;
  ob_pair<LA, LB>(b, t, s1, s2);
  const int np = (b.po[s1 + 1] - b.po[s1]) * (b.po[s2 + 1] - b.po[s2]);
  double A[3], B[3];
  for (int d = 0; d < 3; ++d) {
    A[d] = b.cen[3 * s1 + d];
    B[d] = b.cen[3 * s2 + d];
  }
  double acc[NA * NB];
  sfor<NA * NB>([&](auto k) { acc[k] = 0.0; });
  for (int i0 = 0; i0 < np; i0 += 64) {
    const int n = ob_prims<LA, LB, op, false>(b, s1, s2, i0, np, list);
    if constexpr (op <= 1) {
      if (lane < n) {
        const ObPrim q = list[lane];
        const double o2p = 0.5 / q.p, s00 = pow(kPi1 / q.p, 1.5) * q.K;
        double S[3][LA + 1][LB + 3];
        sfor<3>([&](auto d) { ob_os1d<LA, LB + 2>(q.PA[d], q.a / q.p * (A[d] - B[d]), o2p, S[d]); });
        sfor<NA * NB>([&](auto k) {
          constexpr int ca = k / NB, cb = k % NB;
          constexpr int ax = cart_x(LA, ca), ay = cart_y(LA, ca), az = cart_z(LA, ca);
          constexpr int bx = cart_x(LB, cb), by = cart_y(LB, cb), bz = cart_z(LB, cb);
          const double x = S[0][ax][bx], y = S[1][ay][by], z = S[2][az][bz];
          double v;
          if constexpr (op == 0)
            v = x * y * z;
          else
            v = ob_t1<ax, bx>(S[0], q.b) * y * z + x * ob_t1<ay, by>(S[1], q.b) * z + x * y * ob_t1<az, bz>(S[2], q.b);
          acc[k] += s00 * v;
          ob_fence<LA, LB>();
        });
      }
    } else {
      for (int c = lane; c < n * b.natoms; c += 64) {
        const ObPrim& q = list[c / b.natoms];
        const int cn = c % b.natoms;
        const double p = q.p;
        double PA[3], PC[3], PC2 = 0.0;
        sfor<3>([&](auto d) {
          PA[d] = q.PA[d];
          PC[d] = PA[d] + (A[d] - b.R[3 * cn + d]);
          PC2 += PC[d] * PC[d];
        });
        double u[NR], w[NR];
        rys_roots<NR>(p * PC2, ra, u, w);
        const double pref = -b.Z[cn] * 2.0 * kPi1 / p * q.K, h2p = 0.5 / p;
        sfor<NR>([&](auto r) {
          double I[3][LA + 1][LB + 1];
          sfor<3>([&](auto d) {
            ob_1d<L, LA, LB>(d == 2 ? w[r] * pref : 1.0, PA[d] - u[r] * PC[d], (1.0 - u[r]) * h2p, A[d] - B[d], I[d]);
          });
          sfor<NA * NB>([&](auto k) {
            constexpr int ca = k / NB, cb = k % NB;
            acc[k] = fma(I[0][cart_x(LA, ca)][cart_x(LB, cb)] * I[1][cart_y(LA, ca)][cart_y(LB, cb)],
                         I[2][cart_z(LA, ca)][cart_z(LB, cb)], acc[k]);
          });
          ob_fence<LA, LB>();
        });
      }
    }
  }
  sfor<NA * NB>([&](auto k) {
    const double v = ob_wave_sum(acc[k]);
    if (lane == k % 64) blk[k] = v;
  });
  __syncthreads();
  const int n1 = ob_nfun(b, LA), n2 = ob_nfun(b, LB);
  const size_t n = (size_t)b.nbf;
  for (int o = lane; o < n1 * n2; o += 64) {
    const int i = o / n2, j = o % n2;
    double v = 0.0;
    for (int c = 0; c < NA; ++c) {
      const double f = ob_coef(b, LA, i, c);
      if (f == 0.0) continue;
      double w = 0.0;
      for (int e = 0; e < NB; ++e) w = fma(ob_coef(b, LB, j, e), blk[c * NB + e], w);
      v = fma(f, w, v);
    }
    out[(size_t)(b.bf0[s1] + i) * n + b.bf0[s2] + j] = v;
    out[(size_t)(b.bf0[s2] + j) * n + b.bf0[s1] + i] = v;
  }
}

// Weights of the derivative of block (s1, s2) in cartesians: wa of the
// derivative by the first centre (2 W[s1][s2]), wb by the second (2 W[s2][s1],
// transposed); s1 == s2 is one ordered pair and has the first only.  W of
// whole-wave blocks, one barrier.  diff: the two derivatives are each other's
// negatives and belong to one atom (S and T of shells on one centre), so their
// weights go into wa as one difference (half of it where the pair is one) and
// wb is zero: exactly nothing for a symmetric W, however large 2a makes the
// terms.  Returns whether a weight of this lane is not zero.
template <int LA, int LB>
__device__ bool ob_weights(const OneBodyView& b, const double* __restrict__ W, int s1, int s2, bool diff, double* wa,
                           double* wb) {
  constexpr int NA = ncart(LA), NB = ncart(LB);
  const int n1 = ob_nfun(b, LA), n2 = ob_nfun(b, LB), f1 = b.bf0[s1], f2 = b.bf0[s2];
  const size_t n = (size_t)b.nbf;
  bool any = false;
  __syncthreads();  // the last pair's weights have been read
  for (int k = (int)threadIdx.x; k < NA * NB; k += 64) {
    const int c = k / NB, e = k % NB;
    double va = 0.0, vb = 0.0;
    for (int i = 0; i < n1; ++i) {
      const double f = ob_coef(b, LA, i, c);
      if (f == 0.0) continue;
      for (int j = 0; j < n2; ++j) {
        const double g = 2.0 * f * ob_coef(b, LB, j, e);
        if (g == 0.0) continue;
        va = fma(g, W[(size_t)(f1 + i) * n + f2 + j], va);
        vb = fma(g, W[(size_t)(f2 + j) * n + f1 + i], vb);
      }
    }
    if (diff) va = (s1 == s2 ? 0.5 : 1.0) * (va - vb);
    wa[k] = va;
    wb[k] = diff || s1 == s2 ? 0.0 : vb;
    any = any || va != 0.0 || (!diff && vb != 0.0);
  }
  __syncthreads();
  return any;
}

// whether two shells sit on one atom, at one place
__device__ bool ob_same(const OneBodyView& b, int s1, int s2) {
  const double* A = b.cen + 3 * s1;
  const double* B = b.cen + 3 * s2;
  return b.atom[s1] == b.atom[s2] && A[0] == B[0] && A[1] == B[1] && A[2] == B[2];
}

// S and T derivatives, one wave per block over the pairs of its stride; S and
// T depend on A - B only, so the second centre's derivative is minus the
// first's, and a pair on one centre contributes what W is not symmetric by
template <int LA, int LB, int op>
__global__ __launch_bounds__(64) void k_one_body_grad_st(OneBodyView b, long long npair,
                                                         const double* __restrict__ W, double* __restrict__ grad,
                                                         int ncopy) {
  constexpr int NA = ncart(LA), NB = ncart(LB);
  __shared__ ObPrim list[64];
  __shared__ double wa[NA * NB], wb[NA * NB];
  const int lane = (int)threadIdx.x;
  grad += (size_t)(blockIdx.x & (unsigned)(ncopy - 1)) * 3 * b.natoms;
  for (long long t = blockIdx.x; t < npair; t += gridDim.x) {
    int s1, s2;
    ob_pair<LA, LB>(b, t, s1, s2);
    const bool one = ob_same(b, s1, s2);
    const int np = (b.po[s1 + 1] - b.po[s1]) * (b.po[s2 + 1] - b.po[s2]);
    bool have = false;
    double ga[3] = {0.0, 0.0, 0.0}, gb[3] = {0.0, 0.0, 0.0};
    for (int i0 = 0; i0 < np; i0 += 64) {
      const int n = ob_prims<LA, LB, op, true>(b, s1, s2, i0, np, list);
      if (n == 0) continue;  // the same for the whole wave
      if (!have && !__any(ob_weights<LA, LB>(b, W, s1, s2, one, wa, wb)) && one) break;
      have = true;
      if (lane >= n) continue;
      const ObPrim q = list[lane];
      const double o2p = 0.5 / q.p, s00 = pow(kPi1 / q.p, 1.5) * q.K;
      double S[3][LA + 2][LB + 3];
      sfor<3>([&](auto d) {
        ob_os1d<LA + 1, LB + 2>(q.PA[d], q.a / q.p * (b.cen[3 * s1 + d] - b.cen[3 * s2 + d]), o2p, S[d]);
      });
      sfor<NA * NB>([&](auto k) {
        constexpr int ca = k / NB, cb = k % NB;
        constexpr int ae[3] = {cart_x(LA, ca), cart_y(LA, ca), cart_z(LA, ca)};
        constexpr int be[3] = {cart_x(LB, cb), cart_y(LB, cb), cart_z(LB, cb)};
        double s[3], ds[3], tt[3], dt[3];
        sfor<3>([&](auto d) {
          s[d] = S[d][ae[d]][be[d]];
          ds[d] = 2.0 * q.a * S[d][ae[d] + 1][be[d]];
          if constexpr (ae[d] > 0) ds[d] -= ae[d] * S[d][ae[d] - 1][be[d]];
          if constexpr (op == 1) {
            tt[d] = ob_t1<ae[d], be[d]>(S[d], q.b);
            dt[d] = 2.0 * q.a * ob_t1<ae[d] + 1, be[d]>(S[d], q.b);
            if constexpr (ae[d] > 0) dt[d] -= ae[d] * ob_t1<ae[d] - 1, be[d]>(S[d], q.b);
          }
        });
        const double va = s00 * wa[k], vb = s00 * wb[k];
        sfor<3>([&](auto x) {
          constexpr int y = (x + 1) % 3, z = (x + 2) % 3;
          double v;
          if constexpr (op == 0)
            v = ds[x] * s[y] * s[z];
          else
            v = dt[x] * s[y] * s[z] + ds[x] * (tt[y] * s[z] + s[y] * tt[z]);
          ga[x] = fma(va, v, ga[x]);
          gb[x] = fma(-vb, v, gb[x]);
        });
        ob_fence<LA, LB>();
      });
    }
    if (!have) continue;
    sfor<3>([&](auto x) {
      ga[x] = ob_wave_sum(ga[x]);
      gb[x] = ob_wave_sum(gb[x]);
    });
    if (lane < 6) {
      const int x = lane % 3;
      const double v = lane < 3 ? (x == 0 ? ga[0] : (x == 1 ? ga[1] : ga[2])) : (x == 0 ? gb[0] : (x == 1 ? gb[1] : gb[2]));
      if (v != 0.0) unsafeAtomicAdd(&grad[3 * b.atom[lane < 3 ? s1 : s2] + x], v);
    }
  }
}

// V derivative: a wave walks the pairs of its stride for up to 64 nuclei
// (blockIdx.y), lane (primitive pair, nucleus) with the nucleus fixed, so the
// nuclei's own forces stay in registers until the wave ends; by translation
// invariance a nucleus takes minus the derivatives of both centres.
template <int LA, int LB>
__global__ __launch_bounds__(64) void k_one_body_grad_v(OneBodyView b, RysArgs ra, long long npair,
                                                        const double* __restrict__ W, double* __restrict__ grad,
                                                        int ncopy) {
  constexpr int NA = ncart(LA), NB = ncart(LB), L1 = LA + LB + 1, NR = L1 / 2 + 1;
  __shared__ ObPrim list[64];
  __shared__ double wa[NA * NB], wb[NA * NB];
  const int lane = (int)threadIdx.x;
  grad += (size_t)(blockIdx.x & (unsigned)(ncopy - 1)) * 3 * b.natoms;
  const int c0 = (int)blockIdx.y * 64, nn = b.natoms - c0 < 64 ? b.natoms - c0 : 64;  // nuclei of this wave
  const int npar = 64 / nn;                                                           // primitive pairs at a time
  const bool on = lane < npar * nn;
  const int cn = c0 + lane % nn, sub = lane / nn;
  double R[3], gc[3] = {0.0, 0.0, 0.0};
  for (int d = 0; d < 3; ++d) R[d] = b.R[3 * cn + d];
  const double Zf = -b.Z[cn] * 2.0 * kPi1;
  for (long long t = blockIdx.x; t < npair; t += gridDim.x) {
    int s1, s2;
    ob_pair<LA, LB>(b, t, s1, s2);
    const int np = (b.po[s1 + 1] - b.po[s1]) * (b.po[s2 + 1] - b.po[s2]);
    // both shells on this lane's nucleus: the three derivatives cancel
    const bool mine = on && !(cn == b.atom[s1] && ob_same(b, s1, s2) && b.cen[3 * s1] == R[0] &&
                              b.cen[3 * s1 + 1] == R[1] && b.cen[3 * s1 + 2] == R[2]);
    bool have = false;
    double ga[3] = {0.0, 0.0, 0.0}, gb[3] = {0.0, 0.0, 0.0};
    for (int i0 = 0; i0 < np; i0 += 64) {
      const int n = ob_prims<LA, LB, 2, true>(b, s1, s2, i0, np, list);
      if (n == 0) continue;  // the same for the whole wave
      if (!have) ob_weights<LA, LB>(b, W, s1, s2, false, wa, wb);
      have = true;
      for (int i = sub; mine && i < n; i += npar) {
        const ObPrim& q = list[i];
        const double p = q.p;
        double PA[3], PC[3], PC2 = 0.0;
        sfor<3>([&](auto d) {
          PA[d] = q.PA[d];
          PC[d] = PA[d] + (b.cen[3 * s1 + d] - R[d]);
          PC2 += PC[d] * PC[d];
        });
        double u[NR], w[NR];
        rys_roots<NR>(p * PC2, ra, u, w);
        const double pref = Zf / p * q.K, h2p = 0.5 / p, ta = 2.0 * q.a, tb = 2.0 * q.b;
        sfor<NR>([&](auto r) {
          double I[3][LA + 2][LB + 2];
          sfor<3>([&](auto d) {
            ob_1d<L1, LA + 1, LB + 1>(d == 2 ? w[r] * pref : 1.0, PA[d] - u[r] * PC[d], (1.0 - u[r]) * h2p,
                                      b.cen[3 * s1 + d] - b.cen[3 * s2 + d], I[d]);
          });
          sfor<NA * NB>([&](auto k) {
            constexpr int ca = k / NB, cb = k % NB;
            constexpr int ae[3] = {cart_x(LA, ca), cart_y(LA, ca), cart_z(LA, ca)};
            constexpr int be[3] = {cart_x(LB, cb), cart_y(LB, cb), cart_z(LB, cb)};
            double v[3];
            sfor<3>([&](auto d) { v[d] = I[d][ae[d]][be[d]]; });
            const double va = wa[k], vb = wb[k];
            sfor<3>([&](auto x) {
              const double o = v[(x + 1) % 3] * v[(x + 2) % 3];
              double dA = ta * I[x][ae[x] + 1][be[x]], dB = tb * I[x][ae[x]][be[x] + 1];
              if constexpr (ae[x] > 0) dA -= ae[x] * I[x][ae[x] - 1][be[x]];
              if constexpr (be[x] > 0) dB -= be[x] * I[x][ae[x]][be[x] - 1];
              ga[x] = fma(va * o, dA, ga[x]);
              gb[x] = fma(vb * o, dB, gb[x]);
            });
            ob_fence<LA, LB>();
          });
        });
      }
    }
    if (!have) continue;
    sfor<3>([&](auto x) {
      gc[x] -= ga[x] + gb[x];
      ga[x] = ob_wave_sum(ga[x]);
      gb[x] = ob_wave_sum(gb[x]);
    });
    if (lane < 6) {
      const int x = lane % 3;
      const double v = lane < 3 ? (x == 0 ? ga[0] : (x == 1 ? ga[1] : ga[2])) : (x == 0 ? gb[0] : (x == 1 ? gb[1] : gb[2]));
      if (v != 0.0) unsafeAtomicAdd(&grad[3 * b.atom[lane < 3 ? s1 : s2] + x], v);
    }
  }
  if (on)
    sfor<3>([&](auto x) {
      if (gc[x] != 0.0) unsafeAtomicAdd(&grad[3 * cn + x], gc[x]);
    });
}

namespace {

// f(LA, LB) for every class with LA >= LB up to f
template <typename F>
void ob_classes(F&& f) {
  f(std::integral_constant<int, 0>{}, std::integral_constant<int, 0>{});
  f(std::integral_constant<int, 1>{}, std::integral_constant<int, 0>{});
  f(std::integral_constant<int, 1>{}, std::integral_constant<int, 1>{});
  f(std::integral_constant<int, 2>{}, std::integral_constant<int, 0>{});
  f(std::integral_constant<int, 2>{}, std::integral_constant<int, 1>{});
  f(std::integral_constant<int, 2>{}, std::integral_constant<int, 2>{});
  f(std::integral_constant<int, 3>{}, std::integral_constant<int, 0>{});
  f(std::integral_constant<int, 3>{}, std::integral_constant<int, 1>{});
  f(std::integral_constant<int, 3>{}, std::integral_constant<int, 2>{});
  f(std::integral_constant<int, 3>{}, std::integral_constant<int, 3>{});
}

// waves of a gradient launch: enough to fill the GPU several times over, few
// enough that their final atomics stay a small part
constexpr long long kObWaves = 4096;
// blocks of a matrix launch in x; the rest of a class's pairs go to y, as a
// dimension of 2^32 threads (2^26 pairs: 11586 s shells) is not run whole
constexpr long long kObGridX = 1ll << 20;

}  // namespace

void launch_one_body(const OneBodyView& b, const RysArgs& ra, int op, double* out, hipStream_t s) {
  ob_classes([&](auto la, auto lb) {
    const long long n = ob_npairs<la, lb>(b);
    if (n <= 0) return;
    const long long gx = std::min(n, kObGridX);
    const dim3 grid((unsigned)gx, (unsigned)((n + gx - 1) / gx)), block(64);
    if (op == 0)
      hipLaunchKernelGGL((k_one_body<la, lb, 0>), grid, block, 0, s, b, ra, n, out);
    else if (op == 1)
      hipLaunchKernelGGL((k_one_body<la, lb, 1>), grid, block, 0, s, b, ra, n, out);
    else
      hipLaunchKernelGGL((k_one_body<la, lb, 2>), grid, block, 0, s, b, ra, n, out);
  });
}

void launch_one_body_grad(const OneBodyView& b, const RysArgs& ra, int op, const double* W, double* grad, int ncopy,
                          hipStream_t s) {
  ob_classes([&](auto la, auto lb) {
    const long long n = ob_npairs<la, lb>(b);
    if (n <= 0) return;
    const dim3 grid((unsigned)std::min(n, kObWaves));
    if (op == 0) {
      hipLaunchKernelGGL((k_one_body_grad_st<la, lb, 0>), grid, dim3(64), 0, s, b, n, W, grad, ncopy);
    } else if (op == 1) {
      hipLaunchKernelGGL((k_one_body_grad_st<la, lb, 1>), grid, dim3(64), 0, s, b, n, W, grad, ncopy);
    } else if (b.natoms > 0) {
      hipLaunchKernelGGL((k_one_body_grad_v<la, lb>),
                         dim3((unsigned)std::min(n, kObWaves), (unsigned)((b.natoms + 63) / 64)), dim3(64), 0, s, b, ra,
                         n, W, grad, ncopy);
    }
  });
}

}  // namespace qfe
