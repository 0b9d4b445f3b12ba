// Density-fitted Coulomb (DF-J) on the GPU: the three-centre integrals
// B[P][mu nu] = (mu nu|P) over an auxiliary basis, mu >= nu only (the packed
// lower triangle: half the HBM and half the bytes a build reads, against the
// full square of the reference's INCORE DF engine,
// scf/src/eri/INCORE/incore_impl_df.cpp:53-80), and the two-centre metric
// V[P][Q] = (P|Q), kept in HBM.  The
// build itself is X = B . vec(D), V c = X, J = B^T c (incore_impl_df.cpp:
// 81-200); the last product, a plain GEMV that rocBLAS streams at 5.7 TB/s,
// runs in engine.cpp.
//
// The integrals are Rys quadrature with runtime angular momenta (orbital
// shells up to d, auxiliary shells up to g): per primitive triple and root,
// 2-D recursions I(i, k) for i <= la + lb on the bra and k <= lc on the
// auxiliary centre, the transfer to (a, b), and the solid-harmonic
// transforms.  An auxiliary function is a ket pair (c, s0) with s0 an s
// function of exponent 0 at the same centre, so q = gamma, Q = C and the
// ket transfer term vanishes.  The work is far below the Fock build's; the
// kernels are plain code (one thread per block).
#include <hip/hip_runtime.h>

#include "dfj.hpp"
#include "eri_core.hpp"

namespace qfe {

namespace {

constexpr double kTwoPi52 = 34.98683665524972;  // 2 pi^(5/2)
constexpr int kMaxLo = 2;                        // orbital shells up to d
constexpr int kMaxLx = 4;                        // auxiliary shells up to g
constexpr int kMaxAB = 2 * kMaxLo;               // bra recursion extent (also an auxiliary shell with s0)
constexpr int kNCo = (kMaxLo + 1) * (kMaxLo + 2) / 2;
constexpr int kNCx = (kMaxLx + 1) * (kMaxLx + 2) / 2;

struct ShellRef {
  int l, n;          // angular momentum, primitives
  const double* e;   // exponents
  const double* c;   // contraction coefficients (normalised)
  const double* O;   // centre
};

__device__ int df_ncart(int l) { return (l + 1) * (l + 2) / 2; }

__device__ void df_cart_xyz(int l, int c, int& x, int& y, int& z) {
  int k = 0;
  while ((k + 1) * (k + 2) / 2 <= c) ++k;
  x = l - k;
  z = c - k * (k + 1) / 2;
  y = l - x - z;
}

__device__ void df_rys(int n, double T, const RysArgs& ra, double* u, double* w) {
  switch (n) {
#define QFE_DF_ROOTS(N)                 \
  case N: {                             \
    double uu[N], ww[N];                \
    rys_roots<N>(T, ra, uu, ww);        \
    for (int i = 0; i < N; ++i) {       \
      u[i] = uu[i];                     \
      w[i] = ww[i];                     \
    }                                   \
    break;                              \
  }
    QFE_DF_ROOTS(1)
    QFE_DF_ROOTS(2)
    QFE_DF_ROOTS(3)
    QFE_DF_ROOTS(4)
    QFE_DF_ROOTS(5)
    default:
      QFE_DF_ROOTS(6)
#undef QFE_DF_ROOTS
  }
}

// cartesian block (a b | c): out[na][nb][nc]
__device__ void df_cart(const ShellRef& a, const ShellRef& b, const ShellRef& c, const RysArgs& ra,
                        double* out) {
  const int la = a.l, lb = b.l, lc = c.l, lab = la + lb;
  const int na = df_ncart(la), nb = df_ncart(lb), nc = df_ncart(lc);
  for (int i = 0; i < na * nb * nc; ++i) out[i] = 0.0;
  double AB[3], AB2 = 0.0;
  for (int d = 0; d < 3; ++d) {
    AB[d] = a.O[d] - b.O[d];
    AB2 += AB[d] * AB[d];
  }
  const int nroots = (lab + lc) / 2 + 1;
  for (int ia = 0; ia < a.n; ++ia)
    for (int ib = 0; ib < b.n; ++ib) {
      const double p = a.e[ia] + b.e[ib];
      const double Kab = a.c[ia] * b.c[ib] * exp(-a.e[ia] * b.e[ib] / p * AB2) / p;
      if (Kab == 0.0) continue;
      double P[3], PA[3];
      for (int d = 0; d < 3; ++d) {
        P[d] = (a.e[ia] * a.O[d] + b.e[ib] * b.O[d]) / p;
        PA[d] = P[d] - a.O[d];
      }
      for (int ic = 0; ic < c.n; ++ic) {
        const double q = c.e[ic];
        const double Kc = c.c[ic] / q;
        double PQ[3], PQ2 = 0.0;
        for (int d = 0; d < 3; ++d) {
          PQ[d] = P[d] - c.O[d];
          PQ2 += PQ[d] * PQ[d];
        }
        const double rpq = 1.0 / (p + q);
        const double T = p * q * rpq * PQ2;
        const double pref = kTwoPi52 * Kab * Kc * sqrt(rpq);
        double u[6], w[6];
        df_rys(nroots, T, ra, u, w);
        const double h2p = 0.5 / p, h2q = 0.5 / q, qr = q * rpq, pr = p * rpq;
        for (int r = 0; r < nroots; ++r) {
          const double ur = u[r];
          const double B00 = 0.5 * rpq * ur, B10 = h2p - h2p * qr * ur, B01 = h2q - h2q * pr * ur;
          double I[3][kMaxAB + 1][kMaxLo + 1][kMaxLx + 1];  // first bra index up to la <= lab
          for (int d = 0; d < 3; ++d) {
            const double C00 = PA[d] - qr * ur * PQ[d], D00 = pr * ur * PQ[d];
            double G[kMaxAB + 1][kMaxLx + 1];
            G[0][0] = (d == 2) ? w[r] * pref : 1.0;
            for (int i = 0; i < lab; ++i) G[i + 1][0] = C00 * G[i][0] + (i > 0 ? i * B10 * G[i - 1][0] : 0.0);
            for (int k = 0; k < lc; ++k)
              for (int i = 0; i <= lab; ++i) {
                double v = D00 * G[i][k];
                if (k > 0) v += k * B01 * G[i][k - 1];
                if (i > 0) v += i * B00 * G[i - 1][k];
                G[i][k + 1] = v;
              }
            // transfer to the second bra centre: (a, b+1) = (a+1, b) + AB (a, b)
            for (int k = 0; k <= lc; ++k) {
              double t[kMaxAB + 1][kMaxLo + 1];
              for (int i = 0; i <= lab; ++i) t[i][0] = G[i][k];
              for (int j = 1; j <= lb; ++j)
                for (int i = 0; i <= lab - j; ++i) t[i][j] = t[i + 1][j - 1] + AB[d] * t[i][j - 1];
              for (int i = 0; i <= la; ++i)
                for (int j = 0; j <= lb; ++j) I[d][i][j][k] = t[i][j];
            }
          }
          for (int x = 0; x < na; ++x) {
            int ax, ay, az;
            df_cart_xyz(la, x, ax, ay, az);
            for (int y = 0; y < nb; ++y) {
              int bx, by, bz;
              df_cart_xyz(lb, y, bx, by, bz);
              for (int z = 0; z < nc; ++z) {
                int cx, cy, cz;
                df_cart_xyz(lc, z, cx, cy, cz);
                out[(x * nb + y) * nc + z] += I[0][ax][bx][cx] * I[1][ay][by][cy] * I[2][az][bz][cz];
              }
            }
          }
        }
      }
    }
}

// output functions of a shell: solid harmonics from d on when pure
__device__ int df_nfun(int l, int pure) { return (pure && l >= 2) ? 2 * l + 1 : df_ncart(l); }

// block [na][nb][nc] cartesian -> [ma][mb][mc] output functions
__device__ void df_to_out(const double* sph, int la, int lb, int lc, int pure_o, int pure_x, const double* in,
                          double* out) {
  const int na = df_ncart(la), nb = df_ncart(lb), nc = df_ncart(lc);
  const int ma = df_nfun(la, pure_o), mb = df_nfun(lb, pure_o), mc = df_nfun(lc, pure_x);
  const bool pa = pure_o && la >= 2, pb = pure_o && lb >= 2, pc = pure_x && lc >= 2;
  double t1[kNCo * kNCo * kNCx];
  // c index
  for (int x = 0; x < na * nb; ++x)
    for (int m = 0; m < mc; ++m) {
      double s = 0.0;
      if (pc)
        for (int z = 0; z < nc; ++z) s += sph[(lc * 9 + m) * 15 + z] * in[x * nc + z];
      else
        s = in[x * nc + m];
      t1[x * mc + m] = s;
    }
  // b index: t1[na][nb][mc] -> t2[na][mb][mc]
  double t2[kNCo * kNCo * kNCx];
  for (int x = 0; x < na; ++x)
    for (int m = 0; m < mb; ++m)
      for (int z = 0; z < mc; ++z) {
        double s = 0.0;
        if (pb)
          for (int y = 0; y < nb; ++y) s += sph[(lb * 9 + m) * 15 + y] * t1[(x * nb + y) * mc + z];
        else
          s = t1[(x * nb + m) * mc + z];
        t2[(x * mb + m) * mc + z] = s;
      }
  // a index
  for (int m = 0; m < ma; ++m)
    for (int y = 0; y < mb; ++y)
      for (int z = 0; z < mc; ++z) {
        double s = 0.0;
        if (pa)
          for (int x = 0; x < na; ++x) s += sph[(la * 9 + m) * 15 + x] * t2[(x * mb + y) * mc + z];
        else
          s = t2[(m * mb + y) * mc + z];
        out[(m * mb + y) * mc + z] = s;
      }
}

__device__ ShellRef df_shell(const DFBasisView& v, int s) {
  return ShellRef{v.l[s], v.po[s + 1] - v.po[s], v.exps + v.po[s], v.coefs + v.po[s], v.cen + 3 * s};
}

}  // namespace

// B[P][mu >= nu] (packed lower triangle, element mu (mu + 1) / 2 + nu) for one
// (orbital shell pair s1 >= s2, auxiliary shell) per thread
__global__ __launch_bounds__(256) void k_df_three_centre(DFBasisView o, DFBasisView x, RysArgs ra,
                                                         const double* __restrict__ sph, double* __restrict__ B) {
  const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  const long long npair = (long long)o.nsh * (o.nsh + 1) / 2;
  if (t >= npair * x.nsh) return;
  const int sc = (int)(t / npair);
  const long long pq = t % npair;
  int s1 = (int)((sqrt(8.0 * (double)pq + 1.0) - 1.0) / 2.0);
  while ((long long)s1 * (s1 + 1) / 2 > pq) --s1;
  while ((long long)(s1 + 1) * (s1 + 2) / 2 <= pq) ++s1;
  const int s2 = (int)(pq - (long long)s1 * (s1 + 1) / 2);
  const ShellRef a = df_shell(o, s1), b = df_shell(o, s2), c = df_shell(x, sc);
  double cart[kNCo * kNCo * kNCx], blk[kNCo * kNCo * kNCx];
  df_cart(a, b, c, ra, cart);
  df_to_out(sph, a.l, b.l, c.l, o.pure, x.pure, cart, blk);
  const int ma = df_nfun(a.l, o.pure), mb = df_nfun(b.l, o.pure), mc = df_nfun(c.l, x.pure);
  const size_t n = (size_t)o.nbf, np = n * (n + 1) / 2;
  for (int i = 0; i < ma; ++i)
    for (int j = 0; j < mb; ++j) {
      const size_t mu = (size_t)o.bf0[s1] + i, nu = (size_t)o.bf0[s2] + j;
      const size_t hi = mu > nu ? mu : nu, lo = mu > nu ? nu : mu;
      const size_t e = hi * (hi + 1) / 2 + lo;
      for (int k = 0; k < mc; ++k) B[(size_t)(x.bf0[sc] + k) * np + e] = blk[(i * mb + j) * mc + k];
    }
}

// V[P][Q] for one auxiliary shell pair c1 >= c2 per thread: (c1 s0 | c2)
__global__ __launch_bounds__(256) void k_df_metric(DFBasisView x, RysArgs ra, const double* __restrict__ sph,
                                                   double* __restrict__ V) {
  const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  const long long npair = (long long)x.nsh * (x.nsh + 1) / 2;
  if (t >= npair) return;
  int c1 = (int)((sqrt(8.0 * (double)t + 1.0) - 1.0) / 2.0);
  while ((long long)c1 * (c1 + 1) / 2 > t) --c1;
  while ((long long)(c1 + 1) * (c1 + 2) / 2 <= t) ++c1;
  const int c2 = (int)(t - (long long)c1 * (c1 + 1) / 2);
  const double zero = 0.0, one = 1.0;
  const ShellRef a = df_shell(x, c1), c = df_shell(x, c2);
  const ShellRef s0{0, 1, &zero, &one, c.O};
  // the bra holds an auxiliary shell (up to g): use the auxiliary limits for it
  double cart[kNCx * kNCx], blk[kNCx * kNCx];
  df_cart(c, s0, a, ra, cart);  // (c2 s0 | c1): c2 on the bra, c1 on the auxiliary side
  df_to_out(sph, c.l, 0, a.l, x.pure, x.pure, cart, blk);
  const int m2 = df_nfun(c.l, x.pure), m1 = df_nfun(a.l, x.pure);
  const size_t n = (size_t)x.nbf;
  for (int j = 0; j < m2; ++j)
    for (int i = 0; i < m1; ++i) {
      const double v = blk[j * m1 + i];
      V[(size_t)(x.bf0[c1] + i) * n + x.bf0[c2] + j] = v;
      V[(size_t)(x.bf0[c2] + j) * n + x.bf0[c1] + i] = v;
    }
}

// d[mu (mu + 1) / 2 + nu] = D[mu][nu] + D[nu][mu] (mu > nu), D[mu][mu] on the
// diagonal: the density in the packed layout of B (one thread per element)
__global__ __launch_bounds__(256) void k_df_pack(const double* __restrict__ D, double* __restrict__ d, int n) {
  const long long e = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= (long long)n * (n + 1) / 2) return;
  long long mu = (long long)((sqrt(8.0 * (double)e + 1.0) - 1.0) / 2.0);
  while (mu * (mu + 1) / 2 > e) --mu;
  while ((mu + 1) * (mu + 2) / 2 <= e) ++mu;
  const long long nu = e - mu * (mu + 1) / 2;
  d[e] = mu == nu ? D[mu * n + mu] : D[mu * n + nu] + D[nu * n + mu];
}

// J[mu][nu] = J[nu][mu] = j[mu (mu + 1) / 2 + nu]: one thread per element of
// the full matrix, so the stores are coalesced
__global__ __launch_bounds__(256) void k_df_unpack(const double* __restrict__ j, double* __restrict__ J, int n) {
  const long long e = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= (long long)n * n) return;
  const long long r = e / n, c = e % n;
  const long long hi = r > c ? r : c, lo = r > c ? c : r;
  J[e] = j[hi * (hi + 1) / 2 + lo];
}

// x = B d reads B once and is bound by HBM.  A block takes kDfRows rows x
// kDfChunk elements, so that d is read from L2 once for kDfRows rows: 0.87 ms
// (6.1 TB/s) at (H2O)32/def2-SVP, where rocBLAS's transposed GEMV took 1.55 ms.
// Rows start at any multiple of 8 bytes (np may be odd), so the loads are
// single doubles.
constexpr int kDfRows = 16;
__global__ __launch_bounds__(256) void k_df_dots(const double* __restrict__ B, const double* __restrict__ d,
                                                 size_t np, int naux, int nchunk, double* __restrict__ part) {
  constexpr int N = kDfChunk / 256;
  __shared__ double sm[4][kDfRows];
  const int tid = (int)threadIdx.x, lane = tid & 63;
  const size_t c0 = (size_t)blockIdx.x * kDfChunk + tid;
  const int r0 = (int)blockIdx.y * kDfRows, nr = naux - r0 < kDfRows ? naux - r0 : kDfRows;
  double dv[N];
#pragma unroll
  for (int k = 0; k < N; ++k) dv[k] = c0 + 256 * k < np ? d[c0 + 256 * k] : 0.0;
  for (int r = 0; r < nr; ++r) {
    const double* row = B + (size_t)(r0 + r) * np;
    double bv[N];
#pragma unroll
    for (int k = 0; k < N; ++k) bv[k] = c0 + 256 * k < np ? row[c0 + 256 * k] : 0.0;
    double s = 0.0;
#pragma unroll
    for (int k = 0; k < N; ++k) s = fma(bv[k], dv[k], s);
    for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o);
    if (lane == 0) sm[tid >> 6][r] = s;
  }
  __syncthreads();
  if (tid < nr) part[(size_t)(r0 + tid) * nchunk + blockIdx.x] = sm[0][tid] + sm[1][tid] + sm[2][tid] + sm[3][tid];
}

// x[P] = sum of its chunks, one wave per P
__global__ __launch_bounds__(256) void k_df_sum(const double* __restrict__ part, int naux, int nchunk,
                                                double* __restrict__ x) {
  const int p = (int)((blockIdx.x * blockDim.x + threadIdx.x) >> 6), lane = (int)(threadIdx.x & 63);
  if (p >= naux) return;
  double s = 0.0;
  for (int k = lane; k < nchunk; k += 64) s += part[(size_t)p * nchunk + k];
  for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o);
  if (lane == 0) x[p] = s;
}

// Triangular solves by blocks of kDfBlock rows: rocSOLVER's potrs spent 0.86 ms
// in two substitutions of 2272 rows, one dependent step after another.  Here a
// launch per block solves its unknowns with the inverse of the diagonal block
// and applies them to all the rows that remain.  The product with the inverse
// alone would be a digit short of substitution (residual 2e-15 of |b| instead
// of 1.4e-16 at a metric of condition 6e10), so it is corrected once by the
// block's own residual, which brings it to 1.3e-16.  36 launches of 10-12 us:
// 0.41 ms.
__global__ __launch_bounds__(kDfBlock) void k_df_inverses(const double* __restrict__ L, int n,
                                                          double* __restrict__ dinv) {
  // thread j: column j of the inverse of block blockIdx.x, by substitution
  const int b0 = (int)blockIdx.x * kDfBlock, nb = n - b0 < kDfBlock ? n - b0 : kDfBlock, j = (int)threadIdx.x;
  double* D = dinv + (size_t)b0 * kDfBlock;
  if (j >= nb) {
    for (int i = 0; i < nb; ++i) D[(size_t)i * kDfBlock + j] = 0.0;
    return;
  }
  for (int i = 0; i < j; ++i) D[(size_t)i * kDfBlock + j] = 0.0;
  for (int i = j; i < nb; ++i) {
    double s = i == j ? 1.0 : 0.0;
    for (int m = j; m < i; ++m) s = fma(-L[(size_t)(b0 + m) * n + b0 + i], D[(size_t)m * kDfBlock + j], s);
    D[(size_t)i * kDfBlock + j] = s / L[(size_t)(b0 + i) * n + b0 + i];
  }
}

// What a step reads does not depend on the unknowns before it, so every load is
// issued before the first product: a step costs one memory latency.
constexpr int kDfThreads = 4 * kDfBlock, kDfPer = kDfBlock / 4;

// zb = the unknowns of block b0 for the right-hand side r: with the block
// itself (FWD) or its transpose.  rows: sixteen lanes a row, along contiguous
// k, four rows a lane; cols: one lane a row and quarter of k, partial sums
// through LDS.
template <bool FWD>
__device__ __forceinline__ void df_block(const double* __restrict__ L, const double* __restrict__ dinv, int n, int b0,
                                         int nb, const double* __restrict__ r, double* rb, double* zb, double* res,
                                         double (*part)[kDfBlock]) {
  constexpr int NK = kDfBlock / 16, RS = kDfThreads / 16, NR = kDfBlock / RS;
  const int tid = (int)threadIdx.x, i = tid >> 4, h = tid & 15, c = tid & (kDfBlock - 1), q = tid / kDfBlock;
  double rows[NR][NK], cols[kDfPer];
#pragma unroll
  for (int p = 0; p < NR; ++p)
#pragma unroll
    for (int m = 0; m < NK; ++m) {
      const int k = h + 16 * m, row = i + RS * p;
      if constexpr (FWD)
        rows[p][m] = k <= row && row < nb ? dinv[(size_t)(b0 + row) * kDfBlock + k] : 0.0;
      else
        rows[p][m] = k >= row && k < nb ? L[(size_t)(b0 + row) * n + b0 + k] : 0.0;
    }
#pragma unroll
  for (int m = 0; m < kDfPer; ++m) {
    const int k = q * kDfPer + m;
    if constexpr (FWD)
      cols[m] = k <= c && c < nb ? L[(size_t)(b0 + k) * n + b0 + c] : 0.0;
    else
      cols[m] = k >= c && k < nb ? dinv[(size_t)(b0 + k) * kDfBlock + c] : 0.0;
  }
  if (tid < kDfBlock) rb[tid] = tid < nb ? r[b0 + tid] : 0.0;
  __syncthreads();
  auto by_rows = [&](const double* v, double* out) {  // valid in the first lane of a row
#pragma unroll
    for (int p = 0; p < NR; ++p) out[p] = 0.0;
#pragma unroll
    for (int m = 0; m < NK; ++m) {
      const double vk = v[h + 16 * m];
#pragma unroll
      for (int p = 0; p < NR; ++p) out[p] = fma(rows[p][m], vk, out[p]);
    }
#pragma unroll
    for (int p = 0; p < NR; ++p)
      for (int o = 8; o > 0; o >>= 1) out[p] += __shfl_xor(out[p], o);
  };
  auto by_cols = [&](const double* v) {  // valid in the first kDfBlock threads
    double s = 0.0;
#pragma unroll
    for (int m = 0; m < kDfPer; ++m) s = fma(cols[m], v[q * kDfPer + m], s);
    part[q][c] = s;
    __syncthreads();
    return (part[0][c] + part[1][c]) + (part[2][c] + part[3][c]);
  };
  if constexpr (FWD) {
    double z[NR], dz[NR];
    by_rows(rb, z);
#pragma unroll
    for (int p = 0; p < NR; ++p)
      if (h == 0) zb[i + RS * p] = z[p];
    __syncthreads();
    const double t = by_cols(zb);
    if (q == 0) res[c] = rb[c] - t;
    __syncthreads();
    by_rows(res, dz);
#pragma unroll
    for (int p = 0; p < NR; ++p)
      if (h == 0) zb[i + RS * p] = z[p] + dz[p];
  } else {
    const double z = by_cols(rb);
    if (q == 0) zb[c] = z;
    __syncthreads();
    double t[NR];
    by_rows(zb, t);
#pragma unroll
    for (int p = 0; p < NR; ++p)
      if (h == 0) res[i + RS * p] = rb[i + RS * p] - t[p];
    __syncthreads();
    const double dz = by_cols(res);
    if (q == 0) zb[c] = z + dz;
  }
  __syncthreads();
}

// forward step: y of block b0 (every thread block forms it, the first stores
// it), then x -= L y for the rows below, kDfBlock rows a thread block
__global__ __launch_bounds__(kDfThreads) void k_df_forward(const double* __restrict__ L,
                                                           const double* __restrict__ dinv, int n, int b0,
                                                           double* __restrict__ x, double* __restrict__ y) {
  __shared__ double rb[kDfBlock], zb[kDfBlock], res[kDfBlock], part[4][kDfBlock];
  const int tid = (int)threadIdx.x, c = tid & (kDfBlock - 1), q = tid / kDfBlock;
  const int nb = n - b0 < kDfBlock ? n - b0 : kDfBlock, i = b0 + nb + (int)blockIdx.x * kDfBlock + c;
  double u[kDfPer];
#pragma unroll
  for (int m = 0; m < kDfPer; ++m) {
    const int k = q * kDfPer + m;
    u[m] = i < n && k < nb ? L[(size_t)(b0 + k) * n + i] : 0.0;
  }
  df_block<true>(L, dinv, n, b0, nb, x, rb, zb, res, part);
  if (blockIdx.x == 0 && tid < nb) y[b0 + tid] = zb[tid];
  double s = 0.0;
#pragma unroll
  for (int m = 0; m < kDfPer; ++m) s = fma(u[m], zb[q * kDfPer + m], s);
  part[q][c] = s;
  __syncthreads();
  if (q == 0 && i < n) x[i] -= (part[0][c] + part[1][c]) + (part[2][c] + part[3][c]);
}

// backward step: x of block b0 from y, then y -= L^T x for the rows above, one
// row a wave at a time (a column of L is contiguous)
__global__ __launch_bounds__(kDfThreads) void k_df_backward(const double* __restrict__ L,
                                                            const double* __restrict__ dinv, int n, int b0,
                                                            double* __restrict__ y, double* __restrict__ x) {
  constexpr int R = kDfBlock * 64 / kDfThreads;  // rows of a wave
  __shared__ double rb[kDfBlock], zb[kDfBlock], res[kDfBlock], part[4][kDfBlock];
  const int tid = (int)threadIdx.x, lane = tid & 63;
  const int nb = n - b0 < kDfBlock ? n - b0 : kDfBlock, i0 = (int)blockIdx.x * kDfBlock + (tid >> 6) * R;
  double u[R][2];
#pragma unroll
  for (int r = 0; r < R; ++r)
#pragma unroll
    for (int w = 0; w < 2; ++w) {
      const int k = lane + 64 * w;
      u[r][w] = i0 + r < b0 && k < nb ? L[(size_t)(i0 + r) * n + b0 + k] : 0.0;
    }
  df_block<false>(L, dinv, n, b0, nb, y, rb, zb, res, part);
  if (blockIdx.x == 0 && tid < nb) x[b0 + tid] = zb[tid];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    double s = fma(u[r][0], zb[lane], u[r][1] * zb[lane + 64]);
    for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o);
    if (lane == 0 && i0 + r < b0) y[i0 + r] -= s;
  }
}

void launch_df_pack(const double* D, double* d, int n, hipStream_t s) {
  const long long m = (long long)n * (n + 1) / 2;
  if (m > 0) hipLaunchKernelGGL(k_df_pack, dim3((unsigned)((m + 255) / 256)), dim3(256), 0, s, D, d, n);
}

void launch_df_dots(const double* B, const double* d, size_t np, int naux, double* part, double* x, hipStream_t s) {
  const int nchunk = (int)df_chunks(np);
  if (nchunk <= 0 || naux <= 0) return;
  hipLaunchKernelGGL(k_df_dots, dim3((unsigned)nchunk, (unsigned)((naux + kDfRows - 1) / kDfRows)), dim3(256), 0, s, B,
                     d, np, naux, nchunk, part);
  hipLaunchKernelGGL(k_df_sum, dim3((unsigned)((naux + 3) / 4)), dim3(256), 0, s, part, naux, nchunk, x);
}

void launch_df_inverses(const double* L, int n, double* dinv, hipStream_t s) {
  if (n > 0)
    hipLaunchKernelGGL(k_df_inverses, dim3((unsigned)((n + kDfBlock - 1) / kDfBlock)), dim3(kDfBlock), 0, s, L, n, dinv);
}

void launch_df_solve(const double* L, const double* dinv, int n, double* x, double* y, hipStream_t s) {
  if (n <= 0) return;
  for (int b0 = 0; b0 < n; b0 += kDfBlock) {
    const int below = n - b0 - kDfBlock;
    hipLaunchKernelGGL(k_df_forward, dim3((unsigned)(below > 0 ? (below + kDfBlock - 1) / kDfBlock : 1)),
                       dim3(kDfThreads), 0, s, L, dinv, n, b0, x, y);
  }
  for (int b0 = (n - 1) / kDfBlock * kDfBlock; b0 >= 0; b0 -= kDfBlock)
    hipLaunchKernelGGL(k_df_backward, dim3((unsigned)(b0 > 0 ? b0 / kDfBlock : 1)), dim3(kDfThreads), 0, s, L, dinv, n,
                       b0, y, x);
}

void launch_df_unpack(const double* j, double* J, int n, hipStream_t s) {
  const long long m = (long long)n * n;
  if (m > 0) hipLaunchKernelGGL(k_df_unpack, dim3((unsigned)((m + 255) / 256)), dim3(256), 0, s, j, J, n);
}

void launch_df_three_centre(const DFBasisView& o, const DFBasisView& x, const RysArgs& ra, const double* sph,
                            double* B, hipStream_t s) {
  const long long n = (long long)o.nsh * (o.nsh + 1) / 2 * x.nsh;
  if (n <= 0) return;
  hipLaunchKernelGGL(k_df_three_centre, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, o, x, ra, sph, B);
}

void launch_df_metric(const DFBasisView& x, const RysArgs& ra, const double* sph, double* V, hipStream_t s) {
  const long long n = (long long)x.nsh * (x.nsh + 1) / 2;
  if (n <= 0) return;
  hipLaunchKernelGGL(k_df_metric, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, x, ra, sph, V);
}

}  // namespace qfe
