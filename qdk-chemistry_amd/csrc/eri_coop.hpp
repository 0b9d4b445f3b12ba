// Shared pieces of the cooperative class kernels: one block per shell quartet.
//
// In a class with high angular momenta one thread cannot hold a quartet's
// block: split into chunks, every chunk kernel repeats the roots, the 2-D
// recursion and the transfers (98 times for (ff|dd)).  Here a block shares
// them: lane (combination, direction) evaluates the 1-D integrals of one
// (primitive quartet, Rys root) combination in one direction, in registers,
// and stores them in LDS; then the block's threads walk the cartesian
// components of the quartet and read three table entries per combination.
#pragma once

#include "eri_class.hpp"

namespace qfe {

// exponents of cartesian component c of a shell of momentum l <= 3 (CCA order)
template <int L>
QFE_DI void coop_xyz(int c, int& x, int& y, int& z) {
  static_assert(L <= 3, "component decoding covers shells up to f");
  int k = 0;
  if constexpr (L >= 1) k = (c >= 1) + (L >= 2 && c >= 3) + (L >= 3 && c >= 6);
  x = L - k;
  z = c - k * (k + 1) / 2;
  y = k - z;
}

// root and weight r of the N-point Rys rule at T
template <int N>
QFE_DI void rys_root_one(double T, const RysArgs& ra, int r, double& u, double& w) {
  if constexpr (N <= 2) {
    double uu[N], ww[N];
    rys_roots<N>(T, ra, uu, ww);
    u = uu[0];
    w = ww[0];
    if constexpr (N == 2) {
      if (r == 1) {
        u = uu[1];
        w = ww[1];
      }
    }
  } else {
    if (T >= ra.tmax[N]) {
      // the limits sit in the kernel arguments: selected with compile-time
      // indices (a runtime one would copy the argument struct to scratch)
      double hx = 0.0, hw = 0.0;
      sfor<N>([&](auto i) {
        if (r == i) {
          hx = ra.hx2[N][i];
          hw = ra.hw[N][i];
        }
      });
      u = hx * frcp(T);
      w = hw * frsq(T);
    } else {
      const int k = (int)T;
      const double x = T - ((double)k + 0.5);
      const double* __restrict__ cu = ra.coef[N] + ((size_t)k * (2 * N) + r) * (RYS_DEG + 1);
      const double* __restrict__ cw = cu + N * (RYS_DEG + 1);
      u = cu[RYS_DEG];
      w = cw[RYS_DEG];
#pragma unroll
      for (int d = RYS_DEG - 1; d >= 0; --d) {
        u = fma(u, x, cu[d]);
        w = fma(w, x, cw[d]);
      }
    }
  }
}


// The 1-D integrals I(a, b, c, d) of one direction and root, a <= AMX, b <=
// BMX, c <= CMX, d <= DMX with a + b <= EA and c + d <= FC, stored at
// out[((a (BMX+1) + b) (CMX+1) + c) (DMX+1) + d].  The 2-D table G stays in
// registers; each (c, d) column is transferred and stored before the next, so
// that (EA+1)(FC+1) + O(EA) values are live, not the whole result.
template <int EA, int FC, int AMX, int BMX, int CMX, int DMX>
QFE_DI void rys_1d_store(double s, double C00, double C00p, double B00, double B10, double B01, double AB, double CD,
                         double* out) {
  double g[EA + 1][FC + 1];
  g[0][0] = s;
  if constexpr (EA >= 1) g[1][0] = C00 * s;
  sfor<(EA >= 2 ? EA - 1 : 0)>([&](auto ii) {
    constexpr int i = ii + 1;
    g[i + 1][0] = C00 * g[i][0] + i * B10 * g[i - 1][0];
  });
  if constexpr (FC >= 1) {
    g[0][1] = C00p * s;
    sfor<EA>([&](auto ii) {
      constexpr int i = ii + 1;
      g[i][1] = C00p * g[i][0] + i * B00 * g[i - 1][0];
    });
    sfor<(FC >= 2 ? FC - 1 : 0)>([&](auto kk) {
      constexpr int k = kk + 1;
      g[0][k + 1] = C00p * g[0][k] + k * B01 * g[0][k - 1];
      sfor<EA>([&](auto ii) {
        constexpr int i = ii + 1;
        g[i][k + 1] = C00p * g[i][k] + k * B01 * g[i][k - 1] + i * B00 * g[i - 1][k];
      });
    });
  }
  // ket transfer in place, one d at a time: g[i][k] becomes (i | k, d) =
  // (i | k + 1, d - 1) + CD (i | k, d - 1), k ascending
  sfor<DMX + 1>([&](auto dd) {
    constexpr int d = dd;
    if constexpr (d > 0)
      sfor<EA + 1>([&](auto i) {
        sfor<FC + 1 - d>([&](auto k) { g[i][k] = g[i][k + 1] + CD * g[i][k]; });
      });
    sfor<CMX + 1>([&](auto c) {
      if constexpr (c + d <= FC) {
        double t[EA + 1];
        sfor<EA + 1>([&](auto i) { t[i] = g[i][c]; });
        sfor<BMX + 1>([&](auto bb) {
          constexpr int b = bb;
          if constexpr (b > 0) sfor<EA + 1 - b>([&](auto i) { t[i] = t[i + 1] + AB * t[i]; });
          sfor<AMX + 1>([&](auto a) {
            if constexpr (a + b <= EA) out[((a * (BMX + 1) + b) * (CMX + 1) + c) * (DMX + 1) + d] = t[a];
          });
        });
      }
    });
  });
}

// one cartesian element (x, y) of a density block of shells (lx at AO bx, ly
// at AO by): sum_{m,k} S_lx[m][x] S_ly[k][y] P[bx + m][by + k]
template <int LX, int LY>
QFE_DI double coop_cart_density(const double* __restrict__ P, int nbf, const double* __restrict__ sph, int bx, int by,
                                int x, int y) {
  constexpr int NX = LX >= 2 ? 2 * LX + 1 : 1, NY = LY >= 2 ? 2 * LY + 1 : 1;
  double s = 0.0;
  for (int m = 0; m < NX; ++m) {
    const double cx = LX >= 2 ? sph[(LX * 9 + m) * 15 + x] : 1.0;
    if (cx == 0.0) continue;
    const double* row = P + (size_t)(bx + (LX >= 2 ? m : x)) * nbf + by;
    for (int k = 0; k < NY; ++k) {
      const double cy = LY >= 2 ? sph[(LY * 9 + k) * 15 + y] : 1.0;
      if (cy != 0.0) s = fma(cx * cy, row[LY >= 2 ? k : y], s);
    }
  }
  return s;
}

}  // namespace qfe
