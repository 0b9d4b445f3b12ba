// Cooperative J/K kernel: one block per canonical shell quartet (the digestion
// of libint2_direct.cpp:414-567, as in eri_class.hpp).
//
// Phase 1: three lanes build the 1-D integrals of one (primitive quartet,
// root) combination in LDS (eri_coop.hpp).  Phase 2: a thread owns the
// cartesian components (a, b, c, all d) of up to NIT triples and sums them
// over the batch in registers; classes with fewer triples than threads split
// the batch over NSL slices.  Then the block transforms the quartet to solid
// harmonics index by index (one column of the index per thread, coefficients
// known at compile time) and forms its J and K updates, each output by one
// thread in a fixed order; the sums over quartets are the fixed-point ones of
// a deterministic build, so the result does not depend on the schedule.
//
// What bounds it: with few quartets the latency of the phases (10-100 us a
// launch whatever the class); with many, the K atomics, two 64-bit adds an
// update at about 26 ps each ((fd|pp) 162 adds, 5 ns a quartet).  Against the
// chunked segment kernels of eri_class.hpp (us a class): (ff|ff) at 167
// quartets 9436 -> 36 (343 chunks), (fd|dd) at 32,280 2492 -> 574 (70), (ss|ss)
// of one water molecule 1072 -> 103 (one lane ran 4096 primitive quartets).
// One wave a block where the accumulators fit: with four, (fd|dp) took 18.8
// instead of 10.2 ns a quartet, three waves waiting for phase 1.
#pragma once

#include "eri_coop.hpp"

namespace qfe {

template <int LA_, int LB_, int LC_, int LD_>
struct JKCoop {
  static constexpr int LA = LA_, LB = LB_, LC = LC_, LD = LD_;
  static constexpr int L = LA + LB + LC + LD;
  static constexpr int NR = L / 2 + 1;
  static constexpr int NA = ncart(LA), NB = ncart(LB), NC = ncart(LC), ND = ncart(LD);
  static constexpr int MA = nsph(LA, true), MB = nsph(LB, true), MC = nsph(LC, true), MD = nsph(LD, true);
  static constexpr int SC = LD + 1, SB = (LC + 1) * SC, SA = (LB + 1) * SB;
  static constexpr int NI = ((LA + 1) * SA) | 1;
  static constexpr int NABC = NA * NB * NC;
  // one wave per quartet while its accumulators fit (40 a thread), then two
  // or four: phase 1 has few lanes at work, and every wave waits for it
  static constexpr int acc(int blk) { return (NABC + blk - 1) / blk * ND; }
  static constexpr int BLK = acc(64) <= 40 ? 64 : (acc(128) <= 40 ? 128 : 256);
  static constexpr int NSL = NABC >= BLK ? 1 : BLK / NABC;
  static constexpr int NIT = NSL > 1 ? 1 : (NABC + BLK - 1) / BLK;
  // combinations per batch: three lanes each, at most 24 KB of tables
  static constexpr int CM_LDS = 3072 / (3 * NI) < 1 ? 1 : 3072 / (3 * NI);
  static constexpr int CM = BLK / 3 < CM_LDS ? BLK / 3 : CM_LDS;
  // after the primitives the tables' space holds the block: [slice][a][b][c][md],
  // then the ping-pong halves of the transforms
  static constexpr int TAB = CM * 3 * NI, BUF0 = NSL * NABC * MD, BUF1 = NA * NB * MC * MD;
  static constexpr int WORK = TAB > BUF0 + BUF1 ? TAB : BUF0 + BUF1;
  static constexpr int NDEN = MA * MB + MC * MD + MA * MC + MA * MD + MB * MC + MB * MD;
  static constexpr int LDS = WORK + NDEN;  // doubles, dynamic
  static constexpr int NOUT = MA * MB + MC * MD + MA * MC + MA * MD + MB * MC + MB * MD;
};

// out[o][m][i] = sum_c S_l[m][c] in[o][c][i] over [OUT][.][IN] by the block
// (l < 2: a copy); NSL > 1: in holds NSL slices, summed in order
template <int L, int OUT, int IN, int NSL, int BLK>
QFE_DI void coop_transform(const double* in, double* out, int tid) {
  constexpr int N = ncart(L), M = nsph(L, true);
  for (int k = tid; k < OUT * IN; k += BLK) {
    const int o = k / IN, i = k % IN;
    double v[N];
    sfor<N>([&](auto c) {
      double s = in[(o * N + c) * IN + i];
      for (int sl = 1; sl < NSL; ++sl) s += in[((sl * OUT + o) * N + c) * IN + i];
      v[c] = s;
    });
    sfor<M>([&](auto m) {
      double s = 0.0;
      sfor<N>([&](auto c) {
        constexpr double f = sph_coef(L, true, m, c);
        if constexpr (f != 0.0) s = fma(f, v[c], s);
      });
      out[(o * M + m) * IN + i] = s;
    });
  }
}

// table offsets of a thread's (a, b, c) triples (10 bits each: a table holds at
// most 257 entries), and its slice of a batch
template <class G>
struct CoopOffsets {
  static_assert(3 * G::NI < 1024, "packed offsets");
  int o[G::NIT], sl;
  QFE_DI int x(int it) const { return o[it] & 1023; }
  QFE_DI int y(int it) const { return o[it] >> 10 & 1023; }
  QFE_DI int z(int it) const { return o[it] >> 20; }
  QFE_DI explicit CoopOffsets(int tid) {
    sfor<G::NIT>([&](auto it) {
      const int k = (tid + it * G::BLK) % G::NABC;
      int ax, ay, az, bx, by, bz, cx, cy, cz;
      coop_xyz<G::LA>(k / (G::NB * G::NC), ax, ay, az);
      coop_xyz<G::LB>(k / G::NC % G::NB, bx, by, bz);
      coop_xyz<G::LC>(k % G::NC, cx, cy, cz);
      o[it] = (ax * G::SA + bx * G::SB + cx * G::SC) | (G::NI + ay * G::SA + by * G::SB + cy * G::SC) << 10 |
              (2 * G::NI + az * G::SA + bz * G::SB + cz * G::SC) << 20;
    });
    sl = G::NSL > 1 ? tid / G::NABC : 0;
  }
};

// The solid-harmonic block V[ma][mb][mc][md] of one quartet, in lds (WORK
// doubles); every thread of the block calls it and it ends on a barrier.
// With sig, primitives that fail the cut lnp with every partner are skipped.
template <class G>
__device__ __forceinline__ double* coop_quartet(const PairHdr& bra, const PairHdr& ket,
                                                const double4* __restrict__ ppos, const double* __restrict__ pk,
                                                const double* __restrict__ sig, const RysArgs& ra, double lnp,
                                                const CoopOffsets<G>& of, double* lds) {
  constexpr double TWO_PI_52 = 34.98683665524972;
  double* const tab = lds;
  const int tid = (int)threadIdx.x, lane = tid & 63;
  // primitives that can pass the engine's cut: a prefix of both lists
  // (those inside that fail it with their partner are evaluated too)
  int nbp = bra.nprim, nkp = ket.nprim;
  if (sig != nullptr && bra.nprim > 0 && ket.nprim > 0) {
    const double sb0 = sig[bra.prim0], sk0 = sig[ket.prim0];
    nbp = nkp = 0;
    for (int i = lane; i - lane < bra.nprim; i += 64)
      nbp += __popcll(__ballot(i < bra.nprim && !(sig[bra.prim0 + (i < bra.nprim ? i : 0) * bra.pstride] + sk0 < lnp)));
    for (int i = lane; i - lane < ket.nprim; i += 64)
      nkp += __popcll(__ballot(i < ket.nprim && !(sig[ket.prim0 + (i < ket.nprim ? i : 0) * ket.pstride] + sb0 < lnp)));
  }
  double acc[G::NIT][G::ND];
  sfor<G::NIT>([&](auto it) { sfor<G::ND>([&](auto d) { acc[it][d] = 0.0; }); });
  const int ncomb = nbp * nkp * G::NR;
  for (int g0 = 0; g0 < ncomb; g0 += G::CM) {
    const int nc = ncomb - g0 < G::CM ? ncomb - g0 : G::CM;
    if (tid < 3 * nc) {
      const int i = tid / 3, x = tid % 3;
      const int pr = (g0 + i) / G::NR, r = (g0 + i) % G::NR;
      const int ib = bra.prim0 + pr % nbp * bra.pstride, ik = ket.prim0 + pr / nbp * ket.pstride;
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
      rys_1d_store<G::LA + G::LB, G::LC + G::LD, G::LA, G::LB, G::LC, G::LD>(
          s, (Pc - Ac) - xa * PQ, (Qc - Cc) + xc * PQ, 0.5 * rpq * ur, h2p - h2p * xa, h2q - h2q * xc, Ac - Bc,
          Cc - Dc, tab + (i * 3 + x) * G::NI);
    }
    __syncthreads();
    for (int i = of.sl; i < nc; i += G::NSL) {
      const double* tb = tab + i * 3 * G::NI;
      sfor<G::NIT>([&](auto it) {
        double vx[G::LD + 1], vy[G::LD + 1], vz[G::LD + 1];
        sfor<G::LD + 1>([&](auto d) {
          vx[d] = tb[of.x(it) + d];
          vy[d] = tb[of.y(it) + d];
          vz[d] = tb[of.z(it) + d];
        });
        sfor<G::ND>([&](auto d) {
          constexpr int dx = cart_x(G::LD, d), dy = cart_y(G::LD, d), dz = cart_z(G::LD, d);
          acc[it][d] = fma(vx[dx] * vy[dy], vz[dz], acc[it][d]);
        });
      });
    }
    __syncthreads();
  }
  if (ncomb == 0) __syncthreads();  // what the caller put in LDS is in place
  // d index in registers, then c, b and a through LDS
  double* const buf0 = lds;
  double* const buf1 = lds + G::BUF0;
  sfor<G::NIT>([&](auto it) {
    const int k = tid + it * G::BLK;
    if (G::NSL > 1 ? tid < G::NSL * G::NABC : k < G::NABC) {
      double* o = buf0 + (size_t)k * G::MD;  // k = slice * NABC + triple when NSL > 1
      sfor<G::MD>([&](auto m) {
        double s = 0.0;
        sfor<G::ND>([&](auto d) {
          constexpr double f = sph_coef(G::LD, true, m, d);
          if constexpr (f != 0.0) s = fma(f, acc[it][d], s);
        });
        o[m] = s;
      });
    }
  });
  __syncthreads();
  coop_transform<G::LC, G::NA * G::NB, G::MD, G::NSL, G::BLK>(buf0, buf1, tid);
  double* V = buf1;
  double* W = buf0;
  __syncthreads();
  if constexpr (G::LB >= 2) {
    coop_transform<G::LB, G::NA, G::MC * G::MD, 1, G::BLK>(V, W, tid);
    double* s = V;
    V = W;
    W = s;
    __syncthreads();
  }
  if constexpr (G::LA >= 2) {
    coop_transform<G::LA, 1, G::MB * G::MC * G::MD, 1, G::BLK>(V, W, tid);
    V = W;
    __syncthreads();
  }
  return V;
}

template <class G>
__global__ __launch_bounds__(G::BLK) void k_eri_jk_coop(
    const int2* __restrict__ tasks, long long ntask, int run, const PairHdr* __restrict__ pairs,
    const double4* __restrict__ ppos, const double* __restrict__ pk, const double* __restrict__ sig, RysArgs ra,
    const double* __restrict__ P, double* __restrict__ J, double* __restrict__ K, int nbf, double kscale,
    const int2* __restrict__ segs, int bra0, double* __restrict__ jbuf, const long long* __restrict__ jslot,
    const int2* __restrict__ qpos, const double* __restrict__ pmax, int prim_screen, int det,
    unsigned long long* __restrict__ Jx, unsigned long long* __restrict__ Kx, int* __restrict__ fx_over) {
  extern __shared__ double lds[];
  double* const dab = lds + G::WORK;
  double* const dcd = dab + G::MA * G::MB;
  double* const dac = dcd + G::MC * G::MD;
  double* const dad = dac + G::MA * G::MC;
  double* const dbc = dad + G::MA * G::MD;
  double* const dbd = dbc + G::MB * G::MC;
  const int tid = (int)threadIdx.x;
  const bool doJ = det ? Jx != nullptr : J != nullptr, doK = kscale != 0.0;
  const double lnp = prim_ln_cut<double>(pmax, prim_screen);
  const CoopOffsets<G> of(tid);
  int bad = 0;
  // J_ab: thread k < MA MB owns entry k of the current bra pair's block and
  // sums it over the tasks of the run in registers (fixed-point words, or a
  // double), added to J when the bra pair changes: one global add a run
  // instead of one a task
  static_assert(G::MA * G::MB <= G::BLK, "a thread per J_ab entry");
  long long jhi = 0, jlo = 0;
  double jsum = 0.0;
  size_t jent = 0;
  auto flush = [&]() {
    if (det) {
      const long long carry = jlo >> 42;
      jhi += carry;
      jlo -= carry * (1ll << 42);
      if (jhi) atomicAdd(Jx + 2 * jent, (unsigned long long)jhi);
      if (jlo) atomicAdd(Jx + 2 * jent + 1, (unsigned long long)jlo);
    } else if (jsum != 0.0) {
      unsafeAtomicAdd(&J[jent], jsum);
    }
    jhi = jlo = 0;
    jsum = 0.0;
  };
  // runs of consecutive tasks: the tasks of one bra pair are neighbours
  const long long nrun = (ntask + run - 1) / run;
  for (long long rn = blockIdx.x; rn < nrun; rn += gridDim.x) {
    const long long te = (rn + 1) * run < ntask ? (rn + 1) * run : ntask;
    for (long long t = rn * run; t < te; ++t) {
      const int2 tk = tasks[t];
      const PairHdr bra = pairs[tk.x], ket = pairs[tk.y];
      const int i0 = bra.bfa, j0 = bra.bfb, k0 = ket.bfa, l0 = ket.bfb;
      if (doJ && tid < G::MA * G::MB) {
        const size_t e = (size_t)(i0 + tid / G::MB) * nbf + j0 + tid % G::MB;
        if (e != jent) {
          flush();
          jent = e;
        }
      }
      __syncthreads();  // the last task's readers are done
      {
        const size_t n = (size_t)nbf;
        for (int i = tid; i < G::MA * G::MB; i += G::BLK) dab[i] = P[(i0 + i / G::MB) * n + j0 + i % G::MB];
        for (int i = tid; i < G::MC * G::MD; i += G::BLK) dcd[i] = P[(k0 + i / G::MD) * n + l0 + i % G::MD];
        for (int i = tid; i < G::MA * G::MC; i += G::BLK) dac[i] = P[(i0 + i / G::MC) * n + k0 + i % G::MC];
        for (int i = tid; i < G::MA * G::MD; i += G::BLK) dad[i] = P[(i0 + i / G::MD) * n + l0 + i % G::MD];
        for (int i = tid; i < G::MB * G::MC; i += G::BLK) dbc[i] = P[(j0 + i / G::MC) * n + k0 + i % G::MC];
        for (int i = tid; i < G::MB * G::MD; i += G::BLK) dbd[i] = P[(j0 + i / G::MD) * n + l0 + i % G::MD];
      }
      const double* V = coop_quartet<G>(bra, ket, ppos, pk, sig, ra, lnp, of, lds);
      // digestion: V[ma][mb][mc][md], one output per thread
      const double deg =
          (bra.sa == bra.sb ? 1.0 : 2.0) * (ket.sa == ket.sb ? 1.0 : 2.0) * (tk.x == tk.y ? 1.0 : 2.0);
      for (int o = tid; o < G::NOUT; o += G::BLK) {
        int k = o;
        double s = 0.0;
        int row, col;
        bool isJ = false;
        double* slot = nullptr;
        if (k < G::MA * G::MB) {  // J_ab (k = tid)
          const double* v = V + k * (G::MC * G::MD);
          for (int e = 0; e < G::MC * G::MD; ++e) s = fma(v[e], dcd[e], s);
          s *= deg;
          if (doJ && det) {
            long long hi, lo;
            bad |= !(fabs(s) < kFxMax);
            fx_split(s, hi, lo);
            jhi += hi;
            jlo += lo;
          } else {
            jsum += s;
          }
          continue;
        } else if ((k -= G::MA * G::MB) < G::MC * G::MD) {  // J_cd
          isJ = true;
          for (int e = 0; e < G::MA * G::MB; ++e) s = fma(V[e * (G::MC * G::MD) + k], dab[e], s);
          row = k0 + k / G::MD;
          col = l0 + k % G::MD;
          if (jbuf) {
            const int2 qp = qpos[tk.y];
            slot = jbuf + jslot[segs[tk.x - bra0].x + qp.x] + (long long)qp.y * (G::MC * G::MD) + k;
          }
        } else if ((k -= G::MC * G::MD) < G::MA * G::MC) {  // K_ac
          const int a = k / G::MC, c = k % G::MC;
          for (int b = 0; b < G::MB; ++b)
            for (int d = 0; d < G::MD; ++d)
              s = fma(V[((a * G::MB + b) * G::MC + c) * G::MD + d], dbd[b * G::MD + d], s);
          row = i0 + a;
          col = k0 + c;
        } else if ((k -= G::MA * G::MC) < G::MA * G::MD) {  // K_ad
          const int a = k / G::MD, d = k % G::MD;
          for (int b = 0; b < G::MB; ++b)
            for (int c = 0; c < G::MC; ++c)
              s = fma(V[((a * G::MB + b) * G::MC + c) * G::MD + d], dbc[b * G::MC + c], s);
          row = i0 + a;
          col = l0 + d;
        } else if ((k -= G::MA * G::MD) < G::MB * G::MC) {  // K_bc
          const int b = k / G::MC, c = k % G::MC;
          for (int a = 0; a < G::MA; ++a)
            for (int d = 0; d < G::MD; ++d)
              s = fma(V[((a * G::MB + b) * G::MC + c) * G::MD + d], dad[a * G::MD + d], s);
          row = j0 + b;
          col = k0 + c;
        } else {  // K_bd
          k -= G::MB * G::MC;
          const int b = k / G::MD, d = k % G::MD;
          for (int a = 0; a < G::MA; ++a)
            for (int c = 0; c < G::MC; ++c)
              s = fma(V[((a * G::MB + b) * G::MC + c) * G::MD + d], dac[a * G::MC + c], s);
          row = j0 + b;
          col = l0 + d;
        }
        s *= deg;
        const size_t e = (size_t)row * nbf + col;
        if (isJ) {
          if (!doJ) continue;
          if (slot)
            *slot = s;
          else if (det)
            fx_global_add(Jx + 2 * e, s, bad);
          else
            unsafeAtomicAdd(&J[e], s);
        } else if (doK) {
          if (det)
            fx_global_add(Kx + 2 * e, s, bad);
          else
            unsafeAtomicAdd(&K[e], 0.25 * kscale * s);
        }
      }
    }
    if (doJ && tid < G::MA * G::MB) flush();
  }
  if (bad) *fx_over = 1;
}

// allow a launch of kern with `bytes` of dynamic LDS
template <class KERN>
void coop_lds(KERN kern, int bytes) {
  if (bytes > 65536 &&
      hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, bytes) != hipSuccess) {
    (void)hipGetLastError();
    throw std::runtime_error("cooperative kernel: launch configuration rejected");
  }
}

// q2[pair] = sum of squares of (ab|ab) (schwarz.cpp:26-78), one block per pair
template <class G>
__global__ __launch_bounds__(G::BLK) void k_schwarz_coop(const int* __restrict__ plist,
                                                         const PairHdr* __restrict__ pairs,
                                                         const double4* __restrict__ ppos,
                                                         const double* __restrict__ pk, RysArgs ra,
                                                         double* __restrict__ q2) {
  extern __shared__ double lds[];
  const int p = plist[blockIdx.x];
  const PairHdr pr = pairs[p];
  const CoopOffsets<G> of((int)threadIdx.x);
  const double* V = coop_quartet<G>(pr, pr, ppos, pk, nullptr, ra, 0.0, of, lds);
  double s = 0.0;
  for (int i = (int)threadIdx.x; i < G::MA * G::MB * G::MC * G::MD; i += G::BLK) s = fma(V[i], V[i], s);
  s = wave_sum(s);
  double* part = lds + G::WORK;  // past V
  if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = s;
  __syncthreads();
  if (threadIdx.x == 0) {
    double t = part[0];
    for (int w = 1; w < G::BLK / 64; ++w) t += part[w];
    q2[p] = t;
  }
}

template <int LA, int LB>
void schwarz_coop(const SchwarzLaunch& a, hipStream_t s) {
  using G = JKCoop<LA, LB, LA, LB>;
  if (a.npair <= 0) return;
  auto kern = k_schwarz_coop<G>;
  constexpr int bytes = (G::WORK + G::BLK / 64) * (int)sizeof(double);
  coop_lds(kern, bytes);
  hipLaunchKernelGGL(kern, dim3((unsigned)a.npair), dim3(G::BLK), bytes, s, a.plist, a.pairs, a.ppos, a.pk, *a.ra,
                     a.q2);
}

template <int LA, int LB, int LC, int LD>
void jk_coop(const JKLaunch& a, hipStream_t s) {
  using G = JKCoop<LA, LB, LC, LD>;
  if (a.ntask <= 0) return;
  auto kern = k_eri_jk_coop<G>;
  constexpr int bytes = G::LDS * (int)sizeof(double);
  coop_lds(kern, bytes);
  const int run = (int)std::max(1LL, std::min(64LL, a.ntask / 8192));
  const long long grid = std::min((a.ntask + run - 1) / run, 65536LL);
  hipLaunchKernelGGL(kern, dim3((unsigned)grid), dim3(G::BLK), bytes, s, a.tasks, a.ntask, run, a.pairs, a.ppos, a.pk,
                     a.ra->sig, *a.ra, a.P, a.J, a.K, a.nbf, a.kscale, a.segs, a.bra0, a.jbuf, a.jslot, a.qpos, a.pmax,
                     a.prim_screen, a.det, a.Jx, a.Kx, a.fx_over);
}

}  // namespace qfe
