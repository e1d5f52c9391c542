// One-electron integrals S, T, V and their part of the nuclear gradient,
//   dL1/dR  with  L1 = Tr(Dh (T + V)) - Tr(Ws S),
// holding the symmetric matrices Dh and Ws fixed (for RHF, Dh = D and Ws the
// energy-weighted density).
//
// The reference forms the same quantities on the CPU: build_int1e_cart
// (asuka/integrals/int1e_cart.py:1423-1434), contract_dhcore_cart (:1738-) for
// d(T+V) against D and contract_dS_ip_cart (:1545-1737) for the overlap
// (Pulay) term, assembled in asuka/mcscf/nuc_grad_direct.py:151-181.
//
// S and T: 1-D overlap recursion and the kinetic-from-overlap relation
// (int1e_cart.py:77-115, :758-787). V: Rys quadrature with a point-charge ket
// (the q -> infinity limit of the ERI recursion), G[a+1] = (PA - x PC) G[a] +
// a (1-x)/(2p) G[a-1], transfer to the second centre, weight
// -Z 2 pi / p exp(-mu AB^2) sum_u w_u Ix Iy Iz, T = p |PC|^2; equal to the
// reference's McMurchie-Davidson form (int1e_cart.py:1031-1190). Centre
// derivatives of a primitive, d/dA_x <a| = 2 alpha <a+1_x| - a_x <a-1_x|,
// apply to S, T and each nucleus' V; the derivative with respect to the
// position of nucleus C follows from translational invariance,
// dV^C/dC = -(dV^C/dA + dV^C/dB).
//
// Work mapping: one wavefront per shell pair, the pair's angular momenta as
// template parameters. 64 primitive pairs at a time, one per lane (zero
// coefficient products, which general contractions are full of, are skipped
// by compacting the lanes); S and T are summed by the primitive's own lane.
// For V the lanes are split into groups over the nuclei (group size: the
// number of nuclei rounded up to a power of two, at most 64) and each group
// takes one primitive pair, so a lane is one (primitive pair, nucleus) and a
// small molecule fills the wave with primitives, a large one with nuclei. The
// primitive's data come from its lane by shuffles: no LDS, no barriers. What
// bounds it is FP64 arithmetic (root polynomials and 1-D tables) and, below
// about 10 nuclei, the launches. Measured at (H2O)16 cc-pVDZ, S, T, V and the
// gradient term together: 121.5 ms with one thread per shell pair and run-time
// angular momenta (tables in scratch memory, 289 wavefronts on the chip), now
// 0.60 ms (kernels 0.17 and 0.36 ms).
#include "jk_internal.h"
#include "rys_eval.h"

namespace {

constexpr double kPi = 3.14159265358979323846;
constexpr int kWaves = 4;             // shell pairs (wavefronts) in flight per workgroup
constexpr int kLdsGradMaxAtoms = 512;  // LDS accumulator of the nuclei's gradient up to this many

constexpr int nc1(int l) { return (l + 1) * (l + 2) / 2; }
// exponent of component i of angular momentum l on axis ax (lx-descending, ly-descending)
constexpr int ce(int l, int i, int ax) {
  int k = 0;
  for (int x = l; x >= 0; --x)
    for (int y = l - x; y >= 0; --y) {
      if (k == i) return ax == 0 ? x : ax == 1 ? y : l - x - y;
      ++k;
    }
  return 0;
}

__device__ __forceinline__ double lane_get(double v, int src) { return __shfl(v, src); }

// One primitive pair of a shell pair, one per lane.
struct Prim {
  double a, b, p, ip, cK, c;  // exponents, p = a + b, 1/p, c exp(-mu AB^2), coefficient product c
  double P[3];
};

// Primitive pair `cand` of shells A and B; false for a zero coefficient
// product or past the end.
__device__ __forceinline__ bool load_prim(const Int1eArgs& g, int A, int B, int npB, int ncand, int cand,
                                          const double* cA, const double* cB, double AB2, Prim& r) {
  const bool in = cand < ncand;
  const int ia = in ? cand / npB : 0, ib = in ? cand - ia * npB : 0;
  const int pa = g.pstart[A] + ia, pb = g.pstart[B] + ib;
  r.a = g.pexp[pa];
  r.b = g.pexp[pb];
  r.c = in ? g.pcoef[pa] * g.pcoef[pb] : 0.0;
  r.p = r.a + r.b;
  r.ip = 1.0 / r.p;
  r.cK = r.c * exp(-r.a * r.b * r.ip * AB2);
#pragma unroll
  for (int x = 0; x < 3; ++x) r.P[x] = (r.a * cA[x] + r.b * cB[x]) * r.ip;
  return r.cK != 0.0;
}

// 1-D overlaps S[i][j], i <= I, j <= J, in units of S[0][0].
template <int I, int J>
__device__ __forceinline__ void ovl1(double PA, double PB, double i2p, double (&S)[I + 1][J + 1]) {
  S[0][0] = 1.0;
#pragma unroll
  for (int j = 0; j < J; ++j) S[0][j + 1] = PB * S[0][j] + (j > 0 ? j * i2p * S[0][j > 0 ? j - 1 : 0] : 0.0);
#pragma unroll
  for (int i = 0; i < I; ++i) {
    S[i + 1][0] = PA * S[i][0] + (i > 0 ? i * i2p * S[i > 0 ? i - 1 : 0][0] : 0.0);
#pragma unroll
    for (int j = 0; j < J; ++j)
      S[i + 1][j + 1] = PA * S[i][j + 1] + (i > 0 ? i * i2p * S[i > 0 ? i - 1 : 0][j + 1] : 0.0) + (j + 1) * i2p * S[i][j];
  }
}

// 1-D kinetic factor -1/2 <i| d2/dx2 |j> with the ket exponent b (i, j compile-time after unrolling).
template <int I, int J>
__device__ __forceinline__ double kin1(const double (&S)[I + 1][J + 1], int i, int j, double b) {
  double v = b * (2.0 * j + 1.0) * S[i][j] - 2.0 * b * b * S[i][j + 2];
  if (j >= 2) v -= 0.5 * (double)(j * (j - 1)) * S[i][j >= 2 ? j - 2 : 0];
  return v;
}

// 1-D nuclear-attraction table N[i][j], i <= I, j <= J, i + j <= M, for one root.
template <int I, int J, int M>
__device__ __forceinline__ void nuc1(double c0, double b1, double AB, double (&N)[I + 1][J + 1]) {
  double G[M + 1];
  G[0] = 1.0;
  if (M > 0) G[1] = c0;
#pragma unroll
  for (int a = 1; a < M; ++a) G[a + 1] = c0 * G[a] + a * b1 * G[a - 1];
#pragma unroll
  for (int j = 0; j <= J; ++j) {
#pragma unroll
    for (int i = 0; i <= I; ++i)
      if (i + j <= M) N[i][j] = G[i];
#pragma unroll
    for (int i = 0; i < M - j; ++i) G[i] = G[i + 1] + AB * G[i];  // |i, j+1) = |i+1, j) + AB |i, j)
  }
}

// Lanes holding a valid primitive pair, packed: on lane r the lane of the
// r-th valid one.
__device__ __forceinline__ int pack_lanes(bool ok, int lane, int& n) {
  const unsigned long long m = __builtin_amdgcn_ballot_w64(ok);
  n = __popcll(m);
  const int rank = __popcll(m & ((1ull << lane) - 1ull));
  // lanes without a valid pair send to the slots after the valid ones
  return __builtin_amdgcn_ds_permute(4 * (ok ? rank : n + lane - rank), lane);
}

// S, T, V of A components [A0, A1) of one shell pair.
template <int LA, int LB, int A0, int A1>
__device__ __forceinline__ void pair_int1e(const DevBasis& b, const Int1eArgs& g, int sp, double* S, double* T,
                                           double* V) {
  constexpr int NB = nc1(LB), NAL = A1 - A0, NC = NAL * NB, NR = (LA + LB) / 2 + 1;
  const int lane = threadIdx.x & 63;
  const int A = __builtin_amdgcn_readfirstlane(b.sp_A[sp]), B = __builtin_amdgcn_readfirstlane(b.sp_B[sp]);
  double cA[3], cB[3], AB[3];
#pragma unroll
  for (int x = 0; x < 3; ++x) {
    cA[x] = b.shell_xyz[3 * A + x];
    cB[x] = b.shell_xyz[3 * B + x];
    AB[x] = cA[x] - cB[x];
  }
  const double AB2 = AB[0] * AB[0] + AB[1] * AB[1] + AB[2] * AB[2];
  const int npB = g.pnum[B], ncand = g.pnum[A] * npB;
  const long long N = b.nao;
  const int a0 = b.shell_ao[A] + A0, b0 = b.shell_ao[B];
  auto put = [&](double* M, const double (&v)[NC]) {  // wave sums, one lane per element writes
#pragma unroll
    for (int e = 0; e < NC; ++e) {
      const double s = wave_total(v[e]);
      if (lane == (e & 63)) {
        const long long r = a0 + e / NB, c = b0 + e % NB;
        if (A == B && c > r) continue;  // the block's lower half serves both: exactly symmetric
        M[r * N + c] = s;
        M[c * N + r] = s;
      }
    }
  };
  if (S || T) {
    double s[NC], t[NC];
#pragma unroll
    for (int e = 0; e < NC; ++e) s[e] = t[e] = 0.0;
    for (int c0 = 0; c0 < ncand; c0 += 64) {
      Prim r;
      if (!load_prim(g, A, B, npB, ncand, c0 + lane, cA, cB, AB2, r)) continue;
      double Sx[3][LA + 1][LB + 3];
#pragma unroll
      for (int x = 0; x < 3; ++x) ovl1<LA, LB + 2>(r.P[x] - cA[x], r.P[x] - cB[x], 0.5 * r.ip, Sx[x]);
      const double u = kPi * r.ip, o = r.cK * u * sqrt(u);
#pragma unroll
      for (int i = 0; i < NAL; ++i)
#pragma unroll
        for (int j = 0; j < NB; ++j) {
          const int ex = ce(LA, A0 + i, 0), ey = ce(LA, A0 + i, 1), ez = ce(LA, A0 + i, 2);
          const int fx = ce(LB, j, 0), fy = ce(LB, j, 1), fz = ce(LB, j, 2);
          const double sx = Sx[0][ex][fx], sy = Sx[1][ey][fy], sz = Sx[2][ez][fz];
          s[i * NB + j] += o * sx * sy * sz;
          t[i * NB + j] += o * (kin1<LA, LB + 2>(Sx[0], ex, fx, r.b) * sy * sz +
                                sx * kin1<LA, LB + 2>(Sx[1], ey, fy, r.b) * sz +
                                sx * sy * kin1<LA, LB + 2>(Sx[2], ez, fz, r.b));
        }
    }
    if (S) put(S, s);
    if (T) put(T, t);
  }
  if (!V) return;
  double v[NC];
#pragma unroll
  for (int e = 0; e < NC; ++e) v[e] = 0.0;
  const int G = 1 << g.lg_group, sub = lane >> g.lg_group, nl = lane & (G - 1);
  for (int c0 = 0; c0 < ncand; c0 += 64) {
    Prim r;
    const bool ok = load_prim(g, A, B, npB, ncand, c0 + lane, cA, cB, AB2, r);
    int n;
    const int who = pack_lanes(ok, lane, n);
    for (int k0 = 0; k0 < n; k0 += 64 >> g.lg_group) {
      const int src = __shfl(who, (k0 + sub) & 63);
      const double p = lane_get(r.p, src), ip = lane_get(r.ip, src), cK = lane_get(r.cK, src);
      const double P[3] = {lane_get(r.P[0], src), lane_get(r.P[1], src), lane_get(r.P[2], src)};
      const double pref = -2.0 * kPi * ip * cK;
      for (int n0 = 0; n0 < g.natm; n0 += G) {
        const int ic = n0 + nl;
        if (k0 + sub >= n || ic >= g.natm || g.aZ[ic] == 0.0) continue;
        const double PC[3] = {P[0] - g.axyz[3 * ic], P[1] - g.axyz[3 * ic + 1], P[2] - g.axyz[3 * ic + 2]};
        double rx[NR], rw[NR];
        rys_roots_blk<NR, double>(p * (PC[0] * PC[0] + PC[1] * PC[1] + PC[2] * PC[2]),
                                  rys_dev::rys_coef + rys_c::coef_off[NR], rx, rw);
        const double zp = pref * g.aZ[ic];
#pragma unroll
        for (int u = 0; u < NR; ++u) {
          double I[3][LA + 1][LB + 1];
#pragma unroll
          for (int x = 0; x < 3; ++x)
            nuc1<LA, LB, LA + LB>(P[x] - cA[x] - rx[u] * PC[x], 0.5 * ip * (1.0 - rx[u]), AB[x], I[x]);
          const double w = zp * rw[u];
#pragma unroll
          for (int i = 0; i < NAL; ++i)
#pragma unroll
            for (int j = 0; j < NB; ++j)
              v[i * NB + j] += w * I[0][ce(LA, A0 + i, 0)][ce(LB, j, 0)] * I[1][ce(LA, A0 + i, 1)][ce(LB, j, 1)] *
                               I[2][ce(LA, A0 + i, 2)][ce(LB, j, 2)];
        }
      }
    }
  }
  put(V, v);
}

// The A components of the large classes are split over blockIdx.y so that a
// lane's sums stay in registers (at most 36 of each matrix).
template <int LA, int LB>
constexpr int kSplit = nc1(LA) * nc1(LB) <= 36 ? 1 : (nc1(LA) * nc1(LB) + 29) / 30;

template <int LA, int LB, int CH>
__device__ __forceinline__ void dispatch_int1e(int ch, const DevBasis& b, const Int1eArgs& g, int sp, double* S,
                                               double* T, double* V) {
  constexpr int SA = kSplit<LA, LB>, NA = nc1(LA);
  if constexpr (CH < SA) {
    if (ch == CH)
      pair_int1e<LA, LB, CH * NA / SA, (CH + 1) * NA / SA>(b, g, sp, S, T, V);
    else
      dispatch_int1e<LA, LB, CH + 1>(ch, b, g, sp, S, T, V);
  }
}

template <int LA, int LB>
__global__ __launch_bounds__(64 * kWaves) void k_int1e(const DevBasis b, const Int1eArgs g, const int* list, int n,
                                                       double* S, double* T, double* V) {
  const int k = __builtin_amdgcn_readfirstlane((int)(blockIdx.x * kWaves + (threadIdx.x >> 6)));
  if (k >= n) return;  // uniform per wave; no barriers below
  dispatch_int1e<LA, LB, 0>(blockIdx.y, b, g, __builtin_amdgcn_readfirstlane(list[k]), S, T, V);
}

// Gradient term of one shell pair; nuclei's forces go to sg (LDS) or the output.
template <int LA, int LB>
__device__ __forceinline__ void pair_grad(const DevBasis& b, const Int1eArgs& g, int sp, const double* Dh,
                                          const double* Ws, double* sg) {
  constexpr int NA = nc1(LA), NB = nc1(LB), NR = (LA + LB + 1) / 2 + 1;
  const int lane = threadIdx.x & 63;
  const int A = __builtin_amdgcn_readfirstlane(b.sp_A[sp]), B = __builtin_amdgcn_readfirstlane(b.sp_B[sp]);
  double cA[3], cB[3], AB[3];
#pragma unroll
  for (int x = 0; x < 3; ++x) {
    cA[x] = b.shell_xyz[3 * A + x];
    cB[x] = b.shell_xyz[3 * B + x];
    AB[x] = cA[x] - cB[x];
  }
  const double AB2 = AB[0] * AB[0] + AB[1] * AB[1] + AB[2] * AB[2];
  const int npB = g.pnum[B], ncand = g.pnum[A] * npB;
  const long long N = b.nao;
  const long long d0 = (long long)b.shell_ao[A] * N + b.shell_ao[B];  // wave-uniform block of Dh and Ws
  const double fold = A != B ? 2.0 : 1.0;
  double gA[3] = {0, 0, 0}, gB[3] = {0, 0, 0};
  const int G = 1 << g.lg_group, sub = lane >> g.lg_group, nl = lane & (G - 1);
  for (int c0 = 0; c0 < ncand; c0 += 64) {
    Prim r;
    const bool ok = load_prim(g, A, B, npB, ncand, c0 + lane, cA, cB, AB2, r);
    if (ok) {  // overlap and kinetic energy
      constexpr int I = LA + 1, J = LB + 3;
      const double a2 = 2.0 * r.a, b2 = 2.0 * r.b;
      double S[3][I + 1][J + 1];
#pragma unroll
      for (int x = 0; x < 3; ++x) ovl1<I, J>(r.P[x] - cA[x], r.P[x] - cB[x], 0.5 * r.ip, S[x]);
      const double u = kPi * r.ip, o = fold * r.cK * u * sqrt(u);
#pragma unroll
      for (int i = 0; i < NA; ++i)
#pragma unroll
        for (int j = 0; j < NB; ++j) {
          const double dh = Dh ? o * Dh[d0 + i * N + j] : 0.0, ws = Ws ? o * Ws[d0 + i * N + j] : 0.0;
          double s1[3], k1[3];
#pragma unroll
          for (int x = 0; x < 3; ++x) {
            s1[x] = S[x][ce(LA, i, x)][ce(LB, j, x)];
            k1[x] = kin1<I, J>(S[x], ce(LA, i, x), ce(LB, j, x), r.b);
          }
#pragma unroll
          for (int x = 0; x < 3; ++x) {
            const int e = ce(LA, i, x), f = ce(LB, j, x), o1 = (x + 1) % 3, o2 = (x + 2) % 3;
            const double so = s1[o1] * s1[o2], ko = k1[o1] * s1[o2] + s1[o1] * k1[o2];
            double dsa = a2 * S[x][e + 1][f], dka = a2 * kin1<I, J>(S[x], e + 1, f, r.b);
            if (e > 0) {
              dsa -= e * S[x][e > 0 ? e - 1 : 0][f];
              dka -= e * kin1<I, J>(S[x], e > 0 ? e - 1 : 0, f, r.b);
            }
            double dsb = b2 * S[x][e][f + 1], dkb = b2 * kin1<I, J>(S[x], e, f + 1, r.b);
            if (f > 0) {
              dsb -= f * S[x][e][f > 0 ? f - 1 : 0];
              dkb -= f * kin1<I, J>(S[x], e, f > 0 ? f - 1 : 0, r.b);
            }
            gA[x] += dh * (dka * so + dsa * ko) - ws * dsa * so;
            gB[x] += dh * (dkb * so + dsb * ko) - ws * dsb * so;
          }
        }
    }
    if (!Dh) continue;
    int n;
    const int who = pack_lanes(ok, lane, n);
    for (int n0 = 0; n0 < g.natm; n0 += G) {
      const int ic = n0 + nl;
      const double Z = ic < g.natm ? g.aZ[ic] : 0.0;
      const bool in = Z != 0.0;
      double C[3], gC[3] = {0, 0, 0};
#pragma unroll
      for (int x = 0; x < 3; ++x) C[x] = in ? g.axyz[3 * ic + x] : 0.0;
      for (int k0 = 0; k0 < n; k0 += 64 >> g.lg_group) {
        const int src = __shfl(who, (k0 + sub) & 63);
        const double p = lane_get(r.p, src), ip = lane_get(r.ip, src), cK = lane_get(r.cK, src);
        const double a2 = 2.0 * lane_get(r.a, src), b2 = 2.0 * lane_get(r.b, src);
        const double P[3] = {lane_get(r.P[0], src), lane_get(r.P[1], src), lane_get(r.P[2], src)};
        if (!in || k0 + sub >= n) continue;
        const double PC[3] = {P[0] - C[0], P[1] - C[1], P[2] - C[2]};
        double rx[NR], rw[NR];
        rys_roots_blk<NR, double>(p * (PC[0] * PC[0] + PC[1] * PC[1] + PC[2] * PC[2]),
                                  rys_dev::rys_coef + rys_c::coef_off[NR], rx, rw);
        const double pref = -2.0 * kPi * ip * cK * Z * fold;
        double vA[3] = {0, 0, 0}, vB[3] = {0, 0, 0};
#pragma unroll
        for (int u = 0; u < NR; ++u) {
          double I[3][LA + 2][LB + 2];
#pragma unroll
          for (int x = 0; x < 3; ++x)
            nuc1<LA + 1, LB + 1, LA + LB + 1>(P[x] - cA[x] - rx[u] * PC[x], 0.5 * ip * (1.0 - rx[u]), AB[x], I[x]);
          const double w = pref * rw[u];
#pragma unroll
          for (int i = 0; i < NA; ++i)
#pragma unroll
            for (int j = 0; j < NB; ++j) {
              const double dh = w * Dh[d0 + i * N + j];
#pragma unroll
              for (int x = 0; x < 3; ++x) {
                const int e = ce(LA, i, x), f = ce(LB, j, x), o1 = (x + 1) % 3, o2 = (x + 2) % 3;
                const double oth = dh * I[o1][ce(LA, i, o1)][ce(LB, j, o1)] * I[o2][ce(LA, i, o2)][ce(LB, j, o2)];
                double da = a2 * I[x][e + 1][f], db = b2 * I[x][e][f + 1];
                if (e > 0) da -= e * I[x][e > 0 ? e - 1 : 0][f];
                if (f > 0) db -= f * I[x][e][f > 0 ? f - 1 : 0];
                vA[x] = fma(da, oth, vA[x]);
                vB[x] = fma(db, oth, vB[x]);
              }
            }
        }
#pragma unroll
        for (int x = 0; x < 3; ++x) {
          gA[x] += vA[x];
          gB[x] += vB[x];
          gC[x] -= vA[x] + vB[x];
        }
      }
      if (in)
#pragma unroll
        for (int x = 0; x < 3; ++x) atomicAdd((sg ? sg : g.grad) + 3 * ic + x, gC[x]);
    }
  }
  const int atA = g.shell_atom[A], atB = g.shell_atom[B];
#pragma unroll
  for (int x = 0; x < 3; ++x) {
    const double sa = wave_total(gA[x]), sb = wave_total(gB[x]);
    if (lane == 0) {
      atomicAdd((sg ? sg : g.grad) + 3 * atA + x, sa);
      atomicAdd((sg ? sg : g.grad) + 3 * atB + x, sb);
    }
  }
}

template <int LA, int LB>
__global__ __launch_bounds__(64 * kWaves) void k_int1e_grad(const DevBasis b, const Int1eArgs g, const int* list,
                                                            int n, const double* Dh, const double* Ws) {
  __shared__ double sgrad[3 * kLdsGradMaxAtoms];
  const bool lds = g.natm <= kLdsGradMaxAtoms;
  if (lds)
    for (int t = threadIdx.x; t < 3 * g.natm; t += 64 * kWaves) sgrad[t] = 0.0;
  __syncthreads();
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  for (int k = blockIdx.x * kWaves + wave; k < n; k += gridDim.x * kWaves)
    pair_grad<LA, LB>(b, g, __builtin_amdgcn_readfirstlane(list[k]), Dh, Ws, lds ? sgrad : nullptr);
  __syncthreads();
  if (lds)
    for (int t = threadIdx.x; t < 3 * g.natm; t += 64 * kWaves) {
      const double v = sgrad[t];
      if (v != 0.0) atomicAdd(&g.grad[t], v);
    }
}

// Workgroups of the gradient kernels: enough to fill the chip, few enough
// that their flushes (3 natm global atomics each) stay cheap.
constexpr int kGradGroups = 1024;

template <int LA, int LB>
hipError_t launch_pair(const DevBasis& b, const Int1eArgs& g, double* S, double* T, double* V, hipStream_t s) {
  const int c = LA * (LA + 1) / 2 + LB, n = g.cls_off[c + 1] - g.cls_off[c];
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL((k_int1e<LA, LB>), dim3((n + kWaves - 1) / kWaves, kSplit<LA, LB>), dim3(64 * kWaves), 0, s, b, g,
                     g.cls_sp + g.cls_off[c], n, S, T, V);
  return hipGetLastError();
}

template <int LA, int LB>
hipError_t launch_pair_grad(const DevBasis& b, const Int1eArgs& g, const double* Dh, const double* Ws, hipStream_t s) {
  const int c = LA * (LA + 1) / 2 + LB, n = g.cls_off[c + 1] - g.cls_off[c];
  if (n <= 0) return hipSuccess;
  const int grid = (n + kWaves - 1) / kWaves;
  hipLaunchKernelGGL((k_int1e_grad<LA, LB>), dim3(grid < kGradGroups ? grid : kGradGroups), dim3(64 * kWaves), 0, s, b,
                     g, g.cls_sp + g.cls_off[c], n, Dh, Ws);
  return hipGetLastError();
}

// log2 of the lanes a group gives to the nuclei
int group_of(int natm) {
  int lg = 0;
  while (lg < 6 && (1 << lg) < natm) ++lg;
  return lg;
}

}  // namespace

#define ASUKA_INT1E_CLASSES(X) X(0, 0) X(1, 0) X(1, 1) X(2, 0) X(2, 1) X(2, 2) X(3, 0) X(3, 1) X(3, 2) X(3, 3)

hipError_t launch_int1e(const DevBasis& b, Int1eArgs g, double* S, double* T, double* V, hipStream_t s) {
  g.lg_group = group_of(g.natm);
#define ASUKA_INT1E_RUN(la, lb) \
  if (hipError_t e = launch_pair<la, lb>(b, g, S, T, V, s)) return e;
  ASUKA_INT1E_CLASSES(ASUKA_INT1E_RUN)
#undef ASUKA_INT1E_RUN
  return hipSuccess;
}

hipError_t launch_int1e_grad(const DevBasis& b, Int1eArgs g, const double* Dh, const double* Ws, hipStream_t s) {
  g.lg_group = group_of(g.natm);
#define ASUKA_INT1E_RUN(la, lb) \
  if (hipError_t e = launch_pair_grad<la, lb>(b, g, Dh, Ws, s)) return e;
  ASUKA_INT1E_CLASSES(ASUKA_INT1E_RUN)
#undef ASUKA_INT1E_RUN
  return hipSuccess;
}
