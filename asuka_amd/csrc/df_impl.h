// Three- and two-centre Coulomb integrals (ab|P) and (P|Q): one lane per
// auxiliary shell, one wavefront per bra shell pair and 64 auxiliary shells of
// one angular momentum.
//
// The auxiliary shell is the ket pair (P, 1) with 1 an s function of exponent 0
// on P's centre, so the ket has l_d = 0, Q = C and no ket transfer; for the
// metric the bra is such a pair too. The bra pair is uniform across the wave:
// its primitive pairs are read with scalar loads, and an uncontracted
// auxiliary set keeps every lane on the same primitive loop. Per primitive
// triple and Rys root the 2-D tables G[i][k], i <= la + lb, k <= lc are built
// in registers and contracted to (e|c), e in cart(la..la+lb), as in the J/K
// register kernels (jk_fast_impl.h, whose index tables these are); the bra
// transfer to (ab|c) goes straight into the stores. Chunks of the auxiliary
// components (gridDim.z) keep at most about 75 intermediates a lane.
//
// What bounds it is FP64 arithmetic for the contracted pairs and, for X, the
// stores: the 64 lanes write 64 matrices, so each store is a line of its own
// until the caches merge it with its neighbours' of other pairs. The root
// tables of up to kLdsRootsMax roots are copied to LDS, once for the many bra
// pairs a workgroup takes. Measured at (H2O)6 cc-pVDZ (150 AOs, 1374 auxiliary
// functions), metric and X together: 15.5 ms with the run-time-class kernel
// (one wavefront a quartet, LDS tables, 440 B of scratch a lane), 1.04 ms with
// these on one stream, 0.65 ms over four streams and with the primitive pairs
// of one-centre bra pairs merged.
#pragma once
#include "jk_fast_impl.h"

namespace asuka_df {

using asuka_fast::binom_;
using asuka_fast::cx_;
using asuka_fast::cy_;
using asuka_fast::nc_;

constexpr int kWaves = 4;

// Bra shell pairs of one class, auxiliary shells of one l, and where element
// (a, b, P) goes: out[a sa + b sb + P sc], and [b sa + a sb + P sc] too for
// pairs of different shells (mirror).
struct DfWork {
  const int* bra;   // shell pairs
  int nbra;
  const int* aux;   // ket pairs (auxiliary shell, unit)
  int naux;
  double* out;
  long long sa, sb, sc;
  int mirror;
};

template <class PL, int CH>
__device__ __forceinline__ void df_item(const DevBasis& b, const DfWork& w, int sp, int ket, bool active,
                                        const double* __restrict__ tab) {
  using CK = asuka_fast::Chunk<PL, CH>;
  constexpr int LA = PL::la, LB = PL::lb, LC = PL::lc, NB = PL::NB, NA = PL::NA;
  constexpr int NMAX = LA + LB, NR = PL::NR, NE = PL::NE;
  constexpr int c0 = CK::c0, NCL = CK::c1 - CK::c0;
  constexpr auto te = PL::RE::tab();
  const int A = asuka_fast::uni(b.sp_A[sp]), B = asuka_fast::uni(b.sp_B[sp]);
  const int C = b.sp_A[ket];
  double cA[3], AB[3], cC[3];
#pragma unroll
  for (int x = 0; x < 3; ++x) {
    cA[x] = b.shell_xyz[3 * A + x];
    AB[x] = cA[x] - b.shell_xyz[3 * B + x];
    cC[x] = b.shell_xyz[3 * C + x];
  }
  const int ab0 = asuka_fast::uni(b.pp_start[sp]), nab = asuka_fast::uni(b.pp_count[sp]);
  const int cd0 = b.pp_start[ket], ncd = active ? b.pp_count[ket] : 0;
  double ef[NE * NCL];
#pragma unroll
  for (int i = 0; i < NE * NCL; ++i) ef[i] = 0.0;
  for (int j = 0; j < ncd; ++j) {
    const PrimPair Y = b.pp[cd0 + j];
    const double q = Y.eta, iq = Y.inv_eta, ckq = 34.98683665524972497 * Y.cK * Y.inv_eta;  // 2 pi^(5/2)
    for (int i = 0; i < nab; ++i) {
      const PrimPair X = b.pp[ab0 + i];  // wave-uniform
      const double p = X.eta, ip = X.inv_eta, spq = p + q, inv_pq = rcp_nr(spq);
      const double d[3] = {X.Px - cC[0], X.Py - cC[1], X.Pz - cC[2]};
      const double base = X.cK * ip * ckq * rsq_nr(spq);
      double rx[NR], rw[NR];
      rys_roots_blk<NR, double, (NR <= kLdsRootsMax ? rys_c::lds_stride(NR, 8) : rys_c::interval_size(NR))>(
          p * q * inv_pq * (d[0] * d[0] + d[1] * d[1] + d[2] * d[2]), tab, rx, rw);
      const double PA[3] = {X.Px - cA[0], X.Py - cA[1], X.Pz - cA[2]};
#pragma unroll
      for (int u = 0; u < NR; ++u) {
        const double x = rx[u], B0 = 0.5 * x * inv_pq;
        const double B1 = 0.5 * (1.0 - x) * ip + B0, B1p = 0.5 * (1.0 - x) * iq + B0;
        const double xq = q * inv_pq * x, xp = p * inv_pq * x;
        double G[3][NMAX + 1][LC + 1];
#pragma unroll
        for (int ax = 0; ax < 3; ++ax) {
          const double Cc = PA[ax] - xq * d[ax], Cp = xp * d[ax];
          G[ax][0][0] = ax == 2 ? rw[u] * base : 1.0;
          if (NMAX > 0) G[ax][NMAX > 0 ? 1 : 0][0] = NMAX > 0 ? Cc * G[ax][0][0] : G[ax][0][0];
#pragma unroll
          for (int a = 2; a <= NMAX; ++a) G[ax][a][0] = B1 * (a - 1) * G[ax][a - 2][0] + Cc * G[ax][a - 1][0];
          if (LC > 0) {
#pragma unroll
            for (int a = 0; a <= NMAX; ++a) {
              G[ax][a][LC > 0 ? 1 : 0] = Cp * G[ax][a][0] + (a > 0 ? a * B0 * G[ax][a > 0 ? a - 1 : 0][0] : 0.0);
#pragma unroll
              for (int c = 2; c <= LC; ++c)
                G[ax][a][c] = B1p * (c - 1) * G[ax][a][c - 2] + Cp * G[ax][a][c - 1] +
                              (a > 0 ? a * B0 * G[ax][a > 0 ? a - 1 : 0][c - 1] : 0.0);
            }
          }
        }
#pragma unroll
        for (int ie = 0; ie < NE; ++ie)
#pragma unroll
          for (int ic = 0; ic < NCL; ++ic) {
            const int fx = cx_(LC, c0 + ic), fy = cy_(LC, c0 + ic), fz = LC - fx - fy;
            ef[ie * NCL + ic] = fma(G[0][te.x[ie]][fx] * G[1][te.y[ie]][fy], G[2][te.z[ie]][fz], ef[ie * NCL + ic]);
          }
      }
    }
  }
  if (!active) return;  // no cross-lane operations below
  double pab[3][LB + 1];
#pragma unroll
  for (int ax = 0; ax < 3; ++ax) {
    pab[ax][0] = 1.0;
#pragma unroll
    for (int e = 1; e <= LB; ++e) pab[ax][e] = pab[ax][e - 1] * AB[ax];
  }
  const int aoA = b.shell_ao[A], aoB = b.shell_ao[B];
  double* out = w.out + (long long)(b.shell_ao[C] + c0) * w.sc;
  const bool mirror = w.mirror && A != B;  // uniform
#pragma unroll
  for (int ia = 0; ia < NA; ++ia)
#pragma unroll
    for (int ib = 0; ib < NB; ++ib) {
      const int ax = cx_(LA, ia), ay = cy_(LA, ia), az = LA - ax - ay;
      const int bx = cx_(LB, ib), by = cy_(LB, ib), bz = LB - bx - by;
      const long long o1 = (aoA + ia) * w.sa + (aoB + ib) * w.sb, o2 = (aoB + ib) * w.sa + (aoA + ia) * w.sb;
#pragma unroll
      for (int ic = 0; ic < NCL; ++ic) {
        double s = 0.0;
#pragma unroll
        for (int nx = 0; nx <= bx; ++nx)
#pragma unroll
          for (int ny = 0; ny <= by; ++ny)
#pragma unroll
            for (int nz = 0; nz <= bz; ++nz)
              s = fma(binom_(bx, nx) * binom_(by, ny) * binom_(bz, nz) * pab[0][bx - nx] * pab[1][by - ny] *
                          pab[2][bz - nz],
                      ef[PL::RE::index(ax + nx, ay + ny, az + nz) * NCL + ic], s);
        out[ic * w.sc + o1] = s;
        if (mirror) out[ic * w.sc + o2] = s;
      }
    }
}

template <class PL, int CH>
__device__ __forceinline__ void df_dispatch(int ch, const DevBasis& b, const DfWork& w, int sp, int ket, bool active,
                                            const double* __restrict__ tab) {
  if constexpr (CH < PL::SPLIT_C) {
    if (ch == CH)
      df_item<PL, CH>(b, w, sp, ket, active, tab);
    else
      df_dispatch<PL, CH + 1>(ch, b, w, sp, ket, active, tab);
  }
}

template <class PL>
__global__ __launch_bounds__(64 * kWaves) void k_df(const DevBasis b, const DfWork w) {
  constexpr int NR = PL::NR;
  constexpr bool kLds = NR <= kLdsRootsMax;
  constexpr int NFI = rys_c::interval_size(NR), S64 = rys_c::lds_stride(NR, 8);
  __shared__ double t64[kLds ? rys_c::nint[NR] * S64 : 1];
  const double* gtab = rys_dev::rys_coef + rys_c::coef_off[NR];
  if constexpr (kLds) {
    for (int t = threadIdx.x; t < rys_c::block_size(NR); t += 64 * kWaves) t64[(t / NFI) * S64 + t % NFI] = gtab[t];
    __syncthreads();
  }
  const int wave = asuka_fast::uni((int)(threadIdx.x >> 6));
  const int k = blockIdx.y * 64 + (threadIdx.x & 63);
  const bool active = k < w.naux;
  const int ket = w.aux[active ? k : 0];
  for (int p = blockIdx.x * kWaves + wave; p < w.nbra; p += gridDim.x * kWaves)
    df_dispatch<PL, 0>(blockIdx.z, b, w, asuka_fast::uni(w.bra[p]), ket, active, kLds ? t64 : gtab);
}

// Workgroups of a launch: about eight a CU, each taking several bra pairs.
constexpr int kGroups = 2048;

template <class PL>
hipError_t launch_df(const DevBasis& b, const DfWork& w, hipStream_t s) {
  const int gy = (w.naux + 63) / 64, gz = PL::SPLIT_C;
  int gx = (w.nbra + kWaves - 1) / kWaves;
  const int most = kGroups / (gy * gz);
  if (gx > most) gx = most > 0 ? most : 1;
  hipLaunchKernelGGL((k_df<PL>), dim3(gx, gy, gz), dim3(64 * kWaves), 0, s, b, w);
  return hipGetLastError();
}

using DfLauncher = hipError_t (*)(const DevBasis&, const DfWork&, hipStream_t);

}  // namespace asuka_df

// Each df_p*.hip translation unit instantiates a subset of the classes
// (la lb|lc): (la, lb, lc, chunks of the auxiliary components).
#define ASUKA_DF_FIND(FN, LIST)                               \
  asuka_df::DfLauncher FN(int la, int lb, int lc) {          \
    using namespace asuka_df;                                \
    LIST(ASUKA_DF_CASE)                                      \
    return nullptr;                                          \
  }
#define ASUKA_DF_CASE(a, b_, c, sc) \
  if (la == a && lb == b_ && lc == c) return &launch_df<asuka_fast::Plan<a, b_, c, 0, 1, sc>>;
