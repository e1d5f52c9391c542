// Class-specialised register kernels: one lane per shell quartet.
//
// For a class (la lb|lc ld) every lane loops over the primitive quartets of its
// shell quartet and, per Rys root, builds the 2-D tables
//   G_x[i][k], i <= la+lb, k <= lc+ld   (VRR, weight*prefactor folded into z)
// and accumulates the contracted intermediates
//   (e|f) = sum_prim sum_root G_x[ex][fx] G_y[ey][fy] G_z[ez][fz]
// for e in cart(la..la+lb), f in cart(lc..lc+ld), all in registers. The
// horizontal transfer to (ab|cd) runs once per shell quartet after the
// primitive loop (its coefficients depend only on A-B and C-D):
//   (e|cd) = sum_m prod_i C(d_i,m_i) CD_i^(d_i-m_i) (e|c+m)
//   (ab|cd) = sum_n prod_i C(b_i,n_i) AB_i^(b_i-n_i) (a+n|cd)
// The tile then feeds the J/K (or Fock) digestion of the reference's ordered
// contraction (cueri_cuda_kernels_dense_scatter.cu:246-352) with block sums
// per quartet: nAB + nCD J updates and up to 4 K blocks, instead of one atomic
// per tile element and term. Symmetric pair updates are folded into one (the
// outputs are symmetrised afterwards).
//
// All component indices are compile-time (constexpr tables + full unrolling),
// so the tables and accumulators live in VGPRs.
#pragma once
#include <type_traits>

#include "jk_internal.h"
#include "rys_eval.h"

namespace asuka_fast {

constexpr int nc_(int l) { return (l + 1) * (l + 2) / 2; }

// components of l in lx-descending, ly-descending order
constexpr int cx_(int l, int i) {
  int idx = 0;
  for (int x = l; x >= 0; --x)
    for (int y = l - x; y >= 0; --y) {
      if (idx == i) return x;
      ++idx;
    }
  return 0;
}
constexpr int cy_(int l, int i) {
  int idx = 0;
  for (int x = l; x >= 0; --x)
    for (int y = l - x; y >= 0; --y) {
      if (idx == i) return y;
      ++idx;
    }
  return 0;
}
constexpr int cidx_(int lx, int ly, int lz) {
  const int l = lx + ly + lz;
  return (l - lx) * (l - lx + 1) / 2 + lz;
}
constexpr int binom_(int n, int k) {
  int r = 1;
  for (int i = 1; i <= k; ++i) r = r * (n - k + i) / i;
  return r;
}

// Concatenated Cartesian range l in [lo, hi]: index -> exponents and back.
template <int LO, int HI>
struct Range {
  static constexpr int size() {
    int s = 0;
    for (int l = LO; l <= HI; ++l) s += nc_(l);
    return s;
  }
  static constexpr int off(int l) {
    int s = 0;
    for (int k = LO; k < l; ++k) s += nc_(k);
    return s;
  }
  struct Tab {
    int x[size()], y[size()], z[size()];
  };
  static constexpr Tab tab() {
    Tab t{};
    int i = 0;
    for (int l = LO; l <= HI; ++l)
      for (int c = 0; c < nc_(l); ++c) {
        t.x[i] = cx_(l, c);
        t.y[i] = cy_(l, c);
        t.z[i] = l - t.x[i] - t.y[i];
        ++i;
      }
    return t;
  }
  static constexpr int index(int x, int y, int z) { return off(x + y + z) + cidx_(x, y, z); }
};

template <typename CT>
__device__ __forceinline__ CT pw(const CT* p, int k) {
  return p[k];
}

// Plans split over A components whose wave items carry the J[c,d] sums
// across their A chunks (run_citem). Chosen by measurement at (H2O)8
// cc-pVTZ: for the other split plans the longer items (fewer per row task)
// and the extra live registers cost more than the atomics they save.
constexpr bool carry_jcd(int la, int lb, int lc, int ld) {
  const int k = ((la * 4 + lb) * 4 + lc) * 4 + ld;
  constexpr int on[] = {((2 * 4 + 1) * 4 + 1) * 4 + 1, ((2 * 4 + 1) * 4 + 2) * 4 + 1,
                        ((2 * 4 + 2) * 4 + 1) * 4 + 1, ((2 * 4 + 2) * 4 + 2) * 4 + 0,
                        ((3 * 4 + 0) * 4 + 2) * 4 + 1, ((3 * 4 + 0) * 4 + 2) * 4 + 2,
                        ((3 * 4 + 1) * 4 + 2) * 4 + 0, ((3 * 4 + 1) * 4 + 2) * 4 + 1,
                        ((3 * 4 + 2) * 4 + 2) * 4 + 0, ((3 * 4 + 3) * 4 + 1) * 4 + 0};
  for (int x : on)
    if (x == k) return true;
  return false;
}

template <int LA, int LB, int LC, int LD, int SA, int SC>
struct Plan {
  static constexpr int la = LA, lb = LB, lc = LC, ld = LD;
  static constexpr int NA = nc_(LA), NB = nc_(LB), NC = nc_(LC), ND = nc_(LD);
  static constexpr int NMAX = LA + LB, MMAX = LC + LD;
  static constexpr int NR = (LA + LB + LC + LD) / 2 + 1;
  static constexpr int SPLIT_A = SA, SPLIT_C = SC, NCH = SA * SC;
  static constexpr bool CARRY = SA > 1 && carry_jcd(LA, LB, LC, LD);
  using RE = Range<LA, LA + LB>;
  using RF = Range<LC, LC + LD>;
  static constexpr int NE = RE::size(), NF = RF::size();
};

// The chunk CH of a plan covers A-components [a0, a1) and C-components
// [c0, c1); it needs the intermediates (e|f) for e = a + n (|n| <= lb) and
// f = c + m (|m| <= ld) only.
template <class PL, int CH>
struct Chunk {
  static constexpr int ca = CH / PL::SPLIT_C, cc = CH % PL::SPLIT_C;
  static constexpr int a0 = ca * PL::NA / PL::SPLIT_A, a1 = (ca + 1) * PL::NA / PL::SPLIT_A;
  static constexpr int c0 = cc * PL::NC / PL::SPLIT_C, c1 = (cc + 1) * PL::NC / PL::SPLIT_C;
  struct Lists {
    int e[PL::NE];
    int emap[PL::NE];
    int ne;
    int f[PL::NF];
    int fmap[PL::NF];
    int nf;
  };
  static constexpr Lists lists() {
    Lists L{};
    bool ue[PL::NE] = {}, uf[PL::NF] = {};
    for (int a = a0; a < a1; ++a) {
      const int x = cx_(PL::la, a), y = cy_(PL::la, a), z = PL::la - x - y;
      for (int nx = 0; nx <= PL::lb; ++nx)
        for (int ny = 0; ny + nx <= PL::lb; ++ny)
          for (int nz = 0; nz + ny + nx <= PL::lb; ++nz) ue[PL::RE::index(x + nx, y + ny, z + nz)] = true;
    }
    for (int c = c0; c < c1; ++c) {
      const int x = cx_(PL::lc, c), y = cy_(PL::lc, c), z = PL::lc - x - y;
      for (int mx = 0; mx <= PL::ld; ++mx)
        for (int my = 0; my + mx <= PL::ld; ++my)
          for (int mz = 0; mz + my + mx <= PL::ld; ++mz) uf[PL::RF::index(x + mx, y + my, z + mz)] = true;
    }
    L.ne = 0;
    for (int i = 0; i < PL::NE; ++i) {
      L.emap[i] = -1;
      if (ue[i]) {
        L.e[L.ne] = i;
        L.emap[i] = L.ne++;
      }
    }
    L.nf = 0;
    for (int i = 0; i < PL::NF; ++i) {
      L.fmap[i] = -1;
      if (uf[i]) {
        L.f[L.nf] = i;
        L.fmap[i] = L.nf++;
      }
    }
    return L;
  }
  static constexpr Lists L = lists();
  static constexpr int NEL = L.ne, NFL = L.nf;
};

// Wave votes through the ballot intrinsic, whose result the compiler knows to
// be wave-uniform (branches on it stay scalar).
__device__ __forceinline__ bool wave_any(bool v) { return __builtin_amdgcn_ballot_w64(v) != 0ull; }

// A value known to be the same on every lane, moved to a scalar register.
__device__ __forceinline__ int uni(int v) { return __builtin_amdgcn_readfirstlane(v); }

// Sum over the 64 lanes of the wavefront (all lanes must be converged).
__device__ __forceinline__ double wave_sum(double v) { return wave_total(v); }


// Everything the kernels below read is passed in one struct by value and
// fetched from the kernel-argument segment where it is used (ArgP), not held
// in scalar registers: with three argument structs and their pointers live
// across the item loop the compiler spilled about 160 scalar registers to
// lanes of vector registers and moved them back all over an item ((10|10)
// FP64: 164 spills, 3504 instructions, 137 VGPRs; now 24, 1838 and 109).
// refetch() hides the pointer's origin so that loads through it are not
// hoisted over it. Measured, with the bra's rows as uniform bases, the next bra
// primitive pair in flight and the counting code in a kernel of its own:
// (H2O)27 cc-pVDZ FP64 Fock build 62.9 -> 55.5 ms, (H2O)64 mixed 331 -> 299 ms,
// batch of 14 clusters 30.4 -> 25.4 ms, (H2O)8 cc-pVTZ mixed 56.7 -> 52.8 ms.
// One density of a build: where it is read and what it is digested into
// (null: not wanted). D, J and K of MODE_FOCK builds: J = K = F.
struct FastDen {
  const double* D;
  double* J;
  double* K;
  const double* Dpos;  // EriOut::jblk
  double* Jpos;
  double* Kc;
};
struct FastArgs {
  const WaveUnit* units;
  const RowTask* tasks;
  unsigned int* queue;
  const void* pp;       // bra primitive pairs: PrimPairF, or PrimPairF32 for the FP32 kernels
  const double* kpd;    // ket primitive pairs (DevBasis::kpoff) of this precision
  const float* kpf;
  const long long* kpoff;
  const int *sp_A, *sp_B, *pp_start, *pp_count, *shell_ao, *shell_mol, *mol_n, *mol_lao, *lao_ao, *pos_of_sp;
  const long long *mol_shift, *jblk;
  const double *shell_xyz, *Q, *Dsp, *kq, *kd, *kcd;
  const int2 *kpp, *kao, *klao;
  FastDen den[2];
  double eps_density, eps_prim;
  double ks;  // factor of the K sums: 1, or -1/2 for MODE_FOCK
  int nden, ntasks, wpg;
  int acc_colsC, acc_colsD, lao_offC, lao_offD;
};
#define ASUKA_CONST __attribute__((address_space(4)))
#define ASUKA_GLOB __attribute__((address_space(1)))
using ArgP = const ASUKA_CONST FastArgs*;
__device__ __forceinline__ ArgP refetch(ArgP p) {
  asm volatile("" : "+s"(p));
  return p;
}
// Read-only tables at wave-uniform indices: scalar loads.
template <typename T>
__device__ __forceinline__ T cl(const T* p, long long i) {
  return ((const ASUKA_CONST T*)p)[i];
}
// A wave-uniform base and a 32-bit byte offset per lane.
template <typename T>
__device__ __forceinline__ T gl(const void* base, unsigned off) {
  return *(const ASUKA_GLOB T*)((const ASUKA_GLOB char*)base + off);
}
typedef int i32x2 __attribute__((ext_vector_type(2)));
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));

// A primitive pair in the arithmetic CT of the recursion; P stays FP64 so that
// P - Q is formed in FP64.
template <typename CT>
struct Prim {
  double Px, Py, Pz;
  CT eta, ieta, ck, ax, ay, az, q;
};
template <typename CT>
__device__ __forceinline__ Prim<CT> load_bra(const void* pp, int i) {  // i uniform
  Prim<CT> r;
  if constexpr (sizeof(CT) == 8) {
    const ASUKA_CONST double* d = (const ASUKA_CONST double*)pp + (sizeof(PrimPairF) / 8) * (long long)i;
    r.eta = d[0], r.ieta = d[1], r.ck = d[2], r.Px = d[3], r.Py = d[4], r.Pz = d[5];
    r.ax = d[6], r.ay = d[7], r.az = d[8];
  } else {
    const ASUKA_CONST double* d = (const ASUKA_CONST double*)pp + (sizeof(PrimPairF32) / 8) * (long long)i;
    const ASUKA_CONST float* f = (const ASUKA_CONST float*)(d + 3);
    r.Px = d[0], r.Py = d[1], r.Pz = d[2];
    r.eta = f[0], r.ieta = f[1], r.ck = f[2], r.ax = f[3], r.ay = f[4], r.az = f[5];
  }
  r.q = CT(0);
  return r;
}
// The lane's primitive pair of slot row s of the ket tables (DevBasis::kpoff):
// one scalar base, the fields at immediate offsets.
template <typename CT>
__device__ __forceinline__ Prim<CT> load_ket(const double* kpd, const float* kpf, long long s, unsigned lane) {
  Prim<CT> r;
  if constexpr (sizeof(CT) == 8) {
    const double* k = kpd + s * (64 * kKet64);
    r.eta = gl<double>(k, 8 * lane), r.ieta = gl<double>(k, 8 * lane + 512), r.ck = gl<double>(k, 8 * lane + 1024);
    r.Px = gl<double>(k, 8 * lane + 1536), r.Py = gl<double>(k, 8 * lane + 2048), r.Pz = gl<double>(k, 8 * lane + 2560);
    r.ax = gl<double>(k, 8 * lane + 3072), r.ay = gl<double>(k, 8 * lane + 3584);
    r.az = gl<double>(k + 512, 8 * lane), r.q = gl<double>(k + 512, 8 * lane + 512);
  } else {
    const double* k = kpd + s * (64 * kKet32d);
    const float* f = kpf + s * (64 * kKet32f);
    r.Px = gl<double>(k, 8 * lane), r.Py = gl<double>(k, 8 * lane + 512), r.Pz = gl<double>(k, 8 * lane + 1024);
    r.eta = gl<float>(f, 4 * lane), r.ieta = gl<float>(f, 4 * lane + 256), r.ck = gl<float>(f, 4 * lane + 512);
    r.ax = gl<float>(f, 4 * lane + 768), r.ay = gl<float>(f, 4 * lane + 1024), r.az = gl<float>(f, 4 * lane + 1280);
    r.q = gl<float>(f, 4 * lane + 1536);
  }
  return r;
}

// The bra pair of a row task (uniform).
struct Bra {
  int P, ab0;      // shell pair, its first primitive pair
  int A, B;        // shells
  int aoA, aoB;    // first AOs
  int posP;        // the pair's own ket position, -1 if it has none
  int N;           // row stride of the molecule's D/J/K block
  long long msh;   // element offset of that block (mol_layout)
};

// Arithmetic helpers for the compute type CT of the recursion (double, or
// float on the FP32 path).
__device__ __forceinline__ double fmac(double a, double b, double c) { return fma(a, b, c); }
__device__ __forceinline__ float fmac(float a, float b, float c) { return __builtin_fmaf(a, b, c); }

// Workgroups of up to 8 wavefronts share the root tables and the row
// accumulators; the host picks 4 or 8 per class pair (ClassWork::wpg): 8 when
// the accumulators are large (more waves per LDS byte), else 4 (less idle
// time at the end of short row tasks).
constexpr int kMaxWavesPerGroup = 8;
constexpr int kGroupThreads = 64 * kMaxWavesPerGroup;

// Workgroup accumulators of one row task (one bra pair P), in the dynamic
// LDS array s_acc: the J[a,b] block and the K rows of the bra's AOs, K[a, :]
// and K[b, :], over the columns of the ket class (AOs of angular momentum lc,
// then ld, in the compact per-l numbering). Offsets are in doubles; on ==
// false selects direct global atomics.
extern __shared__ double s_acc[];
struct RowAcc {
  bool on;
  int jab;  // [NA * NB]
  int kac;  // [NA * colsC]
  int kad;  // [NA * colsD] (same as kac when lc == ld)
  int kbc;  // [NB * colsC]
  int kbd;  // [NB * colsD] (same as kbc when lc == ld)
  int colsC, colsD;
  int stride;  // offset of the second density's accumulators (two-density builds)
};

// One chunk of one shell quartet per lane; the bra pair is the same on every
// lane of the wave (bra-uniform wave units), so the bra primitive pairs are
// read with scalar loads in the inner loop while each lane streams its own
// ket primitive pairs in the outer loop. CT is the type of the primitive
// setup, roots, VRR, contracted intermediates and HRR; the digestion always
// accumulates in FP64. Geometric differences are formed in FP64 and rounded.
// `tab` is the NR-root block of the root table in CT (LDS or global).
// col: the unit's first ket position (uniform; a 64-position block boundary).
// jcd: with the plan split over A components, the J[c,d] partial sums of the
// first density over this chunk's A components are added into jcd (the
// lane's registers, NCL*ND values) and the caller issues one atomic per
// element after the last A chunk; nullptr: atomics here.
template <class PL, int CH, typename CT, bool FX>
__device__ __forceinline__ void run_chunk(ArgP ap, const Bra& br, int col, const UnitRange& ur, bool active,
                                          const CT* __restrict__ tab, const RowAcc& acc, double* jcd) {
  using CK = Chunk<PL, CH>;
  constexpr int NEL = CK::NEL, NFL = CK::NFL, NR = PL::NR;
  constexpr int NMAX = PL::NMAX, MMAX = PL::MMAX;
  constexpr int LA = PL::la, LB = PL::lb, LC = PL::lc, LD = PL::ld;
  constexpr int NB = PL::NB, ND = PL::ND;
  constexpr int a0 = CK::a0, a1 = CK::a1, c0 = CK::c0, c1 = CK::c1;
  constexpr int NAL = a1 - a0, NCL = c1 - c0;
  constexpr int NCDL = NCL * ND;
  constexpr auto te = PL::RE::tab();
  constexpr auto tf = PL::RF::tab();
  constexpr auto L = CK::L;
  const CT one = CT(1), half = CT(0.5);
  const unsigned lane = threadIdx.x & 63;

  ap = refetch(ap);
  const int ab0 = br.ab0 + ur.i0, nab = ur.ni;  // the unit's bra primitive pairs
  const int ncd = active ? min(gl<int>(ap->kpp + col, 8 * lane + 4), ur.j1) : 0;

  CT ef[NEL * NFL];
#pragma unroll
  for (int i = 0; i < NEL * NFL; ++i) ef[i] = CT(0);

  // Primitive-quartet screening: the primitive pairs of a shell pair are
  // sorted by their Schwarz bound q (largest first). nab (uniform, from the
  // wave unit) already leaves out the bra pairs whose q times the largest
  // ket-pair bound of the unit is below eps_prim; a lane leaves its ket loop
  // at the first ket pair whose q times the largest bra bound is below it (the
  // shell pair's largest, also in a slice that starts further down, so that a
  // slice leaves out no more than the uncut unit does).
  // Every skipped primitive quartet adds less than eps_prim to each integral.
  if (nab > 0) {
    const void* pp = ap->pp;
    const double* kpd = ap->kpd;
    const float* kpf = ap->kpf;
    CT kcut;
    if constexpr (sizeof(CT) == 8)
      kcut = ap->eps_prim * rcp_nr(((const ASUKA_CONST PrimPairF*)pp)[br.ab0].q);
    else
      kcut = CT(ap->eps_prim * rcp_nr((double)((const ASUKA_CONST PrimPairF32*)pp)[br.ab0].q));
    // slot rows of the unit's block: the lanes' j-th primitive pairs
    const long long ks0 = cl(ap->kpoff, col >> 6);
    Prim<CT> Yn;
    if (ur.j0 < ncd) Yn = load_ket<CT>(kpd, kpf, ks0 + ur.j0, lane);
    Prim<CT> X = load_bra<CT>(pp, ab0);
    for (int j = ur.j0; j < ncd; ++j) {
      const Prim<CT> Y = Yn;
      if (Y.q < kcut) break;  // per lane: the rest of its ket pairs are smaller
      if (j + 1 < ncd) Yn = load_ket<CT>(kpd, kpf, ks0 + uni(j + 1), lane);  // next ket pair, in flight during this one
      const CT q = Y.eta, iq = Y.ieta, ckq = Y.ck;
      const CT QCx = Y.ax, QCy = Y.ay, QCz = Y.az;
      for (int i = 0; i < nab; ++i) {
        // the next bra pair (wave-uniform; the first again for the next ket pair) is in flight during this one
        const Prim<CT> Xn = load_bra<CT>(pp, ab0 + (i + 1 < nab ? i + 1 : 0));
      const CT p = X.eta, ip = X.ieta;
      const CT PAx = X.ax, PAy = X.ay, PAz = X.az;
      const CT spq = p + q;
      const CT inv_pq = rcp_nr(spq);
      const CT dx = CT(X.Px - Y.Px), dy = CT(X.Py - Y.Py), dz = CT(X.Pz - Y.Pz);
      const CT T = p * q * inv_pq * (dx * dx + dy * dy + dz * dz);
      // 2 pi^(5/2) cK_ab cK_cd / (p q sqrt(p+q))
      const CT base = X.ck * ckq * rsq_nr(spq);
      CT rx[NR], rw[NR];
      rys_roots_blk<NR, CT, (NR <= kLdsRootsMax ? rys_c::lds_stride_of<CT>(NR) : rys_c::interval_size_of<CT>(NR))>(
          T, tab, rx, rw);
      const CT qf = q * inv_pq, pf = p * inv_pq;
#pragma unroll
      for (int u = 0; u < NR; ++u) {
        const CT x = rx[u];
        const CT B0 = half * x * inv_pq;
        const CT B1 = half * (one - x) * ip + B0;
        const CT B1p = half * (one - x) * iq + B0;
        const CT xq = qf * x, xp = pf * x;
        CT G[3][NMAX + 1][MMAX + 1];
        const CT c00[3] = {PAx - xq * dx, PAy - xq * dy, PAz - xq * dz};
        const CT c0p[3] = {QCx + xp * dx, QCy + xp * dy, QCz + xp * dz};
#pragma unroll
        for (int ax = 0; ax < 3; ++ax) {
          const CT g0 = (ax == 2) ? rw[u] * base : one;
          const CT Cc = c00[ax], Cp = c0p[ax];
          G[ax][0][0] = g0;
          if (NMAX > 0) G[ax][1][0] = Cc * g0;
#pragma unroll
          for (int a = 2; a <= NMAX; ++a) G[ax][a][0] = B1 * CT(a - 1) * G[ax][a - 2][0] + Cc * G[ax][a - 1][0];
          if (MMAX > 0) {
#pragma unroll
            for (int a = 0; a <= NMAX; ++a) {
              G[ax][a][1] = Cp * G[ax][a][0] + (a > 0 ? CT(a) * B0 * G[ax][a > 0 ? a - 1 : 0][0] : CT(0));
#pragma unroll
              for (int c = 2; c <= MMAX; ++c)
                G[ax][a][c] = B1p * CT(c - 1) * G[ax][a][c - 2] + Cp * G[ax][a][c - 1] +
                              (a > 0 ? CT(a) * B0 * G[ax][a > 0 ? a - 1 : 0][c - 1] : CT(0));
            }
          }
        }
#pragma unroll
        for (int ie = 0; ie < NEL; ++ie) {
#pragma unroll
          for (int jf = 0; jf < NFL; ++jf) {
            const int eg = L.e[ie], fg = L.f[jf];
            const CT gxy = G[0][te.x[eg]][tf.x[fg]] * G[1][te.y[eg]][tf.y[fg]];
            ef[ie * NFL + jf] = fmac(gxy, G[2][te.z[eg]][tf.z[fg]], ef[ie * NFL + jf]);
          }
        }
      }
        X = Xn;
      }
    }
  }

  // ---- horizontal transfer: ket (C-components of the chunk) then bra ----
  ap = refetch(ap);
  CT pab[3][LB + 1], pcd[3][LD + 1];
  {
    CT ab[3], cd[3];
#pragma unroll
    for (int ax = 0; ax < 3; ++ax) {
      ab[ax] = LB > 0 ? CT(cl(ap->shell_xyz, 3 * br.A + ax) - cl(ap->shell_xyz, 3 * br.B + ax)) : CT(0);
      cd[ax] = LD > 0 ? CT(gl<double>(ap->kcd + 3 * (long long)col, 24 * lane + 8 * ax)) : CT(0);
    }
#pragma unroll
    for (int ax = 0; ax < 3; ++ax) {
      pab[ax][0] = one;
      pcd[ax][0] = one;
#pragma unroll
      for (int e = 1; e <= LB; ++e) pab[ax][e] = pab[ax][e - 1] * ab[ax];
#pragma unroll
      for (int e = 1; e <= LD; ++e) pcd[ax][e] = pcd[ax][e - 1] * cd[ax];
    }
  }
  CT ecd[NEL * NCDL];
#pragma unroll
  for (int ie = 0; ie < NEL; ++ie)
#pragma unroll
    for (int ic = 0; ic < NCL; ++ic)
#pragma unroll
      for (int id = 0; id < ND; ++id) {
        const int cxv = cx_(LC, c0 + ic), cyv = cy_(LC, c0 + ic), czv = LC - cxv - cyv;
        const int dxv = cx_(LD, id), dyv = cy_(LD, id), dzv = LD - dxv - dyv;
        CT s = CT(0);
#pragma unroll
        for (int mx = 0; mx <= dxv; ++mx)
#pragma unroll
          for (int my = 0; my <= dyv; ++my)
#pragma unroll
            for (int mz = 0; mz <= dzv; ++mz) {
              const CT coef = CT(binom_(dxv, mx) * binom_(dyv, my) * binom_(dzv, mz)) *
                                  pw(pcd[0], dxv - mx) * pw(pcd[1], dyv - my) * pw(pcd[2], dzv - mz);
              s = fmac(coef, ef[ie * NFL + L.fmap[PL::RF::index(cxv + mx, cyv + my, czv + mz)]], s);
            }
        ecd[ie * NCDL + ic * ND + id] = s;
      }
  CT tile[NAL * NB * NCDL];
#pragma unroll
  for (int ia = 0; ia < NAL; ++ia)
#pragma unroll
    for (int ib = 0; ib < NB; ++ib) {
      const int axv = cx_(LA, a0 + ia), ayv = cy_(LA, a0 + ia), azv = LA - axv - ayv;
      const int bxv = cx_(LB, ib), byv = cy_(LB, ib), bzv = LB - bxv - byv;
#pragma unroll
      for (int jc = 0; jc < NCDL; ++jc) {
        CT s = CT(0);
#pragma unroll
        for (int nx = 0; nx <= bxv; ++nx)
#pragma unroll
          for (int ny = 0; ny <= byv; ++ny)
#pragma unroll
            for (int nz = 0; nz <= bzv; ++nz) {
              const CT coef = CT(binom_(bxv, nx) * binom_(byv, ny) * binom_(bzv, nz)) *
                                  pw(pab[0], bxv - nx) * pw(pab[1], byv - ny) * pw(pab[2], bzv - nz);
              s = fmac(coef, ecd[L.emap[PL::RE::index(axv + nx, ayv + ny, azv + nz)] * NCDL + jc], s);
            }
        tile[(ia * NB + ib) * NCDL + jc] = s;
      }
    }

  // ---- digestion of the chunk's tile block (rows a0..a1 x all b, cols c0..c1 x all d) ----
  // Sums over the chunk's own components are complete; the rest are partial
  // and add up across chunks. J[a,b] and the K rows of a and b go to the
  // workgroup's LDS accumulators when present (flushed once per row task),
  // J[c,d] (distinct per lane) to global atomics. With a second density
  // (two-density builds) the same tile is digested again into (J2, K2).
  const int N = br.N;
  const i32x2 kao = gl<i32x2>(ap->kao + col, 8 * lane);
  const unsigned oC = 8u * (unsigned)(kao.x + c0), oD = 8u * (unsigned)kao.y;  // byte offsets of the lane's columns
  const bool ab_neq = br.A != br.B, cd_neq = kao.x != kao.y, bk = br.posP != col + (int)lane;
  const double fj = (ab_neq ? 2.0 : 1.0) * (cd_neq ? 2.0 : 1.0);
  const double ks = bk ? 2.0 * ap->ks : ap->ks;
  const bool lds = acc.on;  // uniform
  // compact columns of the lane's C (first component of the chunk) and D shells
  const i32x2 klao = gl<i32x2>(ap->klao + col, 8 * lane);
  const int colC = klao.x + c0, colD = klao.y;
  const int nden = ap->nden;  // uniform
  for (int di = 0; di < nden; ++di) {
    const ASUKA_CONST FastDen* dn = &ap->den[di];
    const double* Dm = dn->D + br.msh;
    double* Jo = dn->J;
    const int so = di * acc.stride;  // this density's accumulators in s_acc
    // rows of the bra's AOs (uniform bases)
    auto rowA = [&](int ia) { return Dm + (long long)(br.aoA + a0 + ia) * N; };
    auto rowB = [&](int ib) { return Dm + (long long)(br.aoB + ib) * N; };
    if (Jo) {
      const long long jb = cl(ap->jblk, col >> 6) + 64LL * (c0 * ND);  // the chunk's components of the unit's block
      {
        double dcd[NCDL];
        const double* Dp = dn->Dpos + jb;
#pragma unroll
        for (int c = 0; c < NCDL; ++c) dcd[c] = gl<double>(Dp, 8 * lane + 512 * c);
        // The bra pair, hence the J[a,b] addresses, is the same on every lane:
        // reduce across the wave, one update per element.
#pragma unroll
        for (int r = 0; r < NAL * NB; ++r) {
          double s = 0.0;
#pragma unroll
          for (int c = 0; c < NCDL; ++c) s = fma((double)tile[r * NCDL + c], dcd[c], s);
          s = wave_sum(active ? fj * s : 0.0);
          if (lane == 0) {
            if (lds)
              acc_add(&s_acc[so + acc.jab + (a0 + r / NB) * NB + r % NB], s, FX);
            else
              acc_add(Jo + br.msh + (long long)(br.aoA + a0 + r / NB) * N + br.aoB + r % NB, s, FX);
          }
        }
      }
      if (bk && active) {
        double dab[NAL * NB];
#pragma unroll
        for (int ia = 0; ia < NAL; ++ia)
#pragma unroll
          for (int ib = 0; ib < NB; ++ib) dab[ia * NB + ib] = cl(rowA(ia), br.aoB + ib);
        double* Jp = dn->Jpos + jb;
#pragma unroll
        for (int c = 0; c < NCDL; ++c) {
          double s = 0.0;
#pragma unroll
          for (int r = 0; r < NAL * NB; ++r) s = fma((double)tile[r * NCDL + c], dab[r], s);
          if (jcd && di == 0)
            jcd[c] = fma(fj, s, jcd[c]);
          else
            acc_add((double*)((ASUKA_GLOB char*)Jp + (8 * lane + 512 * c)), fj * s, FX);
        }
      }
    }
    double* Ko = dn->K;
    if (Ko && active) {
      auto addK = [&](int off, int cols, int col0, long long row, unsigned o, double v) {
        if (lds)
          acc_add(&s_acc[so + off + cols + col0], v, FX);
        else
          acc_add((double*)((ASUKA_GLOB char*)(Ko + br.msh + row * N) + o), v, FX);
      };
      {  // K[a,c] += sum_{b,d} v D[b,d]
        double dbd[NB * ND];
#pragma unroll
        for (int ib = 0; ib < NB; ++ib)
#pragma unroll
          for (int id = 0; id < ND; ++id) dbd[ib * ND + id] = gl<double>(rowB(ib), oD + 8 * id);
#pragma unroll
        for (int ia = 0; ia < NAL; ++ia)
#pragma unroll
          for (int ic = 0; ic < NCL; ++ic) {
            double s = 0.0;
#pragma unroll
            for (int ib = 0; ib < NB; ++ib)
#pragma unroll
              for (int id = 0; id < ND; ++id) s = fma((double)tile[(ia * NB + ib) * NCDL + ic * ND + id], dbd[ib * ND + id], s);
            addK(acc.kac, (a0 + ia) * acc.colsC, colC + ic, br.aoA + a0 + ia, oC + 8 * ic, ks * s);
          }
      }
      if (cd_neq) {  // K[a,d] += sum_{b,c} v D[b,c]
        double dbc[NB * NCL];
#pragma unroll
        for (int ib = 0; ib < NB; ++ib)
#pragma unroll
          for (int ic = 0; ic < NCL; ++ic) dbc[ib * NCL + ic] = gl<double>(rowB(ib), oC + 8 * ic);
#pragma unroll
        for (int ia = 0; ia < NAL; ++ia)
#pragma unroll
          for (int id = 0; id < ND; ++id) {
            double s = 0.0;
#pragma unroll
            for (int ib = 0; ib < NB; ++ib)
#pragma unroll
              for (int ic = 0; ic < NCL; ++ic) s = fma((double)tile[(ia * NB + ib) * NCDL + ic * ND + id], dbc[ib * NCL + ic], s);
            addK(acc.kad, (a0 + ia) * acc.colsD, colD + id, br.aoA + a0 + ia, oD + 8 * id, ks * s);
          }
      }
      if (ab_neq) {  // K[b,c] += sum_{a,d} v D[a,d]
        double dad[NAL * ND];
#pragma unroll
        for (int ia = 0; ia < NAL; ++ia)
#pragma unroll
          for (int id = 0; id < ND; ++id) dad[ia * ND + id] = gl<double>(rowA(ia), oD + 8 * id);
#pragma unroll
        for (int ib = 0; ib < NB; ++ib)
#pragma unroll
          for (int ic = 0; ic < NCL; ++ic) {
            double s = 0.0;
#pragma unroll
            for (int ia = 0; ia < NAL; ++ia)
#pragma unroll
              for (int id = 0; id < ND; ++id) s = fma((double)tile[(ia * NB + ib) * NCDL + ic * ND + id], dad[ia * ND + id], s);
            addK(acc.kbc, ib * acc.colsC, colC + ic, br.aoB + ib, oC + 8 * ic, ks * s);
          }
        if (cd_neq) {  // K[b,d] += sum_{a,c} v D[a,c]
          double dac[NAL * NCL];
#pragma unroll
          for (int ia = 0; ia < NAL; ++ia)
#pragma unroll
            for (int ic = 0; ic < NCL; ++ic) dac[ia * NCL + ic] = gl<double>(rowA(ia), oC + 8 * ic);
#pragma unroll
          for (int ib = 0; ib < NB; ++ib)
#pragma unroll
            for (int id = 0; id < ND; ++id) {
              double s = 0.0;
#pragma unroll
              for (int ia = 0; ia < NAL; ++ia)
#pragma unroll
                for (int ic = 0; ic < NCL; ++ic)
                  s = fma((double)tile[(ia * NB + ib) * NCDL + ic * ND + id], dac[ia * NCL + ic], s);
              addK(acc.kbd, ib * acc.colsD, colD + id, br.aoB + ib, oD + 8 * id, ks * s);
            }
        }
      }
    }
  }  // densities
}

template <class PL, int CH, typename CT, bool FX>
__device__ __forceinline__ void dispatch_chunk(int chunk, ArgP ap, const Bra& br, int col, const UnitRange& ur,
                                               bool active, const CT* __restrict__ tab, const RowAcc& acc) {
  if constexpr (CH < PL::NCH) {
    if (chunk == CH) {
      run_chunk<PL, CH, CT, FX>(ap, br, col, ur, active, tab, acc, nullptr);
      return;
    }
    dispatch_chunk<PL, CH + 1, CT, FX>(chunk, ap, br, col, ur, active, tab, acc);
  }
}

// The A chunks CA.. of C chunk CC, in sequence, carrying J[c,d] in jcd.
template <class PL, int CC, int CA, typename CT, bool FX>
__device__ __forceinline__ void run_agroup(ArgP ap, const Bra& br, int col, const UnitRange& ur, bool active,
                                           const CT* __restrict__ tab, const RowAcc& acc, double* jcd) {
  if constexpr (CA < PL::SPLIT_A) {
    run_chunk<PL, CA * PL::SPLIT_C + CC, CT, FX>(ap, br, col, ur, active, tab, acc, jcd);
    run_agroup<PL, CC, CA + 1, CT, FX>(ap, br, col, ur, active, tab, acc, jcd);
  }
}

// One wave item of a CARRY plan: C chunk CC of a unit, all of its A chunks,
// with the J[c,d] sums carried across the A chunks in registers, so J[c,d]
// receives one atomic per element and quartet instead of one per A chunk.
template <class PL, int CC, typename CT, bool FX>
__device__ __forceinline__ void run_citem(ArgP ap, const Bra& br, int col, const UnitRange& ur, bool active,
                                          const CT* __restrict__ tab, const RowAcc& acc) {
  using CK = Chunk<PL, CC>;  // A chunk 0: the C range of every A chunk of CC
  constexpr int ND = PL::ND, NCDL = (CK::c1 - CK::c0) * ND;
  double jcd[NCDL];
#pragma unroll
  for (int c = 0; c < NCDL; ++c) jcd[c] = 0.0;
  run_agroup<PL, CC, 0, CT, FX>(ap, br, col, ur, active, tab, acc, jcd);
  ap = refetch(ap);
  const unsigned lane = threadIdx.x & 63;
  if (ap->den[0].J && active && br.posP != col + (int)lane) {
    double* Jp = ap->den[0].Jpos + cl(ap->jblk, col >> 6) + 64LL * (CK::c0 * ND);
#pragma unroll
    for (int c = 0; c < NCDL; ++c) acc_add((double*)((ASUKA_GLOB char*)Jp + (8 * lane + 512 * c)), jcd[c], FX);
  }
}

// Wave item `item` of a unit: a C chunk with its A chunks for CARRY plans,
// one chunk otherwise.
template <class PL, int CC, typename CT, bool FX>
__device__ __forceinline__ void dispatch_citem(int cc, ArgP ap, const Bra& br, int col, const UnitRange& ur,
                                               bool active, const CT* __restrict__ tab, const RowAcc& acc) {
  if constexpr (!PL::CARRY) {
    dispatch_chunk<PL, 0, CT, FX>(cc, ap, br, col, ur, active, tab, acc);
  } else if constexpr (CC < PL::SPLIT_C) {
    if (cc == CC) {
      run_citem<PL, CC, CT, FX>(ap, br, col, ur, active, tab, acc);
      return;
    }
    dispatch_citem<PL, CC + 1, CT, FX>(cc, ap, br, col, ur, active, tab, acc);
  }
}

// Work mapping: each workgroup pulls row tasks (wave units of one bra pair,
// longest first) from the class pair's queue; its wavefronts take the task's
// (unit, chunk) items in turn, so within a wave the bra pair and the chunk
// (and with it all register indexing) are uniform. With LDS accumulators the
// task's J[a,b] block and K rows of a and b are summed in LDS and added to
// J/K once at the end of the task.
//
// Precision: CT is the kernel's arithmetic. In mixed builds the FP64 and the
// FP32 kernel of a split class pair each walk their own list of units, routed
// once per build (k_route_units). Separate kernels keep the FP32 path's
// register allocation (and so its occupancy) its own.
// FX: accumulate in the 64-bit fixed point of deterministic builds
// (EriOut::fixed), a separate instantiation so that the FP64-atomic kernels
// carry none of its code or registers.
template <class PL, typename CT, bool FX>
__global__ __launch_bounds__(kGroupThreads) void eri_fast_kernel(FastArgs args) {
  (void)args;  // read through the kernel-argument segment, where it starts
  ArgP ap = refetch((ArgP)__builtin_amdgcn_kernarg_segment_ptr());
  constexpr bool kF32 = sizeof(CT) == 4;
  constexpr int NIT = PL::CARRY ? PL::SPLIT_C : PL::NCH, NR = PL::NR;  // wave items per unit
  constexpr int NA = nc_(PL::la), NB = PL::NB;
  constexpr bool kLds = NR <= kLdsRootsMax;
  // LDS copy of the CT root table, intervals padded (rys_c::lds_stride_of)
  constexpr int NFI = rys_c::interval_size_of<CT>(NR);
  constexpr int SCT = rys_c::lds_stride_of<CT>(NR);
  constexpr int TB = kLds ? rys_c::block_size_of<CT>(NR) : 1;
  constexpr int TBC = kLds ? rys_c::nint_of<CT>(NR) * SCT : 1;
  const int wpg = ap->wpg, nthr = 64 * wpg;  // the launch's block size (uniform)
  __shared__ CT tct[TBC];
  const CT* gct;
  if constexpr (kF32)
    gct = rys_dev_f::rys32_coef + rys_c::coef_off32[NR];
  else
    gct = rys_dev::rys_coef + rys_c::coef_off[NR];
  if constexpr (kLds) {
    for (int t = threadIdx.x; t < TB; t += nthr) {
      const int iv = t / NFI, f = t - iv * NFI;
      tct[iv * SCT + f] = gct[t];
    }
  }
  RowAcc acc{};
  int nacc = 0;
  if (ap->acc_colsC > 0) {  // row-task accumulators in s_acc, sized at launch
    const int cC = ap->acc_colsC, cD = ap->acc_colsD;  // cD == 0: D columns share the C space
    acc.on = true;
    acc.colsC = cC;
    acc.colsD = cD > 0 ? cD : cC;
    acc.jab = 0;
    acc.kac = NA * NB;
    acc.kad = cD > 0 ? acc.kac + NA * cC : acc.kac;
    acc.kbc = acc.kac + NA * cC + (cD > 0 ? NA * cD : 0);
    acc.kbd = cD > 0 ? acc.kbc + NB * cC : acc.kbc;
    nacc = NA * NB + (NA + NB) * (cC + cD);
    acc.stride = nacc;
    for (int t = threadIdx.x; t < nacc * ap->nden; t += nthr) s_acc[t] = 0.0;
  }
  __shared__ int s_task, s_work;
  if (threadIdx.x == 0) s_work = 0;
  __syncthreads();
  const CT* tab = kLds ? tct : gct;
  const unsigned lane = threadIdx.x & 63;
  // blockDim is not read because the compiler cannot prove it uniform, which
  // would make the loops divergent
  const int wib = uni((int)(threadIdx.x >> 6));
  for (;;) {  // persistent workgroups pull row tasks from the class pair's queue
    ap = refetch(ap);
    if (threadIdx.x == 0) s_task = (int)atomicAdd(ap->queue, 1u);
    __syncthreads();
    const int t = uni(s_task);
    if (t >= ap->ntasks) break;  // uniform per workgroup; every workgroup gets here
    const int u0 = cl((const int*)ap->tasks, 2LL * t), nu = cl((const int*)ap->tasks, 2LL * t + 1);
    bool worked = false;  // this wave digested an item of the task (uniform)
    if (nu > 0) {         // routed lists hold empty tasks: no unit to read
      Bra br;
      br.P = cl((const int*)ap->units, 4LL * u0);
      br.A = cl(ap->sp_A, br.P);
      br.B = cl(ap->sp_B, br.P);
      br.ab0 = cl(ap->pp_start, br.P);
      br.posP = cl(ap->pos_of_sp, br.P);
      br.aoA = cl(ap->shell_ao, br.A);
      br.aoB = cl(ap->shell_ao, br.B);
      const int mol = cl(ap->shell_mol, br.A);
      br.N = cl(ap->mol_n, mol);
      br.msh = cl(ap->mol_shift, mol);
      // a wave item is one chunk of a unit, or for CARRY plans one C chunk with
      // its A chunks in sequence; items chunk-major: the waves of a workgroup
      // run the same chunk's code over different units (a split plan's chunks
      // are separate code regions, together far larger than the instruction cache)
      for (int item = wib; item < nu * NIT; item += wpg) {  // uniform per wave
        ap = refetch(ap);
        const int chunk = NIT == 1 ? 0 : item / nu;
        const int ui = item - chunk * nu;
        union {
          u32x4 v;
          WaveUnit u;
        } un;
        un.v = cl((const u32x4*)ap->units, u0 + ui);
        // a quartet of a deterministic build is rounded once, as a whole: the
        // last slice of a sliced unit runs all of it, the others nothing
        if constexpr (FX)
          if (!un.u.tail || (int)un.u.j1 != kUnitAll) continue;
        const int col = un.u.col;
        // the lane's ket position is col + lane: units start at 64-position
        // block boundaries, so tail lanes read padding positions of the block
        bool active = lane < (unsigned)un.u.ncol;
        const double bound = (cl(ap->Q, br.P) * gl<double>(ap->kq + col, 8 * lane)) *
                             fmax(cl(ap->Dsp, br.P), gl<double>(ap->kd + col, 8 * lane));
        if (ap->eps_density > 0.0) active = active && bound >= ap->eps_density;
        if (!wave_any(active)) continue;  // the whole unit is density-screened
        worked = true;
        // inactive lanes (tail, screened) run with an empty primitive loop and no
        // atomics so the wave stays converged for the cross-lane reductions
        UnitRange ur = unit_range(un.u, cl(ap->pp_count, br.P), false);
        if constexpr (FX) ur = UnitRange{0, ur.i0 + ur.ni, 0, ur.j1};
        dispatch_citem<PL, 0, CT, FX>(chunk, ap, br, col, ur, active, tab, acc);
      }
      if (acc.on) {
        if (worked && lane == 0) s_work = 1;
        __syncthreads();  // the task's contributions are in LDS
        ap = refetch(ap);
        if (s_work) {
          const long long N = br.N, msh = br.msh, aoA = br.aoA, aoB = br.aoB;
          const int cC = ap->acc_colsC, cD = ap->acc_colsD, nden = ap->nden;
          const int* mlao = ap->mol_lao + mol * (ASUKA_LMAX + 1);  // the molecule's AO lists
          // compact columns of the C and D lists (EriOut::Kc)
          const int gC = ap->lao_offC + mlao[PL::lc], gD = cD > 0 ? ap->lao_offD + mlao[PL::ld] : gC;
          const int* lao_ao = ap->lao_ao;
          const int cDe = cD > 0 ? cD : cC;
          for (int t2 = threadIdx.x; t2 < nacc * nden; t2 += nthr) {
            const double v = s_acc[t2];  // fixed builds: the bits of an integer sum
            if (__double_as_longlong(v) == 0LL) continue;
            s_acc[t2] = 0.0;
            const bool second = t2 >= nacc;
            const ASUKA_CONST FastDen* dn = &ap->den[second ? 1 : 0];
            int r = second ? t2 - nacc : t2;
            if (r < NA * NB) {
              acc_add_sum(dn->J + msh + (aoA + r / NB) * N + aoB + r % NB, v, FX);
              continue;
            }
            r -= NA * NB;
            long long row, k;  // the K row (AO) and the entry's index in its column list
            int g;             // first compact column of that list
            if (r < NA * cC) {
              row = aoA + r / cC, k = r % cC, g = gC;
            } else if ((r -= NA * cC), cD > 0 && r < NA * cD) {
              row = aoA + r / cD, k = r % cD, g = gD;
            } else {
              if (cD > 0) r -= NA * cD;
              if (r < NB * cC) {
                row = aoB + r / cC, k = r % cC, g = gC;
              } else {
                r -= NB * cC;
                row = aoB + r / cDe, k = r % cDe, g = gD;
              }
            }
            if (dn->Kc)  // consecutive entries, consecutive addresses
              acc_add_sum(dn->Kc + row * N + g + k, v, FX);
            else
              acc_add_sum(dn->K + msh + row * N + lao_ao[g + k], v, FX);
          }
        }
      }
    }
    __syncthreads();  // accumulators are zero again; s_task and s_work may be overwritten
    if (acc.on && threadIdx.x == 0) s_work = 0;
  }
}

// Bytes of LDS accumulators for a class pair with ket columns (colsC, colsD),
// per density.
inline size_t row_acc_bytes(int la, int lb, int colsC, int colsD) {
  const int NA = nc_(la), NB = nc_(lb);
  return sizeof(double) * (size_t)(NA * NB + (NA + NB) * (colsC + colsD));
}

// The FP32 kernel's plan of a class: half the FP64 plan's component chunks
// (the FP32 intermediates take half the registers), A chunks halved when
// their count is even, else C chunks; ASUKA_F32_HALVE=0 keeps the FP64 plan's.
// Measured at (H2O)64 cc-pVDZ, single stream: (21|11) 9.6 -> 7.6 ms, (20|11)
// 28.3 -> 18.3 ms, (21|21) 18.0 -> 11.7 ms per build for the FP32 kernels.
#ifndef ASUKA_F32_HALVE
#define ASUKA_F32_HALVE 1
#endif
template <class PL>
struct F32PlanOf {
  static constexpr bool halve_a = ASUKA_F32_HALVE && PL::SPLIT_A % 2 == 0;
  static constexpr bool halve_c = ASUKA_F32_HALVE && !halve_a && PL::SPLIT_C % 2 == 0;
  static constexpr int SA = halve_a ? PL::SPLIT_A / 2 : PL::SPLIT_A;
  static constexpr int SC = halve_c ? PL::SPLIT_C / 2 : PL::SPLIT_C;
  using type = Plan<PL::la, PL::lb, PL::lc, PL::ld, SA, SC>;
};

// The kernel arguments of a class pair's launch in one precision: f32 takes the
// FP32 list of units and tasks (ClassWork::units32).
inline FastArgs fast_args(const DevBasis& b, const ClassWork& w, const EriOut& o, bool f32) {
  FastArgs a{};
  a.units = f32 ? w.units32 : w.units;
  a.tasks = f32 ? w.tasks32 : w.tasks;
  a.queue = f32 ? w.queue32 : w.queue;
  a.pp = f32 ? (const void*)b.ppf32 : (const void*)b.ppf;
  a.kpd = f32 ? b.kp32d : b.kp64;
  a.kpf = b.kp32f;
  a.kpoff = b.kpoff;
  a.sp_A = b.sp_A, a.sp_B = b.sp_B, a.pp_start = b.pp_start, a.pp_count = b.pp_count;
  a.shell_ao = b.shell_ao, a.shell_mol = b.shell_mol, a.mol_n = b.mol_n, a.mol_lao = b.mol_lao;
  a.lao_ao = b.lao_ao, a.pos_of_sp = b.pos_of_sp, a.mol_shift = b.mol_shift, a.jblk = o.jblk;
  a.shell_xyz = b.shell_xyz, a.Q = b.Q, a.Dsp = b.Dsp, a.kq = b.kq, a.kd = b.kd, a.kcd = b.kcd;
  a.kpp = b.kpp, a.kao = b.kao, a.klao = b.klao;
  const bool fock = o.mode == MODE_FOCK;
  a.den[0] = FastDen{o.D, fock ? o.F : o.J, fock ? o.F : o.K, o.Dpos, o.Jpos, o.Kc};
  a.den[1] = FastDen{o.D2, o.J2, o.K2, o.Dpos2, o.Jpos2, o.Kc2};
  a.eps_density = o.eps_density, a.eps_prim = o.eps_prim;
  a.ks = fock ? -0.5 : 1.0;
  a.nden = o.D2 ? 2 : 1;
  a.ntasks = (int)w.ntasks;
  a.wpg = w.wpg;
  a.acc_colsC = w.acc_colsC, a.acc_colsD = w.acc_colsD, a.lao_offC = w.lao_offC, a.lao_offD = w.lao_offD;
  return a;
}

template <class PL, typename CT, bool FX = false>
hipError_t launch_one(const DevBasis& b, const ClassWork& w, const EriOut& o, size_t lds, long long g, hipStream_t s) {
  if (lds > 64 * 1024) {
    const hipError_t e = hipFuncSetAttribute((const void*)eri_fast_kernel<PL, CT, FX>,
                                             hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) return e;
  }
  hipLaunchKernelGGL((eri_fast_kernel<PL, CT, FX>), dim3((unsigned)g), dim3(64 * w.wpg), lds, s,
                     fast_args(b, w, o, sizeof(CT) == 4));
  return hipGetLastError();
}

// The FP64 kernel of a class pair and, for mixed builds, the FP32 kernel after
// it on the same stream (each takes its own units, see eri_fast_kernel).
template <class PL>
hipError_t launch_plan(const DevBasis& b, const ClassWork& w, const EriOut& o, hipStream_t s) {
  long long g = w.ntasks;  // persistent: a few workgroups per CU, tasks from the queue
  const long long gmax = w.wpg == 8 ? 1024 : 2048;
  if (g > gmax) g = gmax;
  if (g < 1) g = 1;
  const size_t lds =
      w.acc_colsC > 0 ? (o.D2 ? 2 : 1) * row_acc_bytes(PL::la, PL::lb, w.acc_colsC, w.acc_colsD) : 0;
  // deterministic builds (no mixed routing: every unit on the FP64 kernel)
  if (o.fixed) return launch_one<PL, double, true>(b, w, o, lds, g, s);
  hipError_t e = launch_one<PL, double>(b, w, o, lds, g, s);
  if (e != hipSuccess || !o.mixed) return e;
  return launch_one<typename F32PlanOf<PL>::type, float>(b, w, o, lds, g, s);
}

using Launcher = hipError_t (*)(const DevBasis&, const ClassWork&, const EriOut&, hipStream_t);

}  // namespace asuka_fast

// Each jk_fast_*.hip translation unit instantiates a subset of class plans;
// FN returns a plan's launcher, FN##_nch its wave items per unit (the number
// of component chunks, or of C chunks for plans that carry J[c,d] across
// their A chunks).
#define ASUKA_FAST_FIND(FN, LIST)                                                     \
  asuka_fast::Launcher FN(int la, int lb, int lc, int ld) {                          \
    using namespace asuka_fast;                                                       \
    LIST(ASUKA_FAST_CASE)                                                             \
    return nullptr;                                                                   \
  }                                                                                   \
  int FN##_nch(int la, int lb, int lc, int ld) {                                      \
    LIST(ASUKA_FAST_NCH_CASE)                                                         \
    return 0;                                                                         \
  }
#define ASUKA_FAST_CASE(a, b_, c, d, sa, sc) \
  if (la == a && lb == b_ && lc == c && ld == d) return &launch_plan<Plan<a, b_, c, d, sa, sc>>;
#define ASUKA_FAST_NCH_CASE(a, b_, c, d, sa, sc) \
  if (la == a && lb == b_ && lc == c && ld == d) return asuka_fast::Plan<a, b_, c, d, sa, sc>::CARRY ? (sc) : (sa) * (sc);
