// Device side of the graph-captured SCF iteration, so that it needs no host
// round trip: the DIIS extrapolation coefficients (asuka/hf/df_scf.py:722-835)
// and the density purification that stands in for eigh and aufbau.
//
// DIIS.
// The driver keeps up to kDiisSlots Fock matrices and commutator errors in a
// ring of slots and their Gram matrix G[i][j] = <e_i, e_j> on the device;
// this kernel forms the reference's bordered system
//   [ G/g  -1 ] [c]   [ 0]
//   [ -1    0 ] [l] = [-1],   g = max |G|,
// solves it by Gaussian elimination with partial pivoting, retrying with
// lambda I added to G/g for lambda in (0, 1e-14, 1e-12, 1e-10, 1e-8, 1e-6)
// until the solve has no zero pivot and a finite result, and renormalises c
// to unit sum. Where the reference would fall back (fewer than 2 vectors, a
// non-finite G, every solve failing, |sum c| < 1e-15), the weights select the
// newest Fock matrix alone; the reference's least-squares retry after every
// solve failed is not taken (it cannot be reached with a finite G, whose
// regularised systems are nonsingular).
#include <hip/hip_runtime.h>

#include <cmath>
#include <string>

#include "../../include/asuka_jk.h"
#include "jk_internal.h"

namespace {

// ---------------------------------------------------------------------------
// Purification (TC2; A. M. N. Niklasson, Phys. Rev. B 66, 155115 (2002)):
// P = (e1 - F) / (e1 - e0) with [e0, e1] the Gershgorin interval of F, then
// P <- P^2 while Tr P exceeds the number of occupied orbitals and 2P - P^2
// otherwise; frozen once ||P^2 - P||_F < tol (further steps would undo it).
//
// Matrices up to kPurifyLds run in one kernel: one workgroup of 16 wavefronts
// holds P in LDS and forms P P^T (P is symmetric) on the FP64 matrix cores, 16
// x 16 tiles of the upper triangle, at most three a wave, kept in registers
// until the whole square is known. A step is two barriers and a few
// microseconds against a dozen launches of separate operations (product,
// norm, trace, selects), which is what bounds small systems: (H2O)3 cc-pVDZ (75
// AOs), about 50 steps in 158 us, where they took about 4 ms; the whole SCF
// 144 -> 55 ms. Larger matrices take one product (by the caller) and two small
// kernels a step. The limit is what LDS holds in whole tiles with a padded row.
// ---------------------------------------------------------------------------
constexpr int kPurifyLds = 128;
constexpr int kPurifyWaves = 16;
constexpr int kPurifyTiles = 3;  // ceil(36 upper tiles of 8 x 8 / 16 waves)
typedef double d4 __attribute__((ext_vector_type(4)));

__host__ __device__ constexpr int purify_ld(int n) { return (n + 15) / 16 * 16 + 1; }
constexpr size_t purify_lds_bytes(int n) {
  return sizeof(double) * ((size_t)(purify_ld(n) - 1) * purify_ld(n) + 2 * kPurifyLds);
}

__global__ __launch_bounds__(64 * kPurifyWaves) void k_purify_lds(const double* __restrict__ F, int n, int nocc,
                                                                  int iters, double tol, double* P, double* err,
                                                                  int* steps) {
  extern __shared__ double s_p[];  // [n16][ld], zero beyond n
  const int ld = purify_ld(n), n16 = ld - 1, nt = n16 / 16;
  double* red = s_p + (size_t)n16 * ld;  // 2 * kPurifyLds
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  constexpr int kThr = 64 * kPurifyWaves;
  for (int e = tid; e < n16 * ld; e += kThr) {
    const int i = e / ld, j = e - i * ld;
    s_p[e] = (i < n && j < n) ? F[(long long)i * n + j] : 0.0;
  }
  __syncthreads();
  if (tid < n) {  // Gershgorin discs
    double r = 0.0;
    for (int j = 0; j < n; ++j) r += fabs(s_p[tid * ld + j]);
    const double d = s_p[tid * ld + tid];
    r -= fabs(d);
    red[tid] = d - r;
    red[kPurifyLds + tid] = d + r;
  }
  __syncthreads();
  double e0 = red[0], e1 = red[kPurifyLds];
  for (int i = 1; i < n; ++i) {
    e0 = fmin(e0, red[i]);
    e1 = fmax(e1, red[kPurifyLds + i]);
  }
  const double sc = e1 - e0;
  for (int e = tid; e < n16 * ld; e += kThr) {
    const int i = e / ld, j = e - i * ld;
    if (i < n && j < n) s_p[e] = ((i == j ? e1 : 0.0) - s_p[e]) / sc;
  }
  __syncthreads();
  // this wave's upper tiles (I <= J), dealt out in order
  int ti[kPurifyTiles], tj[kPurifyTiles];
#pragma unroll
  for (int t = 0; t < kPurifyTiles; ++t) {
    int k = wave + t * kPurifyWaves, I = 0;
    while (I < nt && k >= nt - I) k -= nt - I, ++I;
    ti[t] = I;  // nt: no tile
    tj[t] = I + k;
  }
  const int r16 = lane & 15, kq = lane >> 4;
  double er = 0.0;
  int done = 0;
  for (int it = 0; it < iters; ++it) {
    d4 c[kPurifyTiles];
    double e2 = 0.0, tr = 0.0;
#pragma unroll
    for (int t = 0; t < kPurifyTiles; ++t) {
      if (ti[t] >= nt) continue;  // uniform per wave
      const double* a = s_p + (ti[t] * 16 + r16) * ld + kq;
      const double* b = s_p + (tj[t] * 16 + r16) * ld + kq;
      d4 x = {0, 0, 0, 0}, y = {0, 0, 0, 0};
      for (int k = 0; k < n16; k += 8) {
        x = __builtin_amdgcn_mfma_f64_16x16x4f64(a[k], b[k], x, 0, 0, 0);
        y = __builtin_amdgcn_mfma_f64_16x16x4f64(a[k + 4], b[k + 4], y, 0, 0, 0);
      }
      c[t] = x + y;
      const double w = ti[t] == tj[t] ? 1.0 : 2.0;
#pragma unroll
      for (int q = 0; q < 4; ++q) {  // accumulator q of a lane: row 4 q + lane / 16, column lane % 16
        const int row = ti[t] * 16 + 4 * q + kq, col = tj[t] * 16 + r16;
        const double p = s_p[row * ld + col], d = c[t][q] - p;
        e2 = fma(w * d, d, e2);
        if (row == col) tr += p;
      }
    }
    e2 = wave_total(e2);
    tr = wave_total(tr);
    if (lane == 0) {
      red[wave] = e2;
      red[kPurifyWaves + wave] = tr;
    }
    __syncthreads();  // every wave has read P
    e2 = tr = 0.0;
#pragma unroll
    for (int w = 0; w < kPurifyWaves; ++w) {
      e2 += red[w];
      tr += red[kPurifyWaves + w];
    }
    er = sqrt(e2);
    if (er < tol) {  // uniform: the same sums on every thread
      done = it + 1;
      break;
    }
    const bool square = tr > (double)nocc;
#pragma unroll
    for (int t = 0; t < kPurifyTiles; ++t) {
      if (ti[t] >= nt) continue;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int row = ti[t] * 16 + 4 * q + kq, col = tj[t] * 16 + r16;
        const double v = square ? c[t][q] : 2.0 * s_p[row * ld + col] - c[t][q];
        s_p[row * ld + col] = v;
        if (ti[t] != tj[t]) s_p[col * ld + row] = v;
      }
    }
    __syncthreads();
  }
  __syncthreads();
  for (int e = tid; e < n * n; e += kThr) {
    const int i = e / n, j = e - i * n;
    P[e] = s_p[i * ld + j];
  }
  if (tid == 0) {
    *err = er;
    *steps = done;
  }
}

// One TC2 step of a larger matrix: partial sums of ||P2 - P||^2 and Tr P per
// workgroup, then the update (every workgroup adds up the partial sums itself).
constexpr int kTc2Parts = 128;

__global__ __launch_bounds__(256) void k_tc2_sums(const double* __restrict__ P, const double* __restrict__ P2, int n,
                                                  double* part) {
  __shared__ double s[8];
  double e2 = 0.0, tr = 0.0;
  const long long nn = (long long)n * n, stride = (long long)gridDim.x * 256;
  for (long long e = blockIdx.x * 256LL + threadIdx.x; e < nn; e += stride) {
    const double d = P2[e] - P[e];
    e2 = fma(d, d, e2);
  }
  for (long long i = blockIdx.x * 256LL + threadIdx.x; i < n; i += stride) tr += P[i * n + i];
  e2 = wave_total(e2);
  tr = wave_total(tr);
  if ((threadIdx.x & 63) == 0) {
    s[threadIdx.x >> 6] = e2;
    s[4 + (threadIdx.x >> 6)] = tr;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    part[2 * blockIdx.x] = s[0] + s[1] + s[2] + s[3];
    part[2 * blockIdx.x + 1] = s[4] + s[5] + s[6] + s[7];
  }
}

__global__ __launch_bounds__(256) void k_tc2_update(double* P, const double* __restrict__ P2, int n, int nocc,
                                                    double tol, const double* __restrict__ part, int* done, int it,
                                                    double* err) {
  double e2 = 0.0, tr = 0.0;
  for (int k = 0; k < kTc2Parts; ++k) {
    e2 += part[2 * k];
    tr += part[2 * k + 1];
  }
  const double er = sqrt(e2);
  const bool frozen = (it > 0 && done[it - 1]) || er < tol;
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    done[it] = frozen ? 1 : 0;
    *err = er;
  }
  if (frozen) return;
  const bool square = tr > (double)nocc;
  const long long nn = (long long)n * n, stride = (long long)gridDim.x * 256;
  for (long long e = blockIdx.x * 256LL + threadIdx.x; e < nn; e += stride)
    P[e] = square ? P2[e] : 2.0 * P[e] - P2[e];
}

constexpr int kDiisSlots = 8;

// Solves the (m x m) system A x = b in place (A row-major, partial pivoting);
// false on an exactly zero pivot (numpy/LAPACK getrf info > 0) or a non-finite x.
__device__ bool solve_small(double* A, double* b, int m) {
  for (int k = 0; k < m; ++k) {
    int p = k;
    double pv = fabs(A[k * m + k]);
    for (int i = k + 1; i < m; ++i)
      if (fabs(A[i * m + k]) > pv) {
        pv = fabs(A[i * m + k]);
        p = i;
      }
    if (pv == 0.0) return false;
    if (p != k) {
      for (int j = 0; j < m; ++j) {
        const double t = A[k * m + j];
        A[k * m + j] = A[p * m + j];
        A[p * m + j] = t;
      }
      const double t = b[k];
      b[k] = b[p];
      b[p] = t;
    }
    for (int i = k + 1; i < m; ++i) {
      const double f = A[i * m + k] / A[k * m + k];
      for (int j = k; j < m; ++j) A[i * m + j] -= f * A[k * m + j];
      b[i] -= f * b[k];
    }
  }
  for (int k = m - 1; k >= 0; --k) {
    double s = b[k];
    for (int j = k + 1; j < m; ++j) s -= A[k * m + j] * b[j];
    b[k] = s / A[k * m + k];
    if (!isfinite(b[k])) return false;
  }
  return true;
}

// One thread: G (kDiisSlots x kDiisSlots, row stride kDiisSlots) over a ring
// of nslot <= kDiisSlots slots, count = number of vectors pushed so far (slots
// 0..n-1 in use, n = min(count, nslot); the newest in slot (count - 1) % nslot).
// coeff (kDiisSlots): extrapolation weights per slot; status: 1 extrapolated,
// 0 newest Fock matrix alone.
__global__ void k_diis_solve(const double* G, const long long* count, int nslot, double* coeff, int* status) {
  if (threadIdx.x != 0 || blockIdx.x != 0) return;
  const long long cnt = *count;
  const int n = cnt < nslot ? (int)cnt : nslot;
  const int newest = cnt > 0 ? (int)((cnt - 1) % nslot) : 0;
  for (int i = 0; i < kDiisSlots; ++i) coeff[i] = 0.0;
  coeff[newest] = 1.0;
  *status = 0;
  if (n < 2) return;
  double g = 0.0;
  for (int i = 0; i < n; ++i)
    for (int j = 0; j < n; ++j) {
      const double v = G[i * kDiisSlots + j];
      if (!isfinite(v)) return;
      g = fmax(g, fabs(v));
    }
  const double scale = (isfinite(g) && g > 0.0) ? g : 1.0;
  const int m = n + 1;
  const double ladder[6] = {0.0, 1e-14, 1e-12, 1e-10, 1e-8, 1e-6};
  double A[(kDiisSlots + 1) * (kDiisSlots + 1)], x[kDiisSlots + 1];
  for (int r = 0; r < 6; ++r) {
    for (int i = 0; i < m; ++i) {
      for (int j = 0; j < m; ++j) {
        double v;
        if (i < n && j < n)
          v = G[i * kDiisSlots + j] / scale + (i == j ? ladder[r] : 0.0);
        else if (i == n && j == n)
          v = 0.0;
        else
          v = -1.0;
        A[i * m + j] = v;
      }
      x[i] = (i == n) ? -1.0 : 0.0;
    }
    if (!solve_small(A, x, m)) continue;
    double s = 0.0;
    for (int i = 0; i < n; ++i) s += x[i];
    if (!isfinite(s) || fabs(s) < 1e-15) return;
    for (int i = 0; i < kDiisSlots; ++i) coeff[i] = i < n ? x[i] / s : 0.0;
    *status = 1;
    return;
  }
}

}  // namespace

// sets the message of asuka_jk_last_error (jk_api.hip)
int asuka_fail_msg(int code, const char* msg);

extern "C" {

int asuka_scf_diis_solve(const double* G, const int64_t* count, int nslot, double* coeff, int32_t* status,
                         void* stream) {
  if (!G || !count || !coeff || !status) return asuka_fail_msg(ASUKA_E_INVALID, "G, count, coeff and status must be non-null");
  if (nslot < 1 || nslot > kDiisSlots) return asuka_fail_msg(ASUKA_E_INVALID, "nslot must be in [1, 8]");
  hipLaunchKernelGGL(k_diis_solve, dim3(1), dim3(64), 0, (hipStream_t)stream, G, (const long long*)count, nslot,
                     coeff, (int*)status);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return asuka_fail_msg(ASUKA_E_HIP, (std::string("k_diis_solve: ") + hipGetErrorString(e)).c_str());
  return ASUKA_OK;
}

int asuka_scf_purify_max(void) { return kPurifyLds; }

int asuka_scf_purify(const double* F, int n, int nocc, int iters, double tol, double* P, double* err, int32_t* steps,
                     void* stream) {
  if (!F || !P || !err || !steps) return asuka_fail_msg(ASUKA_E_INVALID, "F, P, err and steps must be non-null");
  if (n < 1 || n > kPurifyLds)
    return asuka_fail_msg(ASUKA_E_INVALID, ("n must be in [1, " + std::to_string(kPurifyLds) + "]").c_str());
  if (iters < 0) return asuka_fail_msg(ASUKA_E_INVALID, "iters must be >= 0");
  const size_t lds = purify_lds_bytes(n);
  hipError_t e = hipSuccess;
  if (lds > 64 * 1024)
    e = hipFuncSetAttribute((const void*)k_purify_lds, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
  if (e == hipSuccess) {
    hipLaunchKernelGGL(k_purify_lds, dim3(1), dim3(64 * kPurifyWaves), lds, (hipStream_t)stream, F, n, nocc, iters, tol,
                       P, err, (int*)steps);
    e = hipGetLastError();
  }
  if (e != hipSuccess) return asuka_fail_msg(ASUKA_E_HIP, (std::string("k_purify_lds: ") + hipGetErrorString(e)).c_str());
  return ASUKA_OK;
}

int asuka_scf_tc2_step(double* P, const double* P2, int n, int nocc, double tol, double* work, int32_t* done, int it,
                       double* err, void* stream) {
  if (!P || !P2 || !work || !done || !err)
    return asuka_fail_msg(ASUKA_E_INVALID, "P, P2, work, done and err must be non-null");
  if (n < 1 || it < 0) return asuka_fail_msg(ASUKA_E_INVALID, "n must be >= 1 and it >= 0");
  hipLaunchKernelGGL(k_tc2_sums, dim3(kTc2Parts), dim3(256), 0, (hipStream_t)stream, P, P2, n, work);
  const long long g = ((long long)n * n + 255) / 256;
  hipLaunchKernelGGL(k_tc2_update, dim3((unsigned)(g < 2048 ? g : 2048)), dim3(256), 0, (hipStream_t)stream, P, P2, n,
                     nocc, tol, work, (int*)done, it, err);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return asuka_fail_msg(ASUKA_E_HIP, (std::string("k_tc2_update: ") + hipGetErrorString(e)).c_str());
  return ASUKA_OK;
}

}  // extern "C"
