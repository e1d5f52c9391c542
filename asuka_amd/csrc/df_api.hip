// C-ABI of the density-fitting integrals: the auxiliary Coulomb metric
// V(P,Q) = (P|Q) and the three-centre integrals X(P, mu, nu) = (mu nu|P).
//
// Replaces metric_2c2e_basis and int3c2e_basis (asuka/cueri/df.py:803-945),
// whose GPU kernels are Rys quadrature with the fourth function a unit s
// (asuka/cueri/cuda/ext/src/cueri_cuda_kernels_rys_generic_part1.cu:1868-2785).
// Here an auxiliary shell P becomes the shell pair (P, u) with u the constant
// function 1 (an s shell of exponent 0 and coefficient 1): its primitive pairs
// are P's primitives (eta = alpha_P, centre R_P, cK = c_P), so (mu nu|P u) =
// (mu nu|P) and (P u|Q u) = (P|Q) run through the same Rys machinery as the
// four-centre integrals with l_d = 0, in kernels of their own (df_impl.h), one
// launch per class (la lb|lc), that write the results straight into X or V.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <map>
#include <memory>
#include <mutex>
#include <string>
#include <vector>

#include "../../include/asuka_jk.h"
#include "df_impl.h"

int asuka_fail_msg(int code, const char* msg);
asuka_df::DfLauncher find_df_p0(int la, int lb, int lc);
asuka_df::DfLauncher find_df_p1(int la, int lb, int lc);
asuka_df::DfLauncher find_df_p2(int la, int lb, int lc);
asuka_df::DfLauncher find_df_p3(int la, int lb, int lc);

struct asuka_df_ctx {
  int nao = 0, naux = 0;
  int nsh_ao = 0, nsh_aux = 0;
  int nsp_ao = 0;  // AO shell pairs; pair nsp_ao + i is (aux shell i, unit)
  int lmax_ao = 0, lmax_aux = 0;
  DevBasis dev{};
  // AO shell pairs by class (la (la + 1) / 2 + lb), longest contraction first,
  // and the auxiliary shells' pairs by l
  static constexpr int kClasses = (ASUKA_LMAX + 1) * (ASUKA_LMAX + 2) / 2;
  int *d_bra = nullptr, *d_aux = nullptr;
  int bra_off[kClasses + 1] = {0}, aux_off[ASUKA_LMAX + 2] = {0};
  std::vector<void*> owned;
  // A call's class launches go round the caller's stream and these, forked from
  // and joined back into it by events: they are short (a few dozen
  // workgroups each at small sizes), so one after another they would leave the
  // chip idle. mu: one call's fork, launches and join at a time.
  static constexpr int kSide = 3;
  hipStream_t side[kSide] = {};
  hipEvent_t ev_fork = nullptr, ev_join[kSide] = {};
  std::mutex mu;
  ~asuka_df_ctx() {
    for (void* p : owned) (void)hipFree(p);  // waits for the work that uses it
    for (int k = 0; k < kSide; ++k) {
      if (ev_join[k]) (void)hipEventDestroy(ev_join[k]);
      if (side[k]) (void)hipStreamDestroy(side[k]);
    }
    if (ev_fork) (void)hipEventDestroy(ev_fork);
  }
};

namespace {

template <typename Tp>
int upload(Tp** dst, const std::vector<Tp>& src, std::vector<void*>& owned) {
  *dst = nullptr;
  const size_t bytes = sizeof(Tp) * std::max<size_t>(1, src.size());
  hipError_t e = hipMalloc((void**)dst, bytes);
  if (e != hipSuccess) return asuka_fail_msg(ASUKA_E_NOMEM, (std::string("hipMalloc: ") + hipGetErrorString(e)).c_str());
  owned.push_back(*dst);
  if (!src.empty()) {
    e = hipMemcpy(*dst, src.data(), sizeof(Tp) * src.size(), hipMemcpyHostToDevice);
    if (e != hipSuccess) return asuka_fail_msg(ASUKA_E_HIP, (std::string("hipMemcpy: ") + hipGetErrorString(e)).c_str());
  }
  return ASUKA_OK;
}

int check_basis(const asuka_basis_desc* bd, const char* what) {
  if (!bd || bd->nshell <= 0 || !bd->shell_cxyz || !bd->shell_prim_start || !bd->shell_nprim || !bd->shell_l ||
      !bd->shell_ao_start || !bd->prim_exp || !bd->prim_coef)
    return asuka_fail_msg(ASUKA_E_INVALID, (std::string(what) + " basis arrays must be non-null").c_str());
  for (int i = 0; i < bd->nshell; ++i) {
    const int l = bd->shell_l[i], ps = bd->shell_prim_start[i], np = bd->shell_nprim[i];
    if (l < 0) return asuka_fail_msg(ASUKA_E_INVALID, "shell_l must be >= 0");
    if (l > ASUKA_LMAX)
      return asuka_fail_msg(ASUKA_E_UNSUPPORTED,
                            (std::string(what) + " shells support only l <= " + std::to_string(ASUKA_LMAX)).c_str());
    if (np <= 0 || ps < 0 || ps + np > bd->nprim)
      return asuka_fail_msg(ASUKA_E_INVALID, "shell primitive range out of bounds");
  }
  return ASUKA_OK;
}

int hip_fail(const char* what, hipError_t e) {
  return asuka_fail_msg(ASUKA_E_HIP, (std::string(what) + ": " + hipGetErrorString(e)).c_str());
}

// The launches of a call over the context's streams (asuka_df_ctx::side).
struct Fan {
  asuka_df_ctx* ctx;
  hipStream_t s;
  std::lock_guard<std::mutex> lk;
  int n = 0;
  Fan(asuka_df_ctx* c, hipStream_t st) : ctx(c), s(st), lk(c->mu) {}
  hipError_t fork() {
    hipError_t e = hipEventRecord(ctx->ev_fork, s);
    for (int k = 0; k < asuka_df_ctx::kSide && e == hipSuccess; ++k) e = hipStreamWaitEvent(ctx->side[k], ctx->ev_fork, 0);
    return e;
  }
  hipStream_t next() {
    const int k = n++ % (asuka_df_ctx::kSide + 1);
    return k ? ctx->side[k - 1] : s;
  }
  hipError_t join() {
    hipError_t r = hipSuccess;
    for (int k = 0; k < asuka_df_ctx::kSide; ++k) {
      hipError_t e = hipEventRecord(ctx->ev_join[k], ctx->side[k]);
      if (e == hipSuccess) e = hipStreamWaitEvent(s, ctx->ev_join[k], 0);
      if (r == hipSuccess) r = e;
    }
    return r;
  }
};

// One class (la lb|lc) of the bra pairs in w against the auxiliary shells of lc.
int run_class(const asuka_df_ctx* ctx, int la, int lb, int lc, asuka_df::DfWork w, const char* what, Fan& fan) {
  w.aux = ctx->d_aux + ctx->aux_off[lc];
  w.naux = ctx->aux_off[lc + 1] - ctx->aux_off[lc];
  if (w.nbra <= 0 || w.naux <= 0) return ASUKA_OK;
  asuka_df::DfLauncher f = nullptr;
  for (auto fn : {find_df_p0, find_df_p1, find_df_p2, find_df_p3})
    if (!f) f = fn(la, lb, lc);
  if (!f) return asuka_fail_msg(ASUKA_E_UNSUPPORTED, (std::string(what) + ": no kernel for this class").c_str());
  const hipError_t e = f(ctx->dev, w, fan.next());
  return e == hipSuccess ? ASUKA_OK : hip_fail(what, e);
}

}  // namespace

extern "C" {

int asuka_df_ctx_create(const asuka_basis_desc* ao, const asuka_basis_desc* aux, void* stream, asuka_df_ctx** out) {
  (void)stream;
  if (!out) return asuka_fail_msg(ASUKA_E_INVALID, "out must be non-null");
  *out = nullptr;
  int rc;
  if ((rc = check_basis(ao, "AO"))) return rc;
  if ((rc = check_basis(aux, "auxiliary"))) return rc;
  auto ctx = std::make_unique<asuka_df_ctx>();
  {
    hipError_t e = hipEventCreateWithFlags(&ctx->ev_fork, hipEventDisableTiming);
    for (int k = 0; k < asuka_df_ctx::kSide && e == hipSuccess; ++k) {
      e = hipStreamCreateWithFlags(&ctx->side[k], hipStreamNonBlocking);
      if (e == hipSuccess) e = hipEventCreateWithFlags(&ctx->ev_join[k], hipEventDisableTiming);
    }
    if (e != hipSuccess) return asuka_fail_msg(ASUKA_E_HIP, (std::string("streams: ") + hipGetErrorString(e)).c_str());
  }
  const int nsa = ao->nshell, nsx = aux->nshell;
  ctx->nsh_ao = nsa;
  ctx->nsh_aux = nsx;
  // shells: AO shells, auxiliary shells (shell_ao = auxiliary function index), the unit s shell
  std::vector<double> xyz;
  std::vector<int> sl, sao;
  for (int i = 0; i < nsa; ++i) {
    for (int k = 0; k < 3; ++k) xyz.push_back(ao->shell_cxyz[3 * i + k]);
    sl.push_back(ao->shell_l[i]);
    sao.push_back(ao->shell_ao_start[i]);
    ctx->lmax_ao = std::max(ctx->lmax_ao, ao->shell_l[i]);
    ctx->nao = std::max(ctx->nao, ao->shell_ao_start[i] + ncart_c(ao->shell_l[i]));
  }
  for (int i = 0; i < nsx; ++i) {
    for (int k = 0; k < 3; ++k) xyz.push_back(aux->shell_cxyz[3 * i + k]);
    sl.push_back(aux->shell_l[i]);
    sao.push_back(aux->shell_ao_start[i]);
    ctx->lmax_aux = std::max(ctx->lmax_aux, aux->shell_l[i]);
    ctx->naux = std::max(ctx->naux, aux->shell_ao_start[i] + ncart_c(aux->shell_l[i]));
  }
  const int unit = nsa + nsx;
  for (int k = 0; k < 3; ++k) xyz.push_back(0.0);
  sl.push_back(0);
  sao.push_back(0);
  // shell pairs: the AO pairs with l_A >= l_B (asuka/cueri/shell_pairs.py:72-116), then (P, unit)
  std::vector<int> spA, spB, pps, ppc;
  std::vector<PrimPair> pp;
  for (int i = 0; i < nsa; ++i)
    for (int j = 0; j <= i; ++j) {
      int A = i, B = j;
      if (ao->shell_l[i] < ao->shell_l[j]) std::swap(A, B);
      spA.push_back(A);
      spB.push_back(B);
      pps.push_back((int)pp.size());
      const double* a3 = ao->shell_cxyz + 3 * A;
      const double* b3 = ao->shell_cxyz + 3 * B;
      const double dx = a3[0] - b3[0], dy = a3[1] - b3[1], dz = a3[2] - b3[2];
      const double AB2 = dx * dx + dy * dy + dz * dz;
      std::map<double, size_t> by_eta;  // one centre: primitive pairs of equal eta differ in cK alone, merged
      for (int ia = 0; ia < ao->shell_nprim[A]; ++ia)
        for (int ib = 0; ib < ao->shell_nprim[B]; ++ib) {
          const int pA = ao->shell_prim_start[A] + ia, pB = ao->shell_prim_start[B] + ib;
          const double al = ao->prim_exp[pA], be = ao->prim_exp[pB];
          const double eta = al + be, ie = 1.0 / eta;
          PrimPair r;
          r.eta = eta;
          r.Px = (al * a3[0] + be * b3[0]) * ie;
          r.Py = (al * a3[1] + be * b3[1]) * ie;
          r.Pz = (al * a3[2] + be * b3[2]) * ie;
          r.cK = ao->prim_coef[pA] * ao->prim_coef[pB] * std::exp(-(al * be) * ie * AB2);
          r.a_exp = al;
          r.b_exp = be;
          r.inv_eta = ie;
          if (r.cK == 0.0) continue;
          if (AB2 == 0.0) {
            r.Px = a3[0], r.Py = a3[1], r.Pz = a3[2];
            const auto f = by_eta.emplace(eta, pp.size());
            if (!f.second) {
              pp[f.first->second].cK += r.cK;
              continue;
            }
          }
          pp.push_back(r);
        }
      ppc.push_back((int)pp.size() - pps.back());
    }
  ctx->nsp_ao = (int)spA.size();
  for (int i = 0; i < nsx; ++i) {
    spA.push_back(nsa + i);
    spB.push_back(unit);
    pps.push_back((int)pp.size());
    for (int k = 0; k < aux->shell_nprim[i]; ++k) {
      const int p = aux->shell_prim_start[i] + k;
      PrimPair r;
      r.eta = aux->prim_exp[p];
      r.Px = aux->shell_cxyz[3 * i];
      r.Py = aux->shell_cxyz[3 * i + 1];
      r.Pz = aux->shell_cxyz[3 * i + 2];
      r.cK = aux->prim_coef[p];
      r.a_exp = aux->prim_exp[p];
      r.b_exp = 0.0;
      r.inv_eta = 1.0 / aux->prim_exp[p];
      if (r.cK != 0.0) pp.push_back(r);
    }
    ppc.push_back((int)pp.size() - pps.back());
  }
  std::vector<void*>& own = ctx->owned;
  double* d_xyz;
  int *d_l, *d_ao, *d_spA, *d_spB, *d_pps, *d_ppc, *d_mol;
  PrimPair* d_pp;
  if ((rc = upload(&d_xyz, xyz, own))) return rc;
  if ((rc = upload(&d_l, sl, own))) return rc;
  if ((rc = upload(&d_ao, sao, own))) return rc;
  if ((rc = upload(&d_spA, spA, own))) return rc;
  if ((rc = upload(&d_spB, spB, own))) return rc;
  if ((rc = upload(&d_pps, pps, own))) return rc;
  if ((rc = upload(&d_ppc, ppc, own))) return rc;
  if ((rc = upload(&d_pp, pp, own))) return rc;
  if ((rc = upload(&d_mol, std::vector<int>(sl.size(), 0), own))) return rc;
  {  // work lists of the kernels
    std::vector<int> bra, auxl;
    for (int la = 0; la <= ASUKA_LMAX; ++la)
      for (int lb = 0; lb <= la; ++lb) {
        const size_t first = bra.size();
        for (int sp = 0; sp < ctx->nsp_ao; ++sp)
          if (sl[spA[sp]] == la && sl[spB[sp]] == lb) bra.push_back(sp);
        std::stable_sort(bra.begin() + first, bra.end(), [&](int x, int y) { return ppc[x] > ppc[y]; });
        ctx->bra_off[la * (la + 1) / 2 + lb + 1] = (int)bra.size();
      }
    for (int l = 0; l <= ASUKA_LMAX; ++l) {
      for (int i = 0; i < nsx; ++i)
        if (sl[nsa + i] == l) auxl.push_back(ctx->nsp_ao + i);
      ctx->aux_off[l + 1] = (int)auxl.size();
    }
    if ((rc = upload(&ctx->d_bra, bra, own))) return rc;
    if ((rc = upload(&ctx->d_aux, auxl, own))) return rc;
  }
  DevBasis& dv = ctx->dev;
  dv.shell_xyz = d_xyz;
  dv.shell_l = d_l;
  dv.shell_ao = d_ao;
  dv.sp_A = d_spA;
  dv.sp_B = d_spB;
  dv.pp_start = d_pps;
  dv.pp_count = d_ppc;
  dv.pp_count0 = d_ppc;
  dv.pp = d_pp;
  dv.shell_mol = d_mol;
  dv.nao = ctx->nao;
  dv.nsp = (int)spA.size();
  *out = ctx.release();
  return ASUKA_OK;
}

int asuka_df_ctx_destroy(asuka_df_ctx* ctx) {
  delete ctx;
  return ASUKA_OK;
}

int asuka_df_ctx_info(const asuka_df_ctx* ctx, int64_t out[4]) {
  if (!ctx || !out) return asuka_fail_msg(ASUKA_E_INVALID, "ctx and out must be non-null");
  out[0] = ctx->nao;
  out[1] = ctx->naux;
  out[2] = ctx->nsp_ao;
  out[3] = ctx->nsh_aux;
  return ASUKA_OK;
}

int asuka_df_metric(asuka_df_ctx* ctx, double* V, void* stream) {
  if (!ctx || !V) return asuka_fail_msg(ASUKA_E_INVALID, "ctx and V must be non-null");
  Fan fan(ctx, (hipStream_t)stream);
  hipError_t e = fan.fork();
  if (e != hipSuccess) return hip_fail("metric", e);
  int rc = ASUKA_OK;
  for (int la = ctx->lmax_aux; la >= 0; --la)
    for (int lc = ctx->lmax_aux; lc >= 0 && rc == ASUKA_OK; --lc) {
      asuka_df::DfWork w{};
      w.bra = ctx->d_aux + ctx->aux_off[la];
      w.nbra = ctx->aux_off[la + 1] - ctx->aux_off[la];
      w.out = V;
      w.sa = ctx->naux;
      w.sc = 1;  // the unit function's index 0: no sb
      rc = run_class(ctx, la, 0, lc, w, "metric", fan);
    }
  e = fan.join();  // also after a failed launch: the caller's stream waits for what was queued
  return rc ? rc : e == hipSuccess ? ASUKA_OK : hip_fail("metric", e);
}

int asuka_df_int3c2e(asuka_df_ctx* ctx, double* X, void* stream) {
  if (!ctx || !X) return asuka_fail_msg(ASUKA_E_INVALID, "ctx and X must be non-null");
  Fan fan(ctx, (hipStream_t)stream);
  hipError_t e = fan.fork();
  if (e != hipSuccess) return hip_fail("int3c2e", e);
  int rc = ASUKA_OK;
  for (int la = ctx->lmax_ao; la >= 0; --la)
    for (int lb = la; lb >= 0; --lb)
      for (int lc = ctx->lmax_aux; lc >= 0 && rc == ASUKA_OK; --lc) {
        const int c = la * (la + 1) / 2 + lb;
        asuka_df::DfWork w{};
        w.bra = ctx->d_bra + ctx->bra_off[c];
        w.nbra = ctx->bra_off[c + 1] - ctx->bra_off[c];
        w.out = X;
        w.sa = ctx->nao;
        w.sb = 1;
        w.sc = (long long)ctx->nao * ctx->nao;
        w.mirror = 1;
        rc = run_class(ctx, la, lb, lc, w, "int3c2e", fan);
      }
  e = fan.join();
  return rc ? rc : e == hipSuccess ? ASUKA_OK : hip_fail("int3c2e", e);
}

}  // extern "C"
