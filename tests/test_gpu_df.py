"""GPU parity of the density-fitting path through the C ABI.

* the auxiliary metric (P|Q) and the three-centre integrals (mu nu|P)
  (asuka_df_metric, asuka_df_int3c2e) against the oracle's tiles, 1e-12
  absolute, for the water monomer and (H2O)2 with cc-pVDZ and the
  even-tempered auxiliary set, and for a cc-pVTZ monomer (f AO shells);
* DF J and K from the whitened tensor against the oracle's DF J/K, 1e-10;
* the DF RHF energy against the oracle's RHF with DF Fock matrices, 1e-9 Eh.
"""

import numpy as np
import pytest

from asuka_amd.basis import build_ao_basis_cart
from asuka_amd.molecule import water_cluster, water_monomer

pytestmark = pytest.mark.gpu


def _bases(mol, basis):
    from asuka_amd.df import build_aux_basis_cart

    ao, _ = build_ao_basis_cart(mol)
    return ao, build_aux_basis_cart(mol, None, basis)


@pytest.mark.parametrize("case", ["h2o_dz", "h2o2_dz", "h2o_tz"])
def test_df_integrals_against_oracle(gpu, oracle, case):
    from asuka_amd.df import make_df_context

    mol, basis = {"h2o_dz": (water_monomer("cc-pVDZ"), "cc-pVDZ"),
                  "h2o2_dz": (water_cluster(2, 2, "cc-pVDZ"), "cc-pVDZ"),
                  "h2o_tz": (water_monomer("cc-pVTZ"), "cc-pVTZ")}[case]
    print(f"\n[df] integrals {case}", flush=True)
    ao, aux = _bases(mol, basis)
    ctx = make_df_context(ao, aux)
    assert ctx.nao == ao.nao and ctx.naux == aux.nao
    X = ctx.int3c2e_Q().cpu().numpy()
    V = ctx.metric().cpu().numpy()
    X0, V0 = oracle.df_integrals(ao, aux, hp=True)
    assert np.abs(V - V0).max() < 1e-12 * max(1.0, np.abs(V0).max())
    assert np.abs(X - X0).max() < 1e-12 * max(1.0, np.abs(X0).max())


def test_df_jk_and_scf_against_oracle(gpu, oracle):
    from asuka_amd.df import df_JK, df_tensors
    from asuka_amd.frontend import run_hf_df

    torch = gpu
    mol = water_cluster(2, 2, "cc-pVDZ")
    print("\n[df] J/K (H2O)2 cc-pVDZ", flush=True)
    ao, aux = _bases(mol, "cc-pVDZ")
    C = np.random.default_rng(6).standard_normal((ao.nao, 10))
    C, _ = np.linalg.qr(C)
    D = 2.0 * C @ C.T
    _, V, L, BQ = df_tensors(ao, aux)
    J, K = df_JK(BQ, torch.as_tensor(D, device="cuda"))
    X0, V0 = oracle.df_integrals(ao, aux, hp=True)
    J0, K0 = oracle.df_JK(X0, V0, D)
    assert np.abs(J.cpu().numpy() - J0).max() < 1e-10
    assert np.abs(K.cpu().numpy() - K0).max() < 1e-10
    print("[df] RHF water monomer", flush=True)
    mol = water_monomer("cc-pVDZ")
    res = run_hf_df(mol, two_e_backend="df")
    assert res.two_e_backend == "df" and res.scf.converged
    ao, aux = _bases(mol, "cc-pVDZ")
    X0, V0 = oracle.df_integrals(ao, aux, hp=True)
    S, T, Vn = oracle.int1e(ao, mol.coords_bohr, mol.charges)
    h = T + Vn

    def fock(Dm):
        Jd, Kd = oracle.df_JK(X0, V0, Dm)
        F = h + Jd - 0.5 * Kd
        return 0.5 * (F + F.T)

    ref = oracle.rhf(S, h, fock, mol.nelectron, mol.energy_nuc())
    assert abs(res.scf.e_tot - ref["e_tot"]) < 1e-9
    # the DF energy is close to the exact (direct) one
    e_direct = run_hf_df(mol, two_e_backend="direct").scf.e_tot
    assert abs(res.scf.e_tot - e_direct) < 2e-3


@pytest.mark.parametrize("naux,nao", [(1145, 125), (1374, 150), (3, 2000)])
def test_whitening_in_several_solves(gpu, naux, nao):
    """Right-hand sides beyond one solve's share (the last part ragged): L B = X
    to rounding, and the first columns as one solve gives them."""
    from asuka_amd.df import whiten_3c2e

    torch = gpu
    g = torch.Generator(device="cuda").manual_seed(naux)
    A = torch.randn(naux, naux, dtype=torch.float64, device="cuda", generator=g)
    L = torch.linalg.cholesky(A @ A.T / naux + torch.eye(naux, dtype=torch.float64, device="cuda"))
    X = torch.randn(naux, nao, nao, dtype=torch.float64, device="cuda", generator=g)
    B = whiten_3c2e(X, L)
    assert B.shape == X.shape
    assert float((L @ B.reshape(naux, -1) - X.reshape(naux, -1)).abs().max()) < 1e-12
    one = torch.linalg.solve_triangular(L, X[:, 0, :].contiguous(), upper=False)
    assert float((B[:, 0, :] - one).abs().max()) < 1e-12


def test_df_scf_of_five_waters(gpu):
    """The default backend beyond one solve's share, near the direct energy."""
    from asuka_amd.frontend import run_hf_df

    mol = water_cluster(5, 3, "cc-pVDZ")
    df = run_hf_df(mol, two_e_backend="df").scf
    direct = run_hf_df(mol, two_e_backend="direct").scf
    assert df.converged and abs(df.e_tot - direct.e_tot) < 5 * 2e-3
