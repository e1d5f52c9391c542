"""The density-fitting kernels where their lanes and groups end: 1, 63, 64, 65
and 130 auxiliary shells of one l, contracted auxiliary shells, a bra pair
without primitives, and f shells on both sides, against the oracle's tiles
(1e-12 of the largest, as in the other density-fitting tests)."""

import numpy as np
import pytest

from asuka_amd.basis import pack_cart_basis, parse_basis_dict

pytestmark = pytest.mark.gpu

ATOMS = [("O", np.array([0.0, 0.1, -0.2])), ("H", np.array([0.4, -0.3, 1.5]))]
AO = {"O": [[0, [9.0, 0.2, 0.1], [2.0, 0.5, 0.0], [0.5, 0.6, 1.0]], [1, [1.2, 0.5], [0.4, 0.7]], [3, [0.9, 1.0]]],
      "H": [[0, [0.7, 1.0]], [2, [0.8, 1.0]]]}


def _pack(spec, atoms=ATOMS):
    return pack_cart_basis(atoms, parse_basis_dict(spec, sorted({s for s, _ in atoms})))


@pytest.mark.parametrize("n", [1, 63, 64, 65, 130])
def test_lane_edges(gpu, oracle, n):
    from asuka_amd.df import make_df_context

    ao = _pack(AO)
    # n s shells in all, and p, d, f shells of which some are contracted
    aux = _pack({"O": [[0, [0.3 * 1.06 ** k, 1.0]] for k in range(n - 1)] + [[1, [1.5, 0.4], [0.6, 0.8]], [2, [0.8, 1.0]]],
                 "H": [[0, [2.0, 0.3], [0.9, 0.4], [0.4, 0.5]], [3, [0.7, 1.0]]]})
    ctx = make_df_context(ao, aux)
    X0, V0 = oracle.df_integrals(ao, aux, hp=True)
    X = gpu.full((aux.nao, ao.nao, ao.nao), float("nan"), dtype=gpu.float64, device="cuda")
    V = gpu.full((aux.nao, aux.nao), float("nan"), dtype=gpu.float64, device="cuda")
    ctx.int3c2e_Q(out=X)
    ctx.metric(out=V)
    assert np.abs(V.cpu().numpy() - V0).max() < 1e-12 * max(1.0, np.abs(V0).max())
    assert np.abs(X.cpu().numpy() - X0).max() < 1e-12 * max(1.0, np.abs(X0).max())


def test_pairs_without_primitives_are_zero(gpu):
    """Two atoms 200 Bohr apart: the products of their functions underflow to exact zeros, which must be written."""
    from asuka_amd.df import make_df_context

    atoms = [("O", np.zeros(3)), ("H", np.array([0.0, 0.0, 200.0]))]
    ao = _pack(AO, atoms)
    ctx = make_df_context(ao, _pack({"O": [[0, [1.0, 1.0]]], "H": [[1, [1.0, 1.0]]]}, atoms))
    X = gpu.full((ctx.naux, ao.nao, ao.nao), float("nan"), dtype=gpu.float64, device="cuda")
    ctx.int3c2e_Q(out=X)
    x = X.cpu().numpy()
    n_o = int(ao.shell_ao_start[int(np.nonzero(ao.shell_atom == 1)[0][0])])
    assert np.isfinite(x).all() and (x[:, :n_o, n_o:] == 0.0).all() and (x[:, n_o:, :n_o] == 0.0).all()
