"""Wave units cut into slices of their primitive quartets (small contexts):
contractions that leave only the bra, only the ket, both or neither to cut,
counts around the cut sizes, with and without primitive screening, in J/K
(FP64, mixed and reproducible) and in the derivative kernels, against the
oracle. 1e-10 as in the other J/K tests: the slices only regroup sums."""

import numpy as np
import pytest

from asuka_amd.basis import pack_cart_basis, parse_basis_dict

pytestmark = pytest.mark.gpu


def _contraction(l, n, lo=0.25, ratio=1.9):
    return [l] + [[lo * ratio ** k, 0.2 + 0.6 / (1 + k)] for k in range(n)]


def _case(ns, np_, nd):
    """Two centres: s, p and d shells of ns, np_ and nd primitives, and an uncontracted s."""
    spec = {"O": [_contraction(0, ns), _contraction(1, np_)] + ([_contraction(2, nd, 0.7)] if nd else []),
            "H": [_contraction(0, 1, 0.4), _contraction(0, ns, 0.3, 2.3)]}
    atoms = [("O", np.array([0.1, -0.2, 0.05])), ("H", np.array([0.3, 0.4, 1.6]))]
    return pack_cart_basis(atoms, parse_basis_dict(spec, ["H", "O"])), np.array([x for _, x in atoms])


CASES = [(1, 1, 0), (3, 2, 1), (7, 1, 0), (8, 5, 0), (17, 3, 2)]


@pytest.mark.parametrize("ns,np_,nd", CASES)
@pytest.mark.parametrize("eps", [0.0, 1e-14])
def test_sliced_jk(gpu, oracle, ns, np_, nd, eps):
    from asuka_amd.hf.direct_jk import direct_JK, make_direct_jk_context

    ao, _ = _case(ns, np_, nd)
    n = ao.nao
    D = np.random.default_rng(n).standard_normal((n, n))
    D = 0.5 * (D + D.T)
    octx = oracle.make_context(ao)
    Jr, Kr = oracle.dense_JK(oracle.dense_eri(octx), D)
    ctx = make_direct_jk_context(ao, eps_schwarz=eps, eps_density=0.0)
    scale = max(1.0, np.abs(Jr).max())
    for kw in ({}, {"deterministic": True}, {"mixed_precision": True}):
        stats = {}
        J, K = direct_JK(ctx, D, stats=stats, **kw)
        tol = (1e-5 if kw.get("mixed_precision") else 1e-10) * scale
        assert np.abs(J.cpu().numpy() - Jr).max() < tol and np.abs(K.cpu().numpy() - Kr).max() < tol
        # the counters take a quartet by its first slice alone
        assert stats["direct_jk_evaluated"] == ctx.ntasks


@pytest.mark.parametrize("ns,np_,nd", CASES)
def test_sliced_gradient(gpu, oracle, ns, np_, nd):
    from asuka_amd.hf.direct_jk import make_direct_jk_context
    from asuka_amd.hf.grad import direct_jk_grad

    ao, xyz = _case(ns, np_, nd)
    n = ao.nao
    rng = np.random.default_rng(n)
    D, WJ, WK = (0.5 * (X + X.T) for X in rng.standard_normal((3, n, n)))
    ref = oracle.grad2e(oracle.make_context(ao), D, WJ, WK, ao.shell_atom, 2, hp=False, threads=0)
    for eps in (0.0, 1e-14):
        ctx = make_direct_jk_context(ao, eps_schwarz=eps, eps_density=0.0, atom_coords_bohr=xyz,
                                     atom_charges=np.array([8.0, 1.0]))
        g = direct_jk_grad(ctx, D, WJ, WK).cpu().numpy()
        assert np.abs(g - ref).max() < 1e-10 * max(1.0, np.abs(ref).max())


def test_slices_skip_the_same_primitive_quartets(gpu):
    """A 4-water cluster alone (cut into slices) and beside a 12-water one in a
    batch (whose units are longer, so it is cut less) leave out the same
    primitive quartets. The sums then differ by their order alone: about 4e4
    terms into elements up to 1e2, under 2e-12 in the positions drawn here."""
    import torch

    from asuka_amd.basis import build_ao_basis_cart
    from asuka_amd.hf.direct_jk import direct_JK_batched, make_direct_jk_batch_context, make_direct_jk_context
    from asuka_amd.molecule import water_cluster

    aos, Ds = [], []
    for n, seed in ((4, 3), (12, 17)):
        ao, _ = build_ao_basis_cart(water_cluster(n, 1000 + seed, "cc-pVDZ"))
        C, _ = np.linalg.qr(np.random.default_rng(2000 + seed).standard_normal((ao.nao, 5 * n)))
        aos.append(ao)
        Ds.append(torch.tensor(2.0 * C @ C.T, device="cuda"))
    batch = direct_JK_batched(make_direct_jk_batch_context(aos, eps_schwarz=1e-12), Ds)
    alone = direct_JK_batched([make_direct_jk_context(ao, eps_schwarz=1e-12) for ao in aos], Ds)
    for a, b in zip(batch, alone):
        for x, y in zip(a, b):
            assert float((x - y).abs().max()) < 2e-12
