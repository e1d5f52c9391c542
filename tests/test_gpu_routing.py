"""Mixed builds: which class pairs are split into an FP64 and an FP32 launch.
By default only those with enough work; with the FP32 cut given by the caller
all of them. A small molecule's default mixed build is then the FP64 build
(equal to the order of its sums), and one with both kinds of class pairs stays
within the mixed bound of it."""

import numpy as np
import pytest

from asuka_amd.basis import build_ao_basis_cart
from asuka_amd.molecule import water_cluster

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,basis,tau,split", [(1, "cc-pVDZ", 0.0, "none"), (3, "cc-pVDZ", 1e-5, "some"),
                                                (7, "cc-pVDZ", 0.0, "some"), (2, "cc-pVTZ", 1e3, "all")])
def test_split_class_pairs(gpu, n, basis, tau, split):
    from asuka_amd.hf.direct_jk import direct_fock_rhf, direct_JK, make_direct_jk_context

    ao, _ = build_ao_basis_cart(water_cluster(n, 5, basis))
    ctx = make_direct_jk_context(ao, tau_mixed=tau)
    C = np.linalg.qr(np.random.default_rng(n).standard_normal((ao.nao, 5 * n)))[0]
    D = 2.0 * C @ C.T
    st = {}
    J, K = direct_JK(ctx, D, mixed_precision=True, stats=st)
    J0, K0 = direct_JK(ctx, D, mixed_precision=False)
    q32, q = sum(c["quartets_fp32"] for c in st["class_counts"]), st["direct_jk_evaluated"]
    assert (q32 == 0) if split == "none" else q32 > 0
    if split == "all":  # every quartet of the register kernels' classes
        assert all(c["quartets_fp32"] == c["bins"].sum() for c in st["class_counts"] if c["prim_quartets_evaluated"])
    assert q32 <= q
    tol = {"none": 1e-12, "some": 1e-8, "all": 1e-5}[split]
    assert float((J - J0).abs().max()) < tol and float((K - K0).abs().max()) < tol
    h = np.eye(ao.nao)
    F, F0 = (direct_fock_rhf(ctx, D, h, mixed_precision=m) for m in (True, False))
    assert float((F - F0).abs().max()) < 2 * tol


def test_split_does_not_depend_on_the_batch(gpu):
    """Default mixed builds of a batch equal those of one-molecule contexts to
    the order of the FP64 sums (fewer than 1e5 terms below 10 in elements below
    1e2: 1e-12), with molecules that split none, some and most of their class
    pairs; with the class pairs' sizes taken over the batch, or FP32 units
    sliced by its work, they differ by 1e-11 to 1e-10."""
    import torch

    from asuka_amd.hf.direct_jk import direct_JK, direct_JK_batched, make_direct_jk_batch_context, \
        make_direct_jk_context

    aos, Ds = [], []
    for n, seed in ((1, 8), (4, 3), (12, 17), (3, 2)):
        ao, _ = build_ao_basis_cart(water_cluster(n, 1000 + seed, "cc-pVDZ"))
        C, _ = np.linalg.qr(np.random.default_rng(2000 + seed).standard_normal((ao.nao, 5 * n)))
        aos.append(ao)
        Ds.append(torch.tensor(2.0 * C @ C.T, device="cuda"))
    batch = direct_JK_batched(make_direct_jk_batch_context(aos), Ds, mixed_precision=True)
    q32 = []
    for ao, D, got in zip(aos, Ds, batch):
        st = {}
        ref = direct_JK(make_direct_jk_context(ao), D, mixed_precision=True, stats=st)
        q32.append(sum(c["quartets_fp32"] for c in st["class_counts"]))
        assert all(float((x - y).abs().max()) < 1e-12 for x, y in zip(got, ref)), ao.nao
    assert q32[0] == 0 < q32[1] < q32[2]
