"""Density purification (asuka_scf_purify, asuka_scf_tc2_step) at the edges of
its 16 x 16 tiles, of the waves' shares of them and of the one-kernel limit:
the projector of a gapped symmetric matrix against eigh (1e-9: the idempotency
tolerance 1e-11 bounds each eigenvalue's distance from 0 or 1, rounding adds
n eps a step), a fixed number of steps against the same steps in numpy, and
the steps replayed from a graph."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SIZES = [1, 2, 15, 16, 17, 31, 64, 75, 96, 112, 113, 127, 128, 129, 200]


def _matrix(n, seed):
    """Symmetric, with nocc eigenvalues in [-2, -0.5] and the rest in [0.2, 3]."""
    rng = np.random.default_rng(seed)
    nocc = max(1, n // 5) if n > 1 else 1
    e = np.concatenate([rng.uniform(-2.0, -0.5, nocc), rng.uniform(0.2, 3.0, n - nocc)])
    Q = np.linalg.qr(rng.standard_normal((n, n)))[0]
    F = (Q * e) @ Q.T
    return 0.5 * (F + F.T), nocc, Q[:, :nocc] @ Q[:, :nocc].T


def _steps(F, nocc, iters, tol):
    n = len(F)
    d, r = np.diag(F), np.abs(F).sum(1) - np.abs(np.diag(F))
    e0, e1 = (d - r).min(), (d + r).max()
    P, err = (e1 * np.eye(n) - F) / (e1 - e0), np.inf
    for _ in range(iters):
        P2 = P @ P
        err = np.linalg.norm(P2 - P)
        if err < tol:
            break
        P = P2 if np.trace(P) > nocc else 2.0 * P - P2
    return P, err


@pytest.mark.parametrize("n", [k for k in SIZES if k > 1])
def test_projector(gpu, n):
    from asuka_amd.hf import direct_scf as S

    F, nocc, ref = _matrix(n, n)
    Fd = gpu.tensor(F, device="cuda")
    P, k = S._purify_converged(gpu, Fd, nocc)
    assert k > 0 and np.abs(P.cpu().numpy() - ref).max() < 1e-9
    P2, err = S._purify(gpu, Fd, nocc, k + 9)  # frozen: steps past convergence change nothing
    assert float(err) < 1e-11 and np.abs((P2 - P).cpu().numpy()).max() < 1e-12
    assert np.array_equal(P2.cpu().numpy(), P2.cpu().numpy().T)


@pytest.mark.parametrize("n", SIZES)
def test_few_steps_and_replay(gpu, n):
    """Seven steps (not converged; for n = 1 the interval is empty and P undefined in both)."""
    from asuka_amd.hf import direct_scf as S

    F, nocc, _ = _matrix(n, n + 100)
    Fd = gpu.tensor(F, device="cuda")
    with np.errstate(all="ignore"):
        ref, eref = _steps(F, nocc, 7, 1e-11)
    P, err = S._purify(gpu, Fd, nocc, 7)
    np.testing.assert_allclose(P.cpu().numpy(), ref, rtol=0, atol=1e-12)
    if n > 1:
        assert abs(float(err) - eref) < 1e-10
    side = gpu.cuda.Stream()
    side.wait_stream(gpu.cuda.current_stream())
    with gpu.cuda.stream(side):
        S._purify(gpu, Fd, nocc, 7)
    gpu.cuda.current_stream().wait_stream(side)
    g = gpu.cuda.CUDAGraph()
    with gpu.cuda.graph(g):
        Pg, _ = S._purify(gpu, Fd, nocc, 7)
    for s in range(3):  # replays on other inputs, against the eager result
        F2, _, _ = _matrix(n, n + 200 + s)
        Fd.copy_(gpu.tensor(F2, device="cuda"))
        g.replay()
        gpu.cuda.synchronize()
        np.testing.assert_allclose(Pg.cpu().numpy(), S._purify(gpu, Fd, nocc, 7)[0].cpu().numpy(), rtol=0, atol=1e-13)


def test_arguments(gpu):
    from asuka_amd import _lib

    L = _lib.lib()
    x = gpu.zeros(400, device="cuda", dtype=gpu.float64)
    for n, it in ((0, 1), (L.asuka_scf_purify_max() + 1, 1), (4, -1)):
        with pytest.raises(ValueError):
            _lib.check(L.asuka_scf_purify(_lib.ptr(x), n, 1, it, 1e-11, _lib.ptr(x), _lib.ptr(x), _lib.ptr(x), 0))
    with pytest.raises(ValueError):
        _lib.check(L.asuka_scf_tc2_step(_lib.ptr(x), 0, 4, 1, 1e-11, _lib.ptr(x), _lib.ptr(x), 0, _lib.ptr(x), 0))
