"""LDS-class Jacobi of orders up to 16 (matrix in registers) against LAPACK:
every order, graded and rank-deficient matrices, equal eigenvalues, a zero
matrix, a non-finite one, and the same bits alone and among others."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

EPS = float(np.finfo(np.float64).eps)


def matrices(g):
    rng = np.random.default_rng(g)
    X = rng.standard_normal((g, 2 * g))
    yield X @ X.T
    D = np.logspace(0, -7, g)
    yield (D[:, None] * X) @ (D[:, None] * X).T
    Y = X[:, :max(1, g // 3)]
    yield Y @ Y.T
    Q = np.linalg.qr(rng.standard_normal((g, g)))[0]
    d = np.repeat([3.0, 1.0], [g // 2, g - g // 2])
    yield (Q * d) @ Q.T
    yield np.zeros((g, g))


@pytest.mark.parametrize("g", range(1, 17))
def test_against_lapack(g):
    import torch

    from syngular_amd import ops

    mats = [0.5 * (m + m.T) for m in matrices(g)]
    dev = [torch.tensor(m, device="cuda") for m in mats]
    together = ops.jacobi_gram_many(dev)
    for G, D, (rt, s) in zip(mats, dev, together):
        rt1, s1 = ops.jacobi_gram_many([D])[0]
        assert torch.equal(rt, rt1) and torch.equal(s, s1)
        V, lam = rt.cpu().numpy(), s.cpu().numpy() ** 2
        ref = np.clip(np.linalg.eigvalsh(G)[::-1], 0.0, None)
        top = max(ref[0], 1e-300)
        # a few sweeps of rotations, each of a few eps
        assert np.all(np.diff(lam) <= 1e-15 * top)
        assert np.abs(lam - ref).max() <= 50 * g * EPS * top
        assert np.abs(V @ V.T - np.eye(g)).max() <= 100 * g * EPS
        assert np.linalg.norm(V.T @ (lam[:, None] * V) - G) <= 100 * g * EPS * np.linalg.norm(G)


def test_non_finite_ends():
    import torch

    from syngular_amd import ops

    G = torch.eye(7, dtype=torch.float64, device="cuda")
    G[2, 3] = G[3, 2] = float("nan")
    rt, s = ops.jacobi_gram_many([G])[0]
    torch.cuda.synchronize()
    assert rt.shape == (7, 7) and s.shape == (7,)
