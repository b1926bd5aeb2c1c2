"""Direct phase of the blocked Gram eigen-solver (tridiagonal reduction and
divide and conquer) against numpy.linalg.eigh, at the edges of its size
classes, leaves and reflector blocks and on the spectra that deflate."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
EPS = np.finfo(np.float64).eps


def spectra(kind, n, rng):
    if kind == "full":
        C = rng.standard_normal((n + 5, n))
    elif kind == "rank":                   # a null space of n - n // 3
        C = rng.standard_normal((n, n // 3)) @ rng.standard_normal((n // 3, n))
    elif kind == "graded":                 # eigenvalues over eight decades
        C = rng.standard_normal((n + 5, n)) * np.logspace(0, -4, n)
    elif kind == "cluster":                # three distinct eigenvalues
        q = np.linalg.qr(rng.standard_normal((n, n)))[0]
        C = np.sqrt(rng.choice([1.0, 2.0, 3.0], n))[:, None] * q
    elif kind == "diagonal":
        C = np.diag(np.sqrt(1.0 + rng.permutation(n)))
    elif kind == "one":                    # rank one
        C = rng.standard_normal((1, n))
    elif kind == "zero":
        C = np.zeros((1, n))
    else:                                  # scaled far from one
        C = float(kind) * rng.standard_normal((n + 5, n))
    return C.T @ C


# a matrix goes through reduction, divide and conquer and products of n-term
# sums: residuals of a modest multiple of n eps, as the Jacobi tests allow
@pytest.mark.parametrize("kind", ["full", "rank", "graded", "cluster", "diagonal", "one", "zero", "1e-100", "1e100"])
def test_direct_eigen_sizes(kind):
    import torch

    from syngular_amd import batch as B

    rng = np.random.default_rng(len(kind))
    orders = [17, 18, 31, 32, 33, 34, 35, 63, 64, 65, 66, 67, 97, 127, 128, 129, 130, 161, 255, 257, 290, 383, 384, 385]
    Gs = [spectra(kind, n, rng) for n in orders]
    dev = torch.device("cuda")
    G = [torch.tensor(x, device=dev) for x in Gs]
    R = [torch.empty_like(x) for x in G]
    S = [torch.empty(x.shape[0], dtype=torch.float64, device=dev) for x in G]
    ptr = lambda ts: np.array([t.data_ptr() for t in ts], dtype=np.uint64)
    B.jacobi_gram_blocked_table(ptr(G), np.array(orders, np.int64), ptr(R), ptr(S))
    torch.cuda.synchronize()
    for n, g0, g1, r, s in zip(orders, Gs, G, R, S):
        g1, r, s = g1.cpu().numpy(), r.cpu().numpy(), s.cpu().numpy()
        w = np.linalg.eigvalsh(g0)[::-1]
        top = max(w[0], 0.0)
        bound = 8 * n * EPS
        assert np.all(np.diff(s) <= 0), n
        np.testing.assert_allclose(r @ r.T, np.eye(n), atol=bound, err_msg=str(n))
        np.testing.assert_allclose(s ** 2, w.clip(0), atol=bound * top, rtol=0, err_msg=str(n))
        np.testing.assert_allclose((r.T * s ** 2) @ r, g0, atol=bound * top, rtol=0, err_msg=str(n))
        # diagonalised in place
        assert np.abs(g1 - np.diag(np.diag(g1))).max() <= bound * top, n


def test_direct_eigen_alone_and_in_a_mix():
    """A matrix gives the same result alone and beside others of every size."""
    import torch

    from syngular_amd import ops
    from syngular_amd import batch as B

    rng = np.random.default_rng(5)
    orders = [40, 100, 200, 300, 40]
    Gs = [spectra("full", n, rng) for n in orders]
    dev = torch.device("cuda")
    G = [torch.tensor(x, device=dev) for x in Gs]
    R = [torch.empty_like(x) for x in G]
    S = [torch.empty(x.shape[0], dtype=torch.float64, device=dev) for x in G]
    ptr = lambda ts: np.array([t.data_ptr() for t in ts], dtype=np.uint64)
    B.jacobi_gram_blocked_table(ptr(G), np.array(orders, np.int64), ptr(R), ptr(S))
    for n, g0, r, s in zip(orders, Gs, R, S):
        rt, sv, _ = ops.jacobi_gram_blocked(torch.tensor(g0, device=dev), tol=B.TOL_BLOCKED)
        assert torch.equal(sv, s) and torch.equal(rt, r), n
