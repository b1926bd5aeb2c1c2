"""Blocked Gram eigen-solver at the edges of its reductions: one block more or
less than a class, orders that leave work-groups without live columns early,
graded spectra, a matrix of few nonzero rows, several matrices a call."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

EPS = float(np.finfo(np.float64).eps)


def check(G, rt, s, what):
    import torch

    n = G.shape[0]
    ref = np.sqrt(np.clip(np.linalg.eigvalsh(G.cpu().numpy())[::-1], 0.0, None))
    top = max(ref[0], 1e-300)
    # eigenvalues to a few n eps of the largest
    assert np.abs(s.cpu().numpy() ** 2 - ref ** 2).max() <= 20 * n * EPS * top ** 2, what
    eye = torch.eye(n, dtype=G.dtype, device=G.device)
    assert float((rt @ rt.t() - eye).abs().max()) <= 20 * n * EPS, what
    assert float((rt.t() @ torch.diag(s * s) @ rt - G).norm()) <= 20 * n * EPS * float(G.norm()) + 1e-300, what


@pytest.mark.parametrize("n", [17, 32, 33, 48, 63, 65, 127, 129, 191, 193, 223, 255, 257, 258, 289, 511, 513, 1023, 1025])
@pytest.mark.parametrize("grade", [0.0, 6.0])
def test_orders(n, grade):
    import torch

    from syngular_amd import ops

    gen = torch.Generator(device="cuda").manual_seed(n)
    X = torch.randn((n, 2 * n), dtype=torch.float64, device="cuda", generator=gen)
    X *= torch.logspace(0, -grade, n, dtype=torch.float64, device="cuda")[:, None]
    G = X @ X.t()
    G = 0.5 * (G + G.t())
    rt, s, _ = ops.jacobi_gram_blocked(G.clone())
    check(G, rt, s, (n, grade))


@pytest.mark.parametrize("n", [40, 200, 300])
def test_few_rows_and_many_matrices(n):
    import torch

    from syngular_amd import batch, ops

    gen = torch.Generator(device="cuda").manual_seed(n)
    X = torch.randn((n, n), dtype=torch.float64, device="cuda", generator=gen)
    X[3:] = 0.0
    G = X @ X.t()
    G = 0.5 * (G + G.t())
    rt, s, _ = ops.jacobi_gram_blocked(G.clone())
    check(G, rt, s, n)
    orders = [n, n - 1, n // 2 + 17, n]
    mats = []
    for m in orders:
        X = torch.randn((m, m + 5), dtype=torch.float64, device="cuda", generator=gen)
        mats.append(0.5 * (X @ X.t() + (X @ X.t()).t()))
    work = [m.clone() for m in mats]
    rts = [torch.empty_like(m) for m in mats]
    ss = [torch.empty(m.shape[0], dtype=torch.float64, device="cuda") for m in mats]
    ptr = lambda ts: np.array([t.data_ptr() for t in ts], np.uint64)   # noqa: E731
    batch.jacobi_gram_blocked_table(ptr(work), np.array(orders, np.int64), ptr(rts), ptr(ss))
    for m, rt, s in zip(mats, rts, ss):
        check(m, rt, s, (n, m.shape[0]))
