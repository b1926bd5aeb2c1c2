"""Gram matrices with nothing to rotate (a bond that no gate has touched) leave
the blocked eigen-solver as they came, alone and beside others."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

TOL = 1e-8


def nearly_diagonal(n, rng):
    """Entries at a tenth of what the rotation test lets through."""
    d = rng.permutation(np.logspace(0, -3, n))
    E = rng.uniform(-0.1, 0.1, (n, n))
    G = TOL * np.sqrt(d[:, None] * d) * 0.5 * (E + E.T)
    np.fill_diagonal(G, d)
    return G


@pytest.mark.parametrize("orders", [[17], [64], [65], [130], [200], [256], [257], [600], [1100], [40, 300, 17, 700, 255]])
def test_nothing_to_rotate(orders):
    import torch

    from syngular_amd import batch

    rng = np.random.default_rng(len(orders) + orders[0])
    mats, kept = [], []
    for n in orders:
        G = nearly_diagonal(n, rng)
        mats += [G]
        kept += [True]
        if len(orders) > 1:
            # one entry that does rotate
            H = G.copy()
            H[n - 1, n // 2] = H[n // 2, n - 1] = 1e-3 * np.sqrt(H[n - 1, n - 1] * H[n // 2, n // 2])
            mats += [H]
            kept += [False]
    dev = [torch.tensor(m, device="cuda") for m in mats]
    rts = [torch.full_like(m, 7.0) for m in dev]
    ss = [torch.full((m.shape[0],), 7.0, dtype=torch.float64, device="cuda") for m in dev]
    ptr = lambda ts: np.array([t.data_ptr() for t in ts], np.uint64)   # noqa: E731
    batch.jacobi_gram_blocked_table(ptr(dev), np.array([m.shape[0] for m in mats]), ptr(rts), ptr(ss), tol=TOL)
    for m, k, g, rt, s in zip(mats, kept, dev, rts, ss):
        g, rt, s = g.cpu().numpy(), rt.cpu().numpy(), s.cpu().numpy()
        n = len(m)
        if k:
            order = np.argsort(-np.diag(m), kind="stable")
            assert np.array_equal(g, m), n
            assert np.array_equal(rt, np.eye(n)[order]), n
            assert np.array_equal(s, np.sqrt(np.diag(m)[order])), n
        else:
            # off-diagonal entries up to the threshold remain
            ref = np.linalg.eigvalsh(m)[::-1]
            assert np.abs(s ** 2 - ref).max() <= 2 * n * TOL * ref[0] * 1e-1, n
            assert np.abs(rt @ rt.T - np.eye(n)).max() <= 1e-12, n
