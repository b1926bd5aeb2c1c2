"""Gram eigen-solvers on matrices scaled by powers of two, to the ends of the
doubles: the scale is exact, so singular values and vectors have to be those of
the unscaled matrix to rounding."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

EPS = float(np.finfo(np.float64).eps)
# even, so that s scales by a power of two; entries from 1e-300 to 1e303
SCALES = [-1000, -560, -534, -500, -300, 0, 300, 480, 520, 1000]


def gram(g):
    X = np.random.default_rng(g).standard_normal((g, 2 * g)) / np.sqrt(2 * g)
    X *= np.logspace(0, -3, g)[:, None]
    G = X @ X.T
    return 0.5 * (G + G.T)


def check(G, rt, s, k):
    """As test_gpu_jacobi16: a few sweeps of rotations, each of a few eps."""
    g = G.shape[0]
    V, lam = rt.cpu().numpy(), np.ldexp(s.cpu().numpy(), -k // 2) ** 2
    ref = np.linalg.eigvalsh(G)[::-1]
    assert np.abs(lam - ref).max() <= 50 * g * EPS * ref[0], k
    assert np.abs(V @ V.T - np.eye(g)).max() <= 100 * g * EPS, k
    assert np.linalg.norm(V.T @ (lam[:, None] * V) - G) <= 100 * g * EPS * np.linalg.norm(G), k


@pytest.mark.parametrize("g", [1, 2, 3, 8, 15, 16, 17, 32, 33, 64])
def test_lds_orders(g):
    import torch

    from syngular_amd import ops

    G = gram(g)
    outs = ops.jacobi_gram_many([torch.tensor(np.ldexp(G, k), device="cuda") for k in SCALES])
    for k, (rt, s) in zip(SCALES, outs):
        check(G, rt, s, k)


@pytest.mark.parametrize("g", [17, 64, 100, 300])
def test_blocked_orders(g):
    import torch

    from syngular_amd import ops

    G = gram(g)
    for k in SCALES:
        rt, s, _ = ops.jacobi_gram_blocked(torch.tensor(np.ldexp(G, k), device="cuda"))
        check(G, rt, s, k)


@pytest.mark.parametrize("k", [-280, 260])
def test_rounding_of_a_scaled_chain(k):
    """A chain whose cores carry 2^k altogether: the rounded chain is that of
    the unscaled one, scaled."""
    import torch

    from syngular_amd import linalg, rounding

    rng = np.random.default_rng(3)
    bonds, n = [1, 2, 4, 8, 8, 4, 2, 1], 7
    cores = [rng.standard_normal((bonds[i], 2, bonds[i + 1])) / np.sqrt(2 * bonds[i]) for i in range(n)]

    def rounded(scale):
        xs = [torch.tensor(c, device="cuda") for c in cores]
        xs[0] = xs[0] * 2.0 ** scale
        rep = rounding.RoundingReport()
        return linalg.dense(rounding.tt_round(xs, chi_max=3, report=rep)).cpu().numpy().reshape(-1), rep

    want, rep0 = rounded(0)
    got, rep1 = rounded(k)
    assert list(rep0.kept) == list(rep1.kept)
    # orders up to 8: a few dozen rotations and products of a few eps
    assert np.linalg.norm(np.ldexp(got, -k) - want) <= 1000 * EPS * np.linalg.norm(want)


@pytest.mark.parametrize("value", [np.nan, np.inf])
@pytest.mark.parametrize("where", [(2, 2), (2, 3), (0, 6)])
def test_lds_non_finite(value, where):
    """A matrix that is not finite gives NaN singular values, writes every
    entry of its results and leaves its neighbours alone."""
    import torch

    from syngular_amd import batch, ops

    orders = [7, 16, 17, 40, 64]
    mats = []
    for g in orders:
        G = torch.eye(g, dtype=torch.float64) + 0.1
        bad = G.clone()
        bad[where] = bad[where[::-1]] = value
        mats += [bad.cuda(), G.cuda()]
    rts = [torch.full_like(m, 7.0) for m in mats]
    ss = [torch.full((m.shape[0],), 7.0, dtype=torch.float64, device="cuda") for m in mats]
    ptr = lambda ts: np.array([t.data_ptr() for t in ts], np.uint64)   # noqa: E731
    batch.jacobi_table(ptr(mats), np.array([m.shape[0] for m in mats]), ptr(rts), ptr(ss))
    for i, (m, rt, s) in enumerate(zip(mats, rts, ss)):
        assert not (rt == 7.0).any() and not (s == 7.0).any(), (m.shape[0], i)
        if i % 2 == 0:
            assert torch.isnan(s).all(), m.shape[0]
        else:
            ref = ops.jacobi_gram_many([m])[0]
            assert torch.equal(rt, ref[0]) and torch.equal(s, ref[1]), m.shape[0]
