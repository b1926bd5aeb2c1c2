"""Reduction of the Gram eigen-solver over several work-groups: the upper edge
of its orders, several large matrices in a call, streams side by side, and
matrices whose work-groups give up waiting, which the Jacobi sweeps then take
from a restored matrix."""
import ctypes
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

EPS = float(np.finfo(np.float64).eps)


def gram(n, seed, grade=0.0, scale=0):
    import torch

    gen = torch.Generator(device="cuda").manual_seed(seed)
    X = torch.randn((n, n + 7), dtype=torch.float64, device="cuda", generator=gen)
    X *= torch.logspace(0, -grade, n, dtype=torch.float64, device="cuda")[:, None]
    G = X @ X.t()
    return 0.5 * (G + G.t()) * 2.0 ** scale


def solve(mats, polls=0):
    import torch

    from syngular_amd import _lib, batch, ops

    n = [m.shape[0] for m in mats]
    G = [m.clone() for m in mats]
    R = [torch.full_like(m, 7.0) for m in mats]
    S = [torch.full((k,), 7.0, dtype=torch.float64, device="cuda") for k in n]
    it = np.zeros(len(mats), dtype=_lib.GBJ_ITEM)
    for i, (g, r, s, k) in enumerate(zip(G, R, S, n)):
        it[i]["g"], it[i]["ldg"], it[i]["rt"], it[i]["ldr"], it[i]["s"], it[i]["nv"] = (
            g.data_ptr(), k, r.data_ptr(), k, s.data_ptr(), k)
    nv = np.array(n, np.int64)
    size = int(_lib.load().syn_jacobi_gram_blocked_workspace(nv.ctypes.data_as(ctypes.c_void_p), len(n)))
    work = torch.empty(size, dtype=torch.float64, device="cuda")
    counters = torch.empty(len(n), dtype=torch.int32, device="cuda")
    table = torch.empty(it.nbytes, dtype=torch.uint8, device="cuda")
    sweeps = ctypes.c_int(0)
    _lib.call("syn_jacobi_gram_blocked_polls_f64", table.data_ptr(), it.ctypes.data_as(ctypes.c_void_p), len(n),
              work.data_ptr(), counters.data_ptr(), batch.TOL_BLOCKED, ops.JACOBI_SWEEPS, polls, ctypes.byref(sweeps),
              ops._stream())
    return list(zip(R, S))


def check(G, rt, s, scale=0):
    """A decomposition with the residuals of a few n eps that the other tests
    of the solver allow."""
    import torch

    n = G.shape[0]
    G, lam = G * 2.0 ** -scale, (s * 2.0 ** -(scale // 2)) ** 2
    eye = torch.eye(n, dtype=G.dtype, device=G.device)
    assert bool((lam[1:] <= lam[:-1]).all()), n
    assert float((rt @ rt.t() - eye).abs().max()) <= 20 * n * EPS, n
    assert float((rt.t() @ (lam[:, None] * rt) - G).norm()) <= 20 * n * EPS * float(G.norm()), n


def gave_up():
    from syngular_amd import ops

    return ops.gram_gave_up()


@pytest.mark.parametrize("orders", [[2047], [2048], [2049], [2048, 1100, 2048, 1500], [300] * 40])
def test_upper_orders_and_many(orders):
    before = gave_up()
    mats = [gram(n, i, grade=2.0 * (i % 2)) for i, n in enumerate(orders)]
    for G, (rt, s) in zip(mats, solve(mats)):
        check(G, rt, s)
    assert gave_up() == before


@pytest.mark.parametrize("polls", [1, 40])
@pytest.mark.parametrize("scale", [0, -540, 540])
def test_giving_up_is_counted_and_right(polls, scale):
    """With next to no polls the work-groups give up in one of the first steps,
    after some have overwritten their part of the upper triangle.  The scales
    are those at which the sweeps' test has to scale its squares."""
    before = gave_up()
    mats = [gram(n, n, 1.0, scale) for n in (300, 40, 700, 257, 1100)]
    for G, (rt, s) in zip(mats, solve(mats, polls)):
        check(G, rt, s, scale)
    if polls == 1:
        assert 1 <= gave_up() - before <= 4


def test_streams_side_by_side():
    """Calls on several streams at once give the bits that each gives alone."""
    import torch

    before = gave_up()
    sets = [[1500, 1500, 1500], [2048, 600], [1100, 300, 300], [512] * 12]
    sets = [[gram(n, 100 * i + j) for j, n in enumerate(orders)] for i, orders in enumerate(sets)]
    ref = [solve(mats) for mats in sets]
    torch.cuda.synchronize()
    differ = []

    def lane(i):
        with torch.cuda.stream(torch.cuda.Stream()):
            for _ in range(6):
                for (a, b), (c, d) in zip(solve(sets[i]), ref[i]):
                    if not (torch.equal(a, c) and torch.equal(b, d)):
                        differ.append(i)

    lanes = [threading.Thread(target=lane, args=(i,)) for i in range(len(sets))]
    for t in lanes:
        t.start()
    for t in lanes:
        t.join()
    assert differ == []
    assert gave_up() == before


def test_non_finite_ends():
    """A NaN or an infinity beside finite matrices: the call returns, and the
    finite ones are what they are alone."""
    import torch

    for n in (100, 300, 600):
        good = gram(n, 1)
        alone = solve([good])[0]
        for value, at in ((np.nan, (3, 5)), (np.inf, (n - 1, 0)), (np.nan, (4, 4))):
            bad = good.clone()
            bad[at] = bad[at[::-1]] = value
            rt, s = solve([bad, good])[1]
            assert torch.equal(rt, alone[0]) and torch.equal(s, alone[1]), (n, value, at)
