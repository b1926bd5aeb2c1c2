"""Grouped QR of more matrices than the chip has compute units: the launches by
rows and by LDS give each matrix the bits it has alone, at the edges of their
classes, and a matrix outside a launch's class is still factored."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

EDGES = [(2, 1), (3, 2), (15, 9), (16, 15), (17, 3), (31, 30), (32, 5), (33, 32), (63, 40), (64, 63), (65, 64), (128, 16),
         (129, 90), (200, 97), (513, 8)]


@pytest.mark.parametrize("columns", [False, True])
def test_many_as_alone(columns):
    import torch

    from syngular_amd import batch

    rng = np.random.default_rng(1)
    shapes = EDGES + [(int(m), int(n)) for m, n in zip(rng.integers(9, 70, 300), rng.integers(1, 9, 300))]
    mats = [rng.standard_normal(s) + 3.0 * np.sqrt(max(s)) * np.eye(*s) for s in shapes]

    def run(sel):
        m, n = (np.array([shapes[i][c] for i in sel], np.int64) for c in (0, 1))
        at, ap = batch.arena(m * n)
        qt, qp = batch.arena(m * n)
        wt, wp = batch.arena(m * n)
        tt, tp = batch.arena(n)
        src = [torch.tensor(mats[i], device="cuda") for i in sel]
        batch.copy_table(np.array([s.data_ptr() for s in src], np.uint64), ap, m * n)
        batch.qr_table(ap, m, n, qp, wp, tp, columns=columns)
        q = qt.cpu().numpy()
        off = [(int(p) - qt.data_ptr()) // 8 for p in qp]
        return [q[o:o + a * b].reshape(a, b) for o, a, b in zip(off, m, n)]

    whole = run(range(len(shapes)))
    for i, q in enumerate(whole):
        np.testing.assert_allclose(q, np.linalg.qr(mats[i])[0], atol=1e-12, err_msg=str(shapes[i]))
        if i < len(EDGES) + 5:
            assert np.array_equal(run([i])[0], q), shapes[i]


@pytest.mark.parametrize("rows", [1, 16, 17, 32, 64])
def test_rows_beyond_the_class(rows):
    """Any keep, strides and orientation, in a launch for fewer rows than some
    of its matrices have."""
    import torch

    from syngular_amd import _lib, ops

    rng = np.random.default_rng(rows)
    probs = []
    for m, n, keep in [(5, 9, 4), (9, 5, 9), (40, 100, 98), (70, 20, 20), (16, 16, 16), (33, 7, 3)]:
        A = rng.standard_normal((m, n)) + 3.0 * np.sqrt(max(m, n)) * np.eye(m, n)
        probs.append((A, keep))
    for trans in (0, 1):
        items = np.zeros(len(probs), dtype=_lib.QR_ITEM)
        hold = []
        for it, (A, keep) in zip(items, probs):
            m, n = A.shape
            nb, kq = min(n, keep), min(keep, m)
            X = torch.tensor(np.ascontiguousarray(A.T), device="cuda").t()
            Q = torch.empty((kq, m) if trans else (m, kq), dtype=torch.float64, device="cuda")
            W = torch.empty(m * (nb + kq), dtype=torch.float64, device="cuda")
            tau = torch.empty(nb, dtype=torch.float64, device="cuda")
            it["a"], it["rs"], it["cs"], it["m"], it["n"], it["keep"] = X.data_ptr(), 1, m, m, n, keep
            it["q"], it["ldq"], it["q_trans"] = Q.data_ptr(), m if trans else kq, trans
            it["work"], it["tau"] = W.data_ptr(), tau.data_ptr()
            hold.append((X, Q, W, tau))
        dev = ops._device_table(items)
        _lib.call("syn_qr_rows_f64", dev.data_ptr(), len(items), rows, ctypes.c_void_p(0))
        torch.cuda.synchronize()
        for (A, keep), (_, Q, _, _) in zip(probs, hold):
            ref = np.linalg.qr(A, "complete")[0][:, :keep]
            got = Q.cpu().numpy()
            np.testing.assert_allclose(got.T if trans else got, ref, atol=1e-12, err_msg=str((A.shape, keep)))


def test_arguments_are_checked():
    from syngular_amd import _lib

    for fn, size in (("syn_qr_rows_f64", 65), ("syn_qr_rows_f64", 0), ("syn_qr_columns_f64", 12289), ("syn_qr_columns_f64", -1)):
        with pytest.raises(ValueError):
            _lib.call(fn, None, 0, size, None)
