"""Householder QR by register panels against numpy.linalg.qr (the LAPACK
convention fixes every sign), at the edges of its row classes, panels and
column tiles, with columns already zero below the diagonal."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

ROWS = [1, 15, 16, 17, 127, 128, 129, 255, 257, 511, 512, 513]
COLS = [1, 15, 16, 17, 31, 32, 33, 63, 65, 95, 96, 97]


def compare(Q, A, keep, q_trans, what):
    kq = min(keep, A.shape[0])
    ref = np.linalg.qr(A, "complete")[0][:, :kq]
    got = Q.cpu().numpy()
    np.testing.assert_allclose(got.T if q_trans else got, ref, atol=1e-12, err_msg=what)


@pytest.mark.parametrize("m", ROWS)
def test_qr_panel_edges(m):
    import torch

    from syngular_amd import ops

    rng = np.random.default_rng(m)
    for n in COLS:
        # well conditioned, so that Q is fixed to a few eps times n
        A = rng.standard_normal((m, n)) + 3.0 * np.sqrt(max(m, n)) * np.eye(m, n)
        for keep in {n, max(1, n // 2), min(m, n) + 1}:
            if keep > 96 and m > 256:
                continue
            X = torch.tensor(A, device="cuda")
            for q_trans in (False, True):
                Q = ops.qr_many([(X, keep)], q_trans=q_trans)[0]
                compare(Q, A, keep, q_trans, f"{m} x {n} keep {keep} trans {q_trans}")
        # a transposed view
        Q = ops.qr_many([(torch.tensor(np.ascontiguousarray(A.T), device="cuda").t(), n)])[0]
        compare(Q, A, n, False, f"{m} x {n} strided")


@pytest.mark.parametrize("m,n,keep", [(255, 100, 100), (256, 256, 128), (513, 140, 120), (1023, 70, 70), (1024, 96, 90),
                                      (1025, 66, 66), (1100, 70, 70)])
def test_blocked_panel_edges(m, n, keep):
    import torch

    from syngular_amd import ops

    rng = np.random.default_rng(m + n)
    A = rng.standard_normal((m, n)) + 3.0 * np.sqrt(m) * np.eye(m, n)
    for q_trans in (False, True):
        compare(ops.qr_blocked(torch.tensor(A, device="cuda"), keep, q_trans), A, keep, q_trans, f"{m} x {n}")


def test_qr_panel_zero_columns():
    """Columns zero below the diagonal are left unreflected, as LAPACK does."""
    import torch

    from syngular_amd import ops

    A = np.triu(np.random.default_rng(3).standard_normal((70, 40)))
    A[5:, 20:] = np.random.default_rng(4).standard_normal((65, 20))
    Q = ops.qr_many([(torch.tensor(A, device="cuda"), 40)])[0].cpu().numpy()
    ref = np.linalg.qr(A, "complete")[0][:, :40]
    np.testing.assert_allclose(Q, ref, atol=1e-12)
