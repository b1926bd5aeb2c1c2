"""Householder QR of a matrix with a NaN: the column that holds it gets no
reflector, as a zero column, and the factor's other columns are those of the
matrix without it."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def with_and_without(m, n, col):
    import torch

    rng = np.random.default_rng(m + n)
    A = rng.standard_normal((m, n))
    A[:, col] = 0.0
    bad = A.copy()
    bad[m - 1, col] = np.nan
    return torch.tensor(bad, device="cuda"), torch.tensor(A, device="cuda")


@pytest.mark.parametrize("m,n,col", [(12, 5, 2), (60, 20, 0), (128, 64, 40), (256, 64, 63), (512, 90, 33), (700, 17, 5)])
def test_one_work_group(m, n, col):
    import torch

    from syngular_amd import ops

    bad, A = with_and_without(m, n, col)
    for trans in (False, True):
        assert torch.equal(ops.qr_many([(bad, n)], q_trans=trans)[0], ops.qr_many([(A, n)], q_trans=trans)[0])


@pytest.mark.parametrize("m,n,col", [(255, 100, 40), (600, 140, 10), (1024, 96, 70), (1100, 70, 3)])
def test_blocked(m, n, col):
    import torch

    from syngular_amd import ops

    bad, A = with_and_without(m, n, col)
    assert torch.equal(ops.qr_blocked(bad, n), ops.qr_blocked(A, n))
