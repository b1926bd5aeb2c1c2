"""The library's own launch census covers the direct phase of the blocked Gram
eigen-solver, with the work of its products."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [40, 300])
def test_direct_phase_is_counted(n):
    import torch

    from syngular_amd import ops

    X = torch.randn((n, 2 * n), dtype=torch.float64, device="cuda")
    G = X @ X.t()
    ops.jacobi_gram_blocked(G.clone())
    ops.profile_begin()
    ops.jacobi_gram_blocked(G.clone())
    census = ops.profile_end()
    for tag in ("td_reduce_kernel", "td_merge_kernels", "td_back_kernel", "td_gemm_kernel"):
        assert census[tag][0] > 0 and census[tag][1] > 0.0, tag
    assert census["td_gemm_kernel"][2] == 4.0 * n ** 3
    assert census["td_back_kernel"][2] == 2.0 * n ** 3
