"""A Linear call on a list equals ``weight @ x`` state by state: mixed shapes,
states that need no truncation, one state, two sites, strided input cores, and
the errors of shapes that do not fit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def chain(rng, bonds, d):
    b = [1, *bonds, 1]
    return [rng.standard_normal((b[k], d, b[k + 1])) / np.sqrt(b[k]) for k in range(len(b) - 1)]


@pytest.mark.parametrize("wbonds,xbonds,d", [
    ((3,), [(2,)], 3),
    ((4, 4), [(3, 5), (1, 1), (9, 9), (3, 5)], 4),
    ((1, 1, 1), [(2, 3, 2), (4, 4, 4)], 2),
    ((8, 8, 8), [(4, 16, 4), (2, 7, 3), (4, 16, 4), (3, 5, 5)] * 3, 4),
])
def test_list_equals_one_by_one(wbonds, xbonds, d):
    import torch

    from syngular_amd.core import matmul_batch
    from syngular_amd.tensor import MatrixProductOperator, MatrixProductState

    rng = np.random.default_rng(len(xbonds) + d)
    w = [1, *wbonds, 1]
    W = MatrixProductOperator.from_sites(
        [rng.standard_normal((w[k], d, d, w[k + 1])) / np.sqrt(w[k] * d) for k in range(len(w) - 1)])
    xs = [MatrixProductState.from_sites(chain(rng, b, d)) for b in xbonds]
    # a core that is not contiguous
    s = xs[0].sites[0]
    xs[0].sites[0] = torch.stack([s, s], dim=-1)[..., 0]
    got = matmul_batch(W, xs)
    assert len(got) == len(xs)
    for y, x in zip(got, xs):
        z = W @ x
        assert (y.shape, y.bond_shape, y.input_shape) == (z.shape, z.bond_shape, z.input_shape)
        assert (y.parameters_number, y.sites_number, y.orthonormalized) == (
            z.parameters_number, z.sites_number, z.orthonormalized)
        for a, b in zip(y.sites, z.sites):
            assert a.shape == b.shape and a.is_contiguous()
        # (the truncation takes the leading columns of each product, which a
        # rounding error cannot exchange: a few eps per bond and column)
        a, b = y.to_tensor(), z.to_tensor()
        assert np.linalg.norm(a - b) <= 1e-12 * np.linalg.norm(b)
    assert matmul_batch(W, []) == []
    bad = MatrixProductState.from_sites(chain(rng, xbonds[0], d + 1))
    with pytest.raises(ValueError):
        matmul_batch(W, [xs[0], bad])
    if len(wbonds) > 1 and min(wbonds) > d:
        # a min bond beyond the first unfolding's rows does not reshape, as one by one
        bad = MatrixProductState.from_sites(chain(rng, [d + 1] * len(wbonds), d))
        with pytest.raises(ValueError, match="cannot reshape"):
            matmul_batch(W, [xs[0], bad])
