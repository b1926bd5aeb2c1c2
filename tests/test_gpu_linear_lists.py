"""A Linear on lists around the length where the batched tables start: each
result has the bits that its state gives in a list of its own."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def chain(rng, bonds, d):
    b = [1, *bonds, 1]
    return [rng.standard_normal((b[k], d, b[k + 1])) / np.sqrt(b[k]) for k in range(len(b) - 1)]


def layer(rng, bonds, d):
    from syngular_amd.tensor import MatrixProductOperator

    w = [1, *bonds, 1]
    return MatrixProductOperator.from_sites(
        [rng.standard_normal((w[k], d, d, w[k + 1])) / np.sqrt(w[k] * d) for k in range(len(w) - 1)])


@pytest.mark.parametrize("count", [1, 2, 3, 4])
@pytest.mark.parametrize("wbonds,xbonds,d", [((8, 8), [(4, 16), (3, 5)], 4), ((3, 3, 3, 3, 3), [(2, 7, 9, 4, 2)], 3),
                                             ((1, 1), [(2, 3)], 2)])
def test_lengths(count, wbonds, xbonds, d):
    import torch

    from syngular_amd.core import matmul_batch
    from syngular_amd.tensor import MatrixProductState

    rng = np.random.default_rng(count)
    W = layer(rng, wbonds, d)
    xs = [MatrixProductState.from_sites(chain(rng, xbonds[i % len(xbonds)], d)) for i in range(count)]
    for y, x in zip(matmul_batch(W, xs), xs):
        z = matmul_batch(W, [x])[0]
        assert (y.shape, y.bond_shape, y.input_shape, y.parameters_number) == (
            z.shape, z.bond_shape, z.input_shape, z.parameters_number)
        assert all(torch.equal(a, b) for a, b in zip(y.sites, z.sites))


@pytest.mark.parametrize("wbonds,xbonds", [((1, 8), (1, 400)), ((12, 12), (20, 20)), ((24, 24), (24, 24))])
def test_a_kept_output_holds_little_else(wbonds, xbonds):
    """Results that are product cores (a min bond of one is kept) and truncated
    ones, small and large."""
    import torch

    from syngular_amd.core import matmul_batch
    from syngular_amd.tensor import MatrixProductState

    rng = np.random.default_rng(xbonds[1])
    W = layer(rng, wbonds, 24)
    xs = [MatrixProductState.from_sites(chain(rng, xbonds, 24)) for _ in range(24)]
    ys = matmul_batch(W, xs)
    alone = matmul_batch(W, xs[3:4])[0]
    for a, b in zip(ys[3].sites, alone.sites):
        assert torch.equal(a, b)
        held = a.untyped_storage().nbytes()
        assert held <= max(a.numel() * 8, 1 << 21)
