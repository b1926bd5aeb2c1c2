"""GEMM launches of few tiles (32 x 32 quadrants) give the bits of launches of
many (64 x 64 tiles), at the edges of tiles and K steps, in both operand
orientations and with the structural-zero hints; both against float64 matmul."""
import pytest

pytestmark = pytest.mark.gpu

SHAPES = [(1, 1, 1), (3, 70, 5), (31, 33, 31), (32, 32, 32), (33, 65, 33), (64, 64, 64), (65, 63, 65), (97, 130, 257)]


@pytest.mark.parametrize("mixed", [False, True])
@pytest.mark.parametrize("ta", [False, True])
@pytest.mark.parametrize("tb", [False, True])
def test_quadrants_match_tiles(ta, tb, mixed):
    import torch

    from syngular_amd import ops

    gen = torch.Generator(device="cuda").manual_seed(1)
    for m, n, k in SHAPES:
        for tri in [0, 1] + ([2, 4] if m == k else []) + ([8, 16] if n == k else []):
            A = torch.randn((m, k), dtype=torch.float64, device="cuda", generator=gen)
            B = torch.randn((k, n), dtype=torch.float64, device="cuda", generator=gen)
            A = A.tril() if tri == 2 else A.triu() if tri == 4 else A
            B = B.triu() if tri == 8 else B.tril() if tri == 16 else B
            A = A.t().contiguous().t() if ta else A.contiguous()
            B = B.t().contiguous().t() if tb else B.contiguous()
            C0 = torch.randn((m, n), dtype=torch.float64, device="cuda", generator=gen)
            few = C0.clone()
            ops.gemm_many([(A, B, few, 0.5, 2.0, tri)], tile=0, mixed=mixed)
            many = [C0.clone() for _ in range(130)]
            ops.gemm_many([(A, B, c, 0.5, 2.0, tri) for c in many], tile=0, mixed=mixed)
            what = f"{m}x{n}x{k} tri {tri}"
            low = (lambda x: x.tril()) if tri == 1 else (lambda x: x)
            for c in (many[0], many[-1]):
                assert torch.equal(low(few), low(c)), what
            ref = 0.5 * (A @ B) + 2.0 * C0
            # k products of order one, each rounded in the compute type
            tol = (4e-7 if mixed else 1e-15) * (k + 4) * 4
            assert float((low(few) - low(ref)).abs().max()) <= tol, what
