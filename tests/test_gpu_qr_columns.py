"""The column-by-column QR of the mixed sweep against numpy.linalg.qr: edges of
its row segments and load groups, in LDS and from the workspace, and the same
bits whatever else is in the launch."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shapes", [[(2, 1)], [(33, 32), (34, 33), (65, 64), (40, 7)], [(128, 95), (129, 1), (600, 20)],
                                    [(700, 60)]])
def test_columns_match_numpy(shapes):
    import torch

    from syngular_amd import batch

    rng = np.random.default_rng(len(shapes))
    mats = [rng.standard_normal(s) + 3.0 * np.sqrt(max(s)) * np.eye(*s) for s in shapes]

    def run(sel):
        m, n = (np.array([shapes[i][c] for i in sel], np.int64) for c in (0, 1))
        at, ap = batch.arena(m * n)
        qt, qp = batch.arena(m * n)
        wt, wp = batch.arena(m * n)
        tt, tp = batch.arena(n)
        src = [torch.tensor(mats[i], device="cuda") for i in sel]
        batch.copy_table(np.array([s.data_ptr() for s in src], np.uint64), ap, m * n)
        batch.qr_table(ap, m, n, qp, wp, tp, columns=True)
        q = qt.cpu().numpy()
        off = [(int(p) - qt.data_ptr()) // 8 for p in qp]
        return [q[o:o + a * b].reshape(a, b) for o, a, b in zip(off, m, n)]

    whole = run(range(len(shapes)))
    for i, q in enumerate(whole):
        np.testing.assert_allclose(q, np.linalg.qr(mats[i])[0], atol=1e-12, err_msg=str(shapes[i]))
        assert np.array_equal(run([i])[0], q), shapes[i]
