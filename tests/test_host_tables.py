"""Item tables by value: the largest host table, refusals beyond it, and the
same bits as the device table on both sides of the limit."""
import numpy as np
import pytest

from syngular_amd import _lib


def test_limits_are_checked_on_the_host():
    for name, host in _lib.HOST_ENTRIES.items():
        assert host in _lib.SIGNATURES and _lib.SIGNATURES[host] == _lib.SIGNATURES[name]
    items = np.zeros(64, dtype=_lib.GEMM_ITEM)
    most = _lib.INLINE_BYTES // _lib.GEMM_ITEM.itemsize
    with pytest.raises(ValueError):
        _lib.call("syn_gemm_f64_host", items.ctypes.data, most + 1, 1, 0, None)
    with pytest.raises(ValueError):
        _lib.call("syn_gemm_f64_host", None, 1, 1, 0, None)
    with pytest.raises(ValueError):
        _lib.call("syn_gemm_f64_host", items.ctypes.data, 1, 1, 2, None)
    with pytest.raises(ValueError):
        _lib.call("syn_qr_sized_f64_host", items.ctypes.data, -1, 0, None)
    with pytest.raises(ValueError):
        _lib.call("syn_jacobi_gram_f64_host", items.ctypes.data, 1, 65, 1e-14, 30, None)
    # nothing to do is not an error
    _lib.call("syn_gemm_f64_host", None, 0, 0, 0, None)


@pytest.mark.gpu
@pytest.mark.parametrize("count", [1, 2, 31, 32, 33])
def test_same_bits_by_value_and_from_the_device(count, monkeypatch):
    import torch

    from syngular_amd import ops

    gen = torch.Generator(device="cuda").manual_seed(count)
    rnd = lambda *s: torch.randn(s, dtype=torch.float64, device="cuda", generator=gen)   # noqa: E731
    A = [rnd(20 + i, 30) for i in range(count)]
    B = [rnd(30, 10 + i % 7) for i in range(count)]
    O, X = rnd(3, 2, 2, 4), [rnd(2 + i % 3, 2, 5) for i in range(count)]
    S = [rnd(6 + i % 11, 6 + i % 11) for i in range(count)]
    S = [s @ s.t() for s in S]

    def work():
        C = [torch.empty((a.shape[0], b.shape[1]), dtype=torch.float64, device="cuda") for a, b in zip(A, B)]
        out = []
        for mixed in (False, True, "bf16"):
            ops.gemm_many([(a, b, c, 1.0, 0.0) for a, b, c in zip(A, B, C)], mixed=mixed)
            out += [c.clone() for c in C]
        out += ops.apply_many([(O, x) for x in X])
        out += ops.qr_many([(a, 5) for a in A])
        for rt, s in ops.jacobi_gram_many(S):
            out += [rt, s]
        keep, disc = ops.truncate_many([(s.diagonal().clone(), 4, 1e-3) for s in S])
        norms = [torch.empty(a.shape[1], dtype=torch.float64, device="cuda") for a in A]
        ops.vecnorms_many([(a, 0, v) for a, v in zip(A, norms)])
        eyes = [torch.empty_like(s) for s in S]
        ops.eye_many(eyes)
        copies = [torch.empty_like(a) for a in A]
        ops.copy_many(list(zip(A, copies)))
        ops.rowscale_many([(c, v, 0) for c, v in zip(copies, [a[:, 0].clone() for a in A])])
        return out + [keep, disc, *norms, *eyes, *copies]

    by_value = work()
    monkeypatch.setattr(ops, "_upload", ops._device_table)
    for a, b in zip(by_value, work()):
        assert torch.equal(a, b)
