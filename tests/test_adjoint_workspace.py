"""The workspace of a gradient that is cut along time: bounded for long runs of many instances, where the checkpoints
alone are asked for, and done without where the device has no room for it."""
import numpy as np
import pytest


def _bytes(N, nterm, n, nt, ckpt):
    from pyqed_amd import _lib
    b = _lib.C.c_int64()
    _lib.check(_lib.lib().pyqed_liouville_adjoint_work_bytes(N, nterm, n, nt, ckpt, _lib.C.byref(b)))
    return b.value, (n * (-(-nt // ckpt) + 1) + n * ckpt) * N * 16


@pytest.mark.parametrize("N,nterm,n,nt,ckpt", [(16, 2, 384, 100000, 300), (9, 2, 1000, 200000, 400), (4, 3, 1000, 1000000, 1000),
                                               (16, 2, 1, 20000000, 4000)])
def test_long_runs_ask_for_checkpoints_only(N, nterm, n, nt, ckpt):
    got, checkpoints = _bytes(N, nterm, n, nt, ckpt)
    assert got == checkpoints


@pytest.mark.parametrize("N,n,nt", [(9, 1, 1000), (9, 256, 1000), (4, 1, 100000)])
def test_cut_workspaces_stay_bounded(N, n, nt):
    got, checkpoints = _bytes(N, 2, n, nt, 50)
    assert checkpoints < got <= 4 << 30


@pytest.mark.gpu
def test_gradient_without_room_for_the_cut(monkeypatch):
    import torch
    from pyqed_amd.adjoint import lambda_system
    mu = np.array([[0, 1, 0], [1, 0, 0.7], [0, 0.7, 0]], complex)
    prob = lambda_system([0.0, 1.0, 2.5], mu, [0.1 * np.diag([0, 1.0, 2.0]).astype(complex)], 0.05, 20, 10, ckpt_every=20)
    rng = np.random.default_rng(1)
    args = ([0.0, 1.1, 2.4], rng.normal(0, 0.1, (1, 10)), np.diag([1.0, 0, 0]).astype(complex), np.diag([0, 0, 1.0]).astype(complex))
    want = prob.gradient(*args)
    limit = (200 // 20 + 1 + 20) * 9 * 16
    empty, asked = torch.empty, []

    def short(*size, **kw):
        if kw.get("dtype") == torch.uint8:
            asked.append(size[0])
            if size[0] > limit:
                raise torch.OutOfMemoryError("no room")
        return empty(*size, **kw)

    monkeypatch.setattr(torch, "empty", short)
    got = prob.gradient(*args)
    assert len(asked) == 2 and asked[1] == limit
    for a, b in zip(got, want):
        assert np.abs(a - b).max() <= 1e-12 * max(1.0, np.abs(b).max())
