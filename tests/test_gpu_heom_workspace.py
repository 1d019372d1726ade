"""Scratch of a small hierarchy's FP64 runs: what powers of its generator need is asked for only by calls that take them,
and a run steps where the device has no room for it."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _engine():
    from pyqed_amd.heom.engine import HeomEngine
    rng = np.random.default_rng(3)
    d = 4
    H = rng.normal(size=(d, d))
    eta = np.array([0.2 - 0.1j, 0.1 + 0.05j])
    return HeomEngine([dict(H=(H + H.T).astype(complex) / 4, Q=np.diag(np.linspace(1, -1, d)).astype(complex)[None], L=7, rho0=np.eye(d) / d + 0j,
                            bath=(eta, eta.conj(), np.abs(eta), np.array([0.7, 1.9]) + 0j, np.zeros(2, int)))])


def test_short_calls_take_little():
    eng = _engine()
    eng.advance(63, 0.01, "fp64")
    assert eng._ws.numel() <= 16 * eng.n_elems + 255 + 32 * 36 * 16   # the state, and two stage buffers of 36 full matrices
    eng.advance(200, 0.01, "fp64")
    assert eng._ws.numel() == eng.ws_bytes[0] > 10 ** 7
    eng.close()


def test_steps_where_there_is_no_room(monkeypatch):
    import torch
    want = _engine()
    for _ in range(5):
        want.advance(40, 0.01, "fp64")
    empty = torch.empty

    def short(*size, **kw):
        if kw.get("dtype") == torch.uint8 and size[0] > 10 ** 6:
            raise torch.OutOfMemoryError("no room")
        return empty(*size, **kw)

    monkeypatch.setattr(torch, "empty", short)
    eng = _engine()
    eng.advance(150, 0.01, "fp64")
    eng.advance(50, 0.01, "fp64")
    assert np.array_equal(eng.hierarchy(0), want.hierarchy(0))
    eng.close()
    want.close()


def test_a_workspace_that_is_too_small_is_refused():
    import torch
    from pyqed_amd import _lib
    eng = _engine()
    ws = torch.empty(16 * eng.n_elems, dtype=torch.uint8, device=eng.device)
    with pytest.raises(_lib.PyqedError):
        _lib.check(eng.L.pyqed_heom_run(eng.plan, _lib.PREC_FP64, eng.y.data_ptr(), ws.data_ptr(), ws.numel(), None, 0, 200, 0.01, None, 1,
                                        torch.cuda.current_stream().cuda_stream))
    eng.close()
