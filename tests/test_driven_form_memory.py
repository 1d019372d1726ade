"""A driven batch whose matrix-form workspace does not fit the device runs on the Liouville-space kernel, which needs the
states alone; forms that were asked for, other errors and sizes that only the matrix form serves are passed on."""
import numpy as np
import pytest

from pyqed_amd import oqs


def _call(monkeypatch, d, form, error):
    import torch
    calls = []

    def matrix(*a, **k):
        calls.append("matrix")
        raise (torch.OutOfMemoryError("no room") if error == "memory" else RuntimeError("other"))

    def liouville(gens, rho0s, dt, nt, *a, **k):
        calls.append("liouville")
        return np.zeros((len(rho0s), nt + 1, 0), complex), np.zeros((len(rho0s), 0, d, d), complex), rho0s

    monkeypatch.setattr(oqs, "propagate_matrix", matrix)
    monkeypatch.setattr(oqs, "propagate", liouville)
    H = np.diag(np.arange(d, dtype=float))
    s = oqs.LindbladSolver([H, [np.eye(d, k=1) + np.eye(d, k=-1), None]], [], form=form)
    try:
        s.run_batch(np.zeros((3, d, d), complex), 0.01, 4, np.zeros((3, 4, 1)))
    except RuntimeError as e:
        calls.append(type(e).__name__)
    return calls


def test_falls_back(monkeypatch):
    assert _call(monkeypatch, 12, "auto", "memory") == ["matrix", "liouville"]


@pytest.mark.parametrize("d,form,error,last", [(12, "matrix", "memory", "OutOfMemoryError"), (33, "auto", "memory", "OutOfMemoryError"),
                                               (12, "auto", "other", "RuntimeError")])
def test_passes_on(monkeypatch, d, form, error, last):
    assert _call(monkeypatch, d, form, error) == ["matrix", last]
