"""Driven Lindblad runs with form "auto": Hermitian Hamiltonians from d = 8 on take the matrix form while
24 n_c <= d d, everything else the Liouville-space form.  Both are FP64 RK4 of the same equation: observables,
states and batches agree to 60 steps of rounding (1e-13 on O(1) states), and a call that keeps the
Liouville-space form gives its very numbers."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _system(d, nc, seed=0):
    rng = np.random.default_rng([seed, d, nc])

    def herm():
        a = rng.normal(size=(d, d)) + 1j * rng.normal(size=(d, d))
        return (a + a.conj().T) / (2 * np.sqrt(d))
    cs = [0.2 * (rng.normal(size=(d, d)) + 1j * rng.normal(size=(d, d))) / d for _ in range(nc)]
    rhos = np.array([np.diag(v / v.sum()) for v in rng.uniform(size=(3, d))]).astype(complex)
    return herm(), [herm(), herm()], cs, rhos, rng.normal(size=(3, 60, 2)) * 0.3


def _both(H0, drives, cs, rhos, fields):
    from pyqed_amd.oqs import LindbladSolver
    nt, out = 60, []
    for form in ("auto", "liouville"):
        s = LindbladSolver([H0] + [[h, None] for h in drives], cs, form=form)
        final = s.run_batch(rhos, 0.02, nt, fields)
        t = LindbladSolver([H0] + [[h, lambda t, k=k: np.cos((k + 1) * t)] for k, h in enumerate(drives)], cs, form=form)
        r = t.run(rhos[0], 0.02, nt, e_ops=[H0, drives[0]])
        out.append((final, np.asarray(r.observables), np.array(r.rholist)))
    return out


@pytest.mark.parametrize("d,nc", [(8, 0), (8, 2), (9, 3), (15, 9), (16, 10), (17, 12), (24, 5), (32, 2)])
def test_matrix_form_for_driven_runs(d, nc):
    a, b = _both(*_system(d, nc))
    for x, y in zip(a, b):
        assert x.shape == y.shape and np.abs(x - y).max() <= 1e-13


@pytest.mark.parametrize("case", ["small", "many", "H", "drive"])
def test_liouville_form_keeps_its_calls(case):
    d, nc = {"small": (7, 1), "many": (8, 3)}.get(case, (8, 2))
    H0, drives, cs, rhos, fields = _system(d, nc)
    if case == "H":
        H0 = H0 + 0.1j * np.eye(d, k=1)
    if case == "drive":
        drives[1] = drives[1] + 0.1 * np.eye(d, k=1)
    a, b = _both(H0, drives, cs, rhos, fields)
    for x, y in zip(a, b):
        assert np.array_equal(x, y)
