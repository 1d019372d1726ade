"""Where a small hierarchy's FP64 call takes powers of its generator: from max(64, N^2 / 2400) steps on, N the elements of
the hierarchy.  Below that the resident kernel steps, and a call equals its parts bit for bit; from there on the powers
agree with steps to 1e-12 (FP64 errors of about nsteps eps on O(1) states)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d,L,nt,powers", [(4, 7, 100, False), (4, 7, 137, False), (4, 7, 138, True), (4, 6, 82, False),
                                           (4, 6, 83, True), (3, 7, 63, False), (3, 7, 64, True)])
def test_rule_follows_the_size(d, L, nt, powers):
    from pyqed_amd.heom.engine import HeomEngine
    rng = np.random.default_rng([d, L])
    H = rng.normal(size=(d, d))
    eta = np.array([0.2 - 0.1j, 0.1 + 0.05j])
    inst = dict(H=(H + H.T).astype(complex) / 4, Q=np.diag(np.linspace(1, -1, d)).astype(complex)[None], L=L, rho0=np.eye(d) / d + 0j,
                bath=(eta, eta.conj(), np.abs(eta), np.array([0.7, 1.9]) + 0j, np.zeros(2, int)))
    eng = HeomEngine([inst])
    assert eng.stats()["resident_instances"] == 1
    eng.advance(nt, 0.01, "fp64")
    whole = eng.hierarchy(0)
    eng.reset()
    for left in range(nt, 0, -40):
        eng.advance(min(40, left), 0.01, "fp64")
    parts = eng.hierarchy(0)
    assert np.array_equal(whole, parts) != powers
    assert np.abs(whole - parts).max() <= 1e-12
    eng.close()
