"""FP64 projector kernels with the commutator on MFMA (12 <= d <= 16: one 16 x 16 tile, 17 <= d <= 32: 2 x 2
tiles) against the generic kernel (element loops) on the same plan inputs: tile edges, complex and real H,
packed and full state, Hermitian and not, driven.  Both are FP64: an element is a sum of fewer than 200
products of O(1) terms scaled by dt, so three steps stay within 1e-13 of each other."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _instance(d, L, seed, real, driven):
    rng = np.random.default_rng([seed, d])
    H = rng.normal(size=(d, d)) + (0 if real else 1j) * rng.normal(size=(d, d))
    H = (H + H.conj().T).astype(complex) / 2
    Q = np.zeros((d, d, d), complex)
    Q[np.arange(d), np.arange(d), np.arange(d)] = rng.uniform(0.5, 1.5, d)
    etal = 0.2 * (rng.normal(size=d) + 1j * rng.normal(size=d))
    rho0 = rng.normal(size=(d, d)) + 1j * rng.normal(size=(d, d))
    rho0 = rho0 @ rho0.conj().T
    inst = dict(H=H, Q=Q, L=L, rho0=rho0 / np.trace(rho0),
                bath=(etal, etal.conj(), np.abs(etal), rng.uniform(0.5, 2.0, d).astype(complex), rng.permutation(d)))
    if driven:
        inst["sdip"] = (np.diag(np.ones(d - 1), 1) + np.diag(np.ones(d - 1), -1)).astype(complex)
    return inst


@pytest.mark.parametrize("layout", [dict(), dict(packed=False), dict(hermitian=False, packed=False)])
@pytest.mark.parametrize("real,driven", [(True, False), (False, False), (True, True)])
@pytest.mark.parametrize("d,L", [(11, 2), (12, 2), (13, 3), (15, 2), (16, 3), (17, 2), (24, 2), (26, 2), (32, 1)])
def test_equals_generic_kernel(d, L, real, driven, layout):
    import torch
    from pyqed_amd.heom.engine import HeomEngine
    inst = _instance(d, L, 2, real, driven)
    out = []
    for generic in (False, True):
        eng = HeomEngine([inst], resident=False, generic=generic, **layout)
        field = torch.full((3, 6), 0.7, dtype=torch.float64, device=eng.device) if driven else None
        eng.advance(3, 0.01, "fp64", field)
        out.append(eng.hierarchy(0))
        cls = eng.classes()["items"]
        assert (cls[0] > 0) == generic
        eng.close()
    assert np.abs(out[0] - out[1]).max() < 1e-13
    assert np.abs(out[0][1:]).max() > 1e-4
