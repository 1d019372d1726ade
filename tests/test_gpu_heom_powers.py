"""Small hierarchies by powers of their dense generator (FP64, no field, 64 steps or more in a call) against
the LDS-resident kernel (shorter calls) on the same engine: diagonal and dense couplings, packed and full
state, non-Hermitian bath coefficients, the adjoint plan, segment ends (1024 rows) and trajectory strides.
Both are FP64 with errors of about nsteps eps on O(1) states: 1e-12."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _instance(d, L, kind, seed=1):
    rng = np.random.default_rng([seed, d, L])
    H = rng.normal(size=(d, d)) + 1j * rng.normal(size=(d, d))
    H = (H + H.conj().T) / 4
    K = 2
    etal = 0.2 * (rng.normal(size=K) + 1j * rng.normal(size=K))
    etar, expn, mode = etal.conj(), rng.uniform(0.5, 2.0, K).astype(complex), np.zeros(K, int)
    Q = np.diag(np.linspace(1.0, -1.0, d)).astype(complex)[None]
    if kind == "dense":   # two couplings that do not commute
        m = rng.normal(size=(d, d))
        Q, mode = np.array([Q[0], (m + m.T) / 4]).astype(complex), np.array([0, 1])
    if kind == "complex":
        expn = expn + 1j * np.array([0.7, -0.7])
    v = rng.normal(size=d) + 1j * rng.normal(size=d)
    v /= np.linalg.norm(v)
    return dict(H=H, Q=Q, L=L, rho0=np.outer(v, v.conj()), bath=(etal, etar, np.abs(etal), expn, mode))


@pytest.mark.parametrize("kind,layout", [("diag", {}), ("diag", dict(packed=False)), ("dense", {}), ("complex", {}),
                                         ("diag", dict(hermitian=False, packed=False, adjoint=True))])
@pytest.mark.parametrize("d,L,nt,every", [(1, 2, 64, 1), (2, 5, 130, 7), (2, 2, 1100, 3), (3, 6, 70, 70), (4, 7, 100, 33)])
def test_powers_equal_resident(d, L, nt, every, kind, layout):
    import torch
    from pyqed_amd.heom.engine import HeomEngine
    inst = _instance(d, L, kind)
    eng = HeomEngine([inst], **layout)
    N = int(eng.nmax[0]) * d * d
    assert eng.stats()["resident_instances"] == 1 and N <= 640
    traj = [torch.full((nt // every, d * d), 7.0, dtype=torch.complex128, device=eng.device) for _ in range(2)]
    eng.advance(nt, 0.01, "fp64", None, traj[0], every)
    got = eng.hierarchy(0)
    eng.reset()
    for s in range(nt // every):       # one saved step at a time, in calls too short for powers
        left = every
        while left:
            m = min(left, 50)
            left -= m
            eng.advance(m, 0.01, "fp64", None, traj[1][s:s + 1] if not left else None, m)
    if nt % every:
        eng.advance(nt % every, 0.01, "fp64")
    want = eng.hierarchy(0)
    assert np.abs(got - want).max() <= 1e-12 * max(1.0, np.abs(want).max())
    assert (traj[0] - traj[1]).abs().max().item() <= 1e-12 * max(1.0, np.abs(want).max())
    eng.close()
