"""Gradients with all stage inputs kept, a segment's kept, and none (the limit set below one state): the same
adjoint in three memory regimes, over one and several sweeps of 32 steps, partial last segments, the VALU, MFMA
and generic classes and a resident instance.  FP64 throughout, at most 71 steps: 1e-12 relative."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _problem(d, L, nt, ck):
    from pyqed_amd.heom.adjoint import HeomAdjoint
    from pyqed_amd.heom.bath import drude
    rng = np.random.default_rng(60 + d)
    H = np.diag(rng.normal(size=d)).astype(complex) + 0.3 * (np.eye(d, k=1) + np.eye(d, k=-1))
    Q = np.array([np.diag(np.eye(d)[j] * 0.8) for j in range(d)]).astype(complex)
    bath = tuple(np.tile(x, d) for x in drude(0.3, 0.8, 1.2, 1)) + (np.repeat(np.arange(d), 2),)
    rho0 = np.zeros((d, d), complex)
    rho0[0, 0] = 1.0
    mu = np.eye(d, k=1) + np.eye(d, k=-1) + 0j
    insts = [dict(H=H, Q=Q, L=L, rho0=rho0, bath=bath, sdip=mu), dict(H=H.conj() + 0.1 * mu, Q=Q, L=2, rho0=rho0, bath=bath, sdip=mu)]
    return HeomAdjoint(insts, 0.02, nt, ckpt_every=ck), rng.normal(size=(nt, 6)) * 0.3


@pytest.mark.parametrize("d,L,nt,ck", [(2, 3, 71, 40), (3, 4, 33, 7), (7, 3, 32, 9), (9, 2, 1, 5), (13, 2, 9, 4), (18, 2, 5, 2)])
def test_kept_stage_inputs_do_not_change_gradients(d, L, nt, ck):
    ref = None
    bar = [np.diag(np.arange(1.0, d + 1)) + 0.2j * np.eye(d, k=1), np.ones((d, d)) + 0j]
    for states in (0, 4 * min(ck, nt), 4 * nt):
        prob, field = _problem(d, L, nt, ck)
        prob.keep_bytes = 16 * prob.fwd.n_elems * states
        r = prob.gradient(bar, field)
        prob.close()
        got = [np.concatenate([np.ravel(r[k][i]) for i in range(2)]) for k in ("rho", "gH", "grho0", "G", "gfield")]
        if ref is None:
            ref = got
        for a, b in zip(got, ref):
            assert np.abs(a - b).max() <= 1e-12 * np.abs(b).max()
