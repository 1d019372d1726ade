"""Constant-generator runs by powers of the RK4 step matrix (pyqed_liouville_run_work) against the
step-by-step kernel (pyqed_liouville_run) on the same inputs: tile edges in N and in the number of rows,
step counts around the largest power (64), every output form, and scratch shorter than the run.  Both are
FP64 with errors of at most about nsteps N eps relative to the largest element (200 x 64 x 1e-16 = 1.3e-12);
1e-12 is asserted up to N = 64 where typical errors are 1e-15."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _run(A, r0, nt, mode, power, dt=0.01, obs=None):
    import torch
    from pyqed_amd import _lib
    L = _lib.lib()
    dev = torch.device("cuda", 0)
    n, N = r0.shape
    t = lambda a: torch.as_tensor(np.ascontiguousarray(a), device=dev)  # noqa: E731
    At, rho, O = t(A), t(r0).clone(), t(obs)
    n_obs = O.shape[0] if mode in ("obs", "both") else 0
    ob = torch.zeros((n, nt + 1, max(n_obs, 1)), dtype=torch.complex128, device=dev)
    out = torch.zeros((n, nt, N), dtype=torch.complex128, device=dev) if mode in ("traj", "both") else None
    st = torch.cuda.current_stream().cuda_stream
    wb = _lib.C.c_int64()
    _lib.check(L.pyqed_liouville_work_bytes(N, 1, n, nt, n_obs, int(out is not None), 1, _lib.C.byref(wb)))
    assert wb.value > 0
    if power:
        work = torch.empty(wb.value, dtype=torch.uint8, device=dev)
        _lib.check(L.pyqed_liouville_run_work(N, 1, At.data_ptr(), n, rho.data_ptr(), None, nt, dt, n_obs, O.data_ptr(), ob.data_ptr(),
                                              _lib.ptr(out), 1, work.data_ptr(), work.numel(), st))
    else:
        _lib.check(L.pyqed_liouville_run(N, 1, At.data_ptr(), n, rho.data_ptr(), None, nt, dt, n_obs, O.data_ptr(), ob.data_ptr(),
                                         _lib.ptr(out), 1, st))
    return [x.cpu().numpy() for x in (rho, ob, out) if x is not None]


@pytest.mark.parametrize("mode", ["final", "obs", "traj", "both"])
@pytest.mark.parametrize("N,n,nt", [(1, 3, 100), (4, 1, 80), (9, 5, 63), (15, 2, 64), (16, 1, 65), (17, 3, 127), (33, 1, 128), (49, 2, 129),
                                    (64, 1, 4), (64, 40, 200), (9, 4096, 100), (33, 600, 70), (25, 4096, 180)])
def test_powers_equal_stepping(N, n, nt, mode):
    if mode in ("traj", "both") and n > 1000:
        nt = 70
    rng = np.random.default_rng([N, n, nt])
    A = (rng.normal(size=(N, N)) + 1j * rng.normal(size=(N, N))) / np.sqrt(N) - 1.5 * np.eye(N)
    r0 = rng.normal(size=(n, N)) + 1j * rng.normal(size=(n, N))
    obs = rng.normal(size=(3, N)) + 1j * rng.normal(size=(3, N))
    for a, b in zip(_run(A, r0, nt, mode, True, obs=obs), _run(A, r0, nt, mode, False, obs=obs)):
        assert np.abs(a - b).max() <= 1e-12 * np.abs(b).max()


def test_unexcited_unstable_mode_stays_zero():
    """A decoupled mode far beyond this dt's stability limit that the state never excites: its powers grow
    but stay finite, so the other modes are untouched and the mode itself is exactly zero."""
    A = np.diag([-0.3 + 1.0j, -0.1 - 2.0j, -2000.0 + 0j, -0.2 + 0j])
    r0 = np.array([[1.0, 0.5j, 0.0, -0.25]], complex)
    obs = np.ones((1, 4), complex)
    p, s = _run(A, r0, 300, "traj", True, obs=obs), _run(A, r0, 300, "traj", False, obs=obs)
    for a, b in zip(p, s):
        assert np.isfinite(a).all() and np.abs(a - b).max() <= 1e-12
    assert not p[0][0, 2]


def test_non_finite_generator_spreads():
    A = -np.eye(20, dtype=complex)
    A[3, 7] = np.nan
    r0 = np.ones((1, 20), complex)
    obs = np.ones((1, 20), complex)
    assert np.isnan(_run(A, r0, 40, "final", True, obs=obs)[0]).all()
