"""What a HEOM gradient holds of the device's memory: the stage inputs of both directions and the contraction's workspace
together stay within HeomAdjoint.keep_bytes."""
import numpy as np
import pytest


@pytest.mark.parametrize("state", [16, 5 * 10**5, 3 * 10**7, 2 * 10**9])
@pytest.mark.parametrize("nt,ckpt", [(0, 50), (1, 50), (7, 3), (33, 50), (60, 20), (1000, 50), (5000, 7)])
@pytest.mark.parametrize("contraction", [0, 10**4, 10**8])
def test_kept_steps_fit(nt, ckpt, state, contraction):
    from pyqed_amd.heom.adjoint import HeomAdjoint
    for keep in (0, 6 * state, 100 * state, 4 << 30):
        seg, b = HeomAdjoint.kept_steps(nt, ckpt, state, contraction, keep)
        if b:
            m = min(seg, nt)
            assert seg in (nt, ckpt) and 1 <= b <= min(m, 32)
            assert (4 * m + 1) * state + (4 * b + 1) * state + state + b * contraction <= keep
        else:
            assert seg == ckpt


@pytest.mark.gpu
@pytest.mark.parametrize("limit,kept", [(300, True), (100, True), (20, False)])
def test_gradient_holds_no_more_than_its_limit(limit, kept):
    import torch
    from pyqed_amd.heom.adjoint import HeomAdjoint
    from pyqed_amd.heom.bath import drude
    d, nt, ck = 7, 60, 10
    rng = np.random.default_rng(4)
    H = np.diag(rng.normal(size=d)).astype(complex) + 0.3 * (np.eye(d, k=1) + np.eye(d, k=-1))
    Q = np.array([np.diag(np.eye(d)[j]) for j in range(d)]).astype(complex)
    bath = tuple(np.tile(x, d) for x in drude(0.3, 0.8, 1.2, 1)) + (np.repeat(np.arange(d), 2),)
    rho0 = np.zeros((d, d), complex)
    rho0[0, 0] = 1.0
    prob = HeomAdjoint([dict(H=H, Q=Q, L=3, rho0=rho0, bath=bath)], 0.02, nt, ckpt_every=ck)
    state = 16 * prob.fwd.n_elems
    bar = [np.eye(d, k=1) + 0j]
    prob.keep_bytes = 0
    want = prob.gradient(bar)
    torch.cuda.synchronize()
    base = torch.cuda.memory_allocated()
    torch.cuda.reset_peak_memory_stats()
    prob.keep_bytes = limit * state
    assert bool(prob.kept_steps(nt, ck, state, prob._wb, prob.keep_bytes)[1]) == kept
    got = prob.gradient(bar)
    # beside the limit: checkpoints, the contraction's results and (where nothing is kept) one segment of states
    other = (nt // ck + ck + 10) * state + 16 * 3 * nt * prob.fwd.traj_stride + (1 << 20)
    assert torch.cuda.max_memory_allocated() - base <= prob.keep_bytes + other
    for a, b in ((got["gH"][0], want["gH"][0]), (got["grho0"][0], want["grho0"][0])):
        assert np.abs(a - b).max() <= 1e-12 * np.abs(b).max()
    prob.close()
