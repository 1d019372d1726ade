"""Register-form Liouville kernels (N <= 16): forward runs and gradients of driven systems, whole chains and
chains cut along time, against a numpy RK4 (phys.py:1051-1063) and its autograd in torch, both FP64 on the
CPU.  Rounding grows as nsteps N eps (about 5e-13 at the largest shape here); 1e-11 of the largest value is
asserted, and whole and cut runs are compared at the same tolerance."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _problem(N, nterm, n, nt, seed=0):
    rng = np.random.default_rng([seed, N, nterm, n, nt])
    A = (rng.normal(size=(nterm, N, N)) + 1j * rng.normal(size=(nterm, N, N))) / np.sqrt(N)
    A[0] -= 1.5 * np.eye(N)
    r0 = rng.normal(size=(n, N)) + 1j * rng.normal(size=(n, N))
    return A, r0, 0.3 * rng.normal(size=(n, nt, nterm - 1)), rng.normal(size=(n, N)) + 1j * rng.normal(size=(n, N))


def _reference(A, r0, f, bar, dt):
    """States after every step, and the gradients of Re sum conj(bar) v(T)."""
    import torch
    At = [torch.tensor(a, requires_grad=True) for a in A]
    ft, vt = torch.tensor(f, requires_grad=True), torch.tensor(r0, requires_grad=True)
    n, nt, nt1 = f.shape
    S = torch.stack([torch.stack(At)] * n)  # per-instance copies, so that their gradients come apart
    S.retain_grad()
    v, out = vt, []
    for s in range(nt):
        M = S[:, 0] + sum((ft[:, s, i, None, None] * S[:, i + 1] for i in range(nt1)), 0)
        mul = lambda u: torch.matmul(M, u[..., None])[..., 0]  # noqa: E731
        k1 = mul(v)
        k2 = mul(v + k1 * (dt / 2))
        k3 = mul(v + k2 * (dt / 2))
        k4 = mul(v + k3 * dt)
        v = v + (k1 + 2 * k2 + 2 * k3 + k4) / 6 * dt
        out.append(v.detach().numpy())
    torch.real(torch.sum(torch.conj(torch.tensor(bar)) * v)).backward()
    return np.array(out).transpose(1, 0, 2), ft.grad.numpy(), S.grad.numpy(), vt.grad.numpy()


def _gpu(A, r0, f, bar, dt, cut, ckpt=7):
    import torch
    from pyqed_amd import _lib
    L = _lib.lib()
    st = torch.cuda.current_stream().cuda_stream
    n, nt, nt1 = f.shape
    nterm, N, _ = A.shape
    t = lambda a: torch.as_tensor(np.ascontiguousarray(a), device="cuda")  # noqa: E731
    At, ft, bt, rho = t(A), t(f), t(bar), t(r0).clone()
    obs = t(np.eye(N, dtype=complex)[:2])
    n_obs = obs.shape[0]
    ob = torch.zeros((n, nt + 1, n_obs), dtype=torch.complex128, device="cuda")
    out = torch.zeros((n, nt, N), dtype=torch.complex128, device="cuda")
    wb = _lib.C.c_int64()
    fp = ft.data_ptr() if nt1 else None
    common = (N, nterm, At.data_ptr(), n, rho.data_ptr(), fp, nt, dt, n_obs, obs.data_ptr(), ob.data_ptr(), out.data_ptr(), 1)
    if cut:
        _lib.check(L.pyqed_liouville_work_bytes(N, nterm, n, nt, n_obs, 1, 1, _lib.C.byref(wb)))
        assert wb.value > 0
        work = torch.empty(wb.value, dtype=torch.uint8, device="cuda")
        _lib.check(L.pyqed_liouville_run_work(*common, work.data_ptr(), wb.value, st))
    else:
        _lib.check(L.pyqed_liouville_run(*common, st))
    gf = torch.zeros((n, nt, max(nt1, 1)), dtype=torch.float64, device="cuda")
    gA = torch.zeros((n, nterm, N, N), dtype=torch.complex128, device="cuda")
    r0b = torch.zeros((n, N), dtype=torch.complex128, device="cuda")
    start = t(r0)
    _lib.check(L.pyqed_liouville_adjoint_work_bytes(N, nterm, n, nt, ckpt, _lib.C.byref(wb)))
    nck = (nt + ckpt - 1) // ckpt + 1
    size = wb.value if cut else n * (nck + ckpt) * N * 16
    work = torch.empty(size, dtype=torch.uint8, device="cuda")
    fn = L.pyqed_liouville_adjoint_work if cut else L.pyqed_liouville_adjoint
    _lib.check(fn(N, nterm, At.data_ptr(), n, start.data_ptr(), fp, nt, dt, ckpt, bt.data_ptr(), gf.data_ptr(), gA.data_ptr(),
                  r0b.data_ptr(), work.data_ptr(), size, st))
    return [x.cpu().numpy() for x in (out, gf, gA, r0b, ob, rho)]


@pytest.mark.parametrize("cut", [False, True])
@pytest.mark.parametrize("N,nterm,n,nt", [(1, 2, 1, 30), (2, 2, 3, 31), (4, 2, 17, 40), (4, 4, 1, 65), (5, 2, 2, 33), (9, 2, 1, 100),
                                          (9, 3, 5, 71), (10, 2, 1, 48), (16, 2, 3, 90), (16, 3, 1, 37)])
def test_forward_and_gradients(N, nterm, n, nt, cut):
    A, r0, f, bar = _problem(N, nterm, n, nt)
    states, gf, gA, g0 = _reference(A, r0, f, bar, 0.02)
    out = _gpu(A, r0, f, bar, 0.02, cut)
    for got, want in zip(out[:4], (states, gf, gA, g0)):
        assert np.abs(got - want).max() <= 1e-11 * max(np.abs(want).max(), 1.0)
    full = np.concatenate([r0[:, None], states], axis=1)
    assert np.abs(out[4] - full[:, :, [0, 1][:out[4].shape[2]]]).max() <= 1e-11
    assert np.abs(out[5] - states[:, -1]).max() <= 1e-11


def test_a_drive_at_zero_is_left_out():
    """A generator with an infinite entry whose drive is zero in every step does not enter."""
    A, r0, f, bar = _problem(9, 3, 2, 20)
    f[:, :, 1] = 0.0
    want = _gpu(A, r0, f, bar, 0.02, False)[0]
    A[2, 3, 4] = np.inf
    assert np.array_equal(_gpu(A, r0, f, bar, 0.02, False)[0], want)


def test_many_instances_cut_and_whole():
    """Enough instances that the number of segments is set by the room on the chip."""
    A, r0, f, bar = _problem(9, 2, 300, 60)
    for a, b in zip(_gpu(A, r0, f, bar, 0.02, True), _gpu(A, r0, f, bar, 0.02, False)):
        assert np.abs(a - b).max() <= 1e-11 * max(np.abs(b).max(), 1.0)
