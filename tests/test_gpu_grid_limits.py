"""Launches whose threads would pass 2^32, the number a grid can hold: observables of many instances in matrix form, and of
many rows of runs by powers.  Against torch's matrix products, both FP64: n eps of the sums of n products, with a margin."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_many_observables_in_matrix_form():
    import torch
    from pyqed_amd import _lib
    L, dev = _lib.lib(), torch.device("cuda")
    d, n, n_obs = 65, 2050, 8400          # 17.2e6 workgroups of 256
    assert n * n_obs * 256 > 2 ** 32
    g = torch.Generator(device=dev).manual_seed(1)
    H = torch.diag(torch.linspace(-1, 1, d, dtype=torch.float64, device=dev)).to(torch.complex128)
    rho = torch.randn((n, d * d), dtype=torch.complex128, device=dev, generator=g) / d
    obs = torch.randn((n_obs, d * d), dtype=torch.complex128, device=dev, generator=g)
    out = torch.zeros((n, 2, n_obs), dtype=torch.complex128, device=dev)
    wb = _lib.C.c_int64()
    _lib.check(L.pyqed_lindblad_work_bytes(d, 0, 0, n, _lib.C.byref(wb)))
    work = torch.empty(wb.value, dtype=torch.uint8, device=dev)
    start = rho.clone()
    _lib.check(L.pyqed_lindblad_run(d, 0, H.data_ptr(), H.data_ptr(), None, None, 0, None, None, n, rho.data_ptr(), None, 1, 0.01, n_obs,
                                    obs.data_ptr(), out.data_ptr(), None, 1, work.data_ptr(), work.numel(),
                                    torch.cuda.current_stream().cuda_stream))
    ot = obs.T.contiguous()
    for row, state in ((0, start), (1, rho)):
        assert (out[:, row] - state @ ot).abs().max().item() <= 1e-12 * d


def test_many_rows_by_powers():
    import torch
    from pyqed_amd import _lib
    L, dev = _lib.lib(), torch.device("cuda")
    N, n, nt = 33, 4096, 16400            # 64 lanes a row
    assert n * nt * 64 > 2 ** 32
    if torch.cuda.mem_get_info()[0] < 60 << 30:
        pytest.skip("needs 60 GB of device memory")
    rng = np.random.default_rng(2)
    A = torch.as_tensor((rng.normal(size=(N, N)) + 1j * rng.normal(size=(N, N))) / np.sqrt(N) - 1.5 * np.eye(N), device=dev) * 0.01
    rho = torch.as_tensor(rng.normal(size=(n, N)) + 1j * rng.normal(size=(n, N)), device=dev)
    obs = torch.as_tensor(rng.normal(size=(1, N)) + 0j, device=dev)
    out = torch.full((n, nt + 1, 1), float("nan"), dtype=torch.complex128, device=dev)
    states = torch.empty((n, nt, N), dtype=torch.complex128, device=dev)
    wb = _lib.C.c_int64()
    _lib.check(L.pyqed_liouville_work_bytes(N, 1, n, nt, 1, 1, 1, _lib.C.byref(wb)))
    work = torch.empty(wb.value, dtype=torch.uint8, device=dev)
    _lib.check(L.pyqed_liouville_run_work(N, 1, A.data_ptr(), n, rho.data_ptr(), None, nt, 0.01, 1, obs.data_ptr(), out.data_ptr(),
                                          states.data_ptr(), 1, work.data_ptr(), work.numel(), torch.cuda.current_stream().cuda_stream))
    o = obs[0].contiguous()
    for i in (0, 1, 2047, 4000, 4094, 4095):
        want = states[i] @ o
        assert (out[i, 1:, 0] - want).abs().max().item() <= 1e-12 * N
    assert not torch.isnan(torch.view_as_real(out)).any()
