"""V rho V^dagger over runs of matrices against numpy: the smallest and largest d, more matrices than one grid
holds.  Sums of d products of O(1) terms: 1e-13."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d,n", [(1, 3), (2, 70000), (5, 1), (16, 400), (17, 9), (31, 3), (32, 20)])
def test_basis_change(d, n):
    import torch
    from pyqed_amd import _lib
    from pyqed_amd.liouville import change_basis
    rng = np.random.default_rng(d)
    V = (rng.normal(size=(d, d)) + 1j * rng.normal(size=(d, d))) / np.sqrt(d)
    rho = (rng.normal(size=(n, d, d)) + 1j * rng.normal(size=(n, d, d))) / d
    t = torch.as_tensor(rho.copy(), device="cuda")
    change_basis(torch, _lib.lib(), V, t)
    torch.cuda.synchronize()
    assert np.abs(t.cpu().numpy() - V @ rho @ V.conj().T).max() <= 1e-13
    assert _lib.lib().pyqed_basis_change(33, 1, t.data_ptr(), t.data_ptr(), None) != 0
