"""Matrix-form Lindblad kernel at the edges of its tiles and block tables: d around multiples of 16 and 32,
both tile forms (16 x 16 split four ways, 32 x 32 once 256 workgroups fill the chip), operators with
all-zero, purely real and purely imaginary 16 x 16 blocks, driven and static, against the oracle's dense
FP64 products.  FP64: every element is a sum of at most a few thousand products of O(1) terms scaled by
dt, so 1e-12 on unit-trace states leaves two decades over rounding."""
import numpy as np
import pytest

from oracle import lindblad as OL

pytestmark = pytest.mark.gpu


def _problem(d, n, kind, seed):
    rng = np.random.default_rng([seed, d])
    a = np.diag(np.sqrt(np.arange(1, d)) / np.sqrt(max(d, 2)), 1).astype(complex)
    num = np.diag(np.arange(d) / d).astype(complex)
    if kind == "ladder":      # banded real operators: most blocks are zero
        H, c = num + 0.3 * (a + a.T), [0.4 * a, 0.2 * num]
    elif kind == "corner":    # one imaginary block far off the diagonal, one empty operator
        H = num.copy()
        if d > 1:
            H[0, d - 1], H[d - 1, 0] = 0.3j, -0.3j
        c = [np.zeros((d, d), complex), 0.3j * a]
    else:                     # dense
        m = rng.normal(size=(d, d)) + 1j * rng.normal(size=(d, d))
        H = (m + m.conj().T) / (2 * np.sqrt(d))
        c = [0.3 / np.sqrt(d) * (rng.normal(size=(d, d)) + 1j * rng.normal(size=(d, d)))]
    v = rng.normal(size=(n, d)) + 1j * rng.normal(size=(n, d))
    v /= np.linalg.norm(v, axis=1, keepdims=True)
    return H, c, v[:, :, None] * v[:, None, :].conj()


@pytest.mark.parametrize("kind", ["ladder", "corner", "dense"])
@pytest.mark.parametrize("d,n", [(1, 2), (15, 1), (16, 3), (17, 1), (31, 2), (32, 1), (33, 1), (48, 2), (49, 1), (17, 1024), (33, 256), (64, 256), (80, 115)])
def test_tiles_and_zero_blocks(d, n, kind):
    from pyqed_amd.oqs import LindbladSolver
    H, c, rhos = _problem(d, n, kind, 3)
    nt = 6
    final = LindbladSolver(H, c, form="matrix").run_batch(rhos, 0.02, nt)
    for i in sorted({0, n // 2, n - 1}):
        ref = OL.run(H, c, rhos[i], 0.02, nt)
        err = np.abs(final[i] - ref["rholist"][-1]).max()
        assert err < 1e-12, (d, n, kind, i, err)


@pytest.mark.parametrize("d,n", [(20, 2), (64, 256)])
def test_driven_zero_blocks(d, n):
    """The drive fills blocks that the static Hamiltonian leaves empty."""
    from pyqed_amd.oqs import LindbladSolver
    H, c, rhos = _problem(d, n, "ladder", 4)
    H1 = np.zeros((d, d), complex)
    H1[0, d - 1], H1[d - 1, 0] = 0.5j, -0.5j
    f = np.random.default_rng(1).normal(size=(n, 5, 1))
    final = LindbladSolver([H, [H1, None]], c, form="matrix").run_batch(rhos, 0.02, 5, f)
    for i in (0, n - 1):
        ref = OL.run_driven([H, [H1, lambda t: f[i, int(round(t / 0.02)) - 1, 0]]], rhos[i], c, 0.02, 5, e_ops=[])
        assert np.abs(final[i] - np.array(ref["rholist"])[-1]).max() < 1e-12


def test_non_finite_input_spreads():
    """0 x NaN is NaN in a full product: a NaN in rho0 reaches every element although the operators' blocks
    are mostly zero."""
    from pyqed_amd.oqs import LindbladSolver
    H, c, rhos = _problem(64, 1, "ladder", 5)
    rhos[0, 3, 50] = np.nan
    final = LindbladSolver(H, c, form="matrix").run_batch(rhos, 0.02, 1)
    assert np.isnan(final).all()


def test_without_block_tables():
    """A workspace of pyqed_lindblad_work_bytes alone (no room for the tables): the full products, equal to
    the run that skips zero blocks up to rounding."""
    import torch
    from pyqed_amd import _lib
    from pyqed_amd.oqs import LindbladSolver
    L = _lib.lib()
    for d, n in ((20, 3), (40, 2), (64, 128), (100, 1)):
        H, c, rhos = _problem(d, n, "ladder", 6)
        want = LindbladSolver(H, c, form="matrix").run_batch(rhos, 0.02, 3)
        t = lambda a: torch.as_tensor(np.ascontiguousarray(a), device="cuda")  # noqa: E731
        Heff = H - 0.5j * sum(x.conj().T @ x for x in c)
        ops = [t(Heff), t(Heff.conj().T), t(np.array(c)), t(np.array([x.conj().T for x in c]))]
        rho = t(rhos)
        wb = _lib.C.c_int64()
        _lib.check(L.pyqed_lindblad_work_bytes(d, len(c), 0, n, _lib.C.byref(wb)))
        work = torch.empty(wb.value, dtype=torch.uint8, device="cuda")
        _lib.check(L.pyqed_lindblad_run(d, len(c), *(o.data_ptr() for o in ops), 0, None, None, n, rho.data_ptr(), None, 3, 0.02, 0, None,
                                        None, None, 1, work.data_ptr(), wb.value, torch.cuda.current_stream().cuda_stream))
        assert np.abs(rho.cpu().numpy() - want).max() < 1e-13
