"""A plan with one LDS-resident hierarchy of more than 256 elements more than the GPU has CUs, where all of them share one
launch of 256 threads each, against the streamed kernels, and with one fewer, where the large ones take 1024 threads in a
launch of their own.  Tiny hierarchies among them.  20 steps: FP64 to rounding (1e-12 on O(1) states), mixed to 20 dt
eps_32 of the right-hand side (1e-6)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _inst(d, L, seed):
    rng = np.random.default_rng([seed, d, L])
    H = rng.normal(size=(d, d)) + 1j * rng.normal(size=(d, d))
    etal = 0.2 * (rng.normal(size=2) + 1j * rng.normal(size=2))
    v = rng.normal(size=d) + 1j * rng.normal(size=d)
    v /= np.linalg.norm(v)
    return dict(H=(H + H.conj().T) / 4, Q=np.diag(rng.normal(size=d)).astype(complex)[None], L=L, rho0=np.outer(v, v.conj()),
                bath=(etal, etal.conj(), np.abs(etal), rng.uniform(0.5, 2.0, 2).astype(complex), np.zeros(2, int)))


@pytest.mark.parametrize("precision,tol", [("fp64", 1e-12), ("mixed", 1e-6)])
@pytest.mark.parametrize("extra", [0, 1])
def test_more_large_ones_than_cus(extra, precision, tol):
    import torch
    from pyqed_amd.heom.engine import HeomEngine
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    insts = []
    for k in range(cus + extra):              # 21 ADOs of 4 x 4: 336 elements, and a few of 36 of 3 x 3
        insts.append(_inst(4, 5, k) if k % 5 else _inst(3, 7, k))
        if k % 7 == 0:
            insts.append(_inst(2, 2, 1000 + k))
    out = []
    for resident in (True, False):
        eng = HeomEngine(insts, resident=resident)
        assert eng.stats()["resident_instances"] == (len(insts) if resident else 0)
        traj = torch.zeros((4, eng.traj_stride), dtype=torch.complex128, device=eng.device)
        eng.advance(20, 0.01, precision, None, traj, 5)
        out.append(traj.cpu().numpy())
        eng.close()
    assert np.abs(out[0] - out[1]).max() <= tol
