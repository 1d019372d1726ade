"""LDS-resident instances on 256 and on 1024 threads (more than 256 elements, at most as many as CUs), alone and
in one plan, against the streamed kernels: one element per thread, several, idle threads; entry lists of every
length modulo four; diagonal and dense couplings, packed and full state, a driven dipole.  20 steps: FP64 to
rounding (1e-12 on O(1) states), mixed to 20 dt eps_32 of the right-hand side (1e-6)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _inst(d, L, kind, seed):
    rng = np.random.default_rng([seed, d, L])
    H = rng.normal(size=(d, d)) + 1j * rng.normal(size=(d, d))
    q = rng.normal(size=(2, d, d))
    Q = (q + q.transpose(0, 2, 1)) / 4 if kind == "dense" else np.array([np.diag(v) for v in q[0]])[:2]
    etal = 0.2 * (rng.normal(size=3) + 1j * rng.normal(size=3))
    mode = np.array([0, len(Q) - 1, 0])
    v = rng.normal(size=d) + 1j * rng.normal(size=d)
    v /= np.linalg.norm(v)
    return dict(H=(H + H.conj().T) / 4, Q=Q.astype(complex), L=L, rho0=np.outer(v, v.conj()), sdip=np.eye(d, k=1) + np.eye(d, k=-1) + 0j,
                bath=(etal, etal.conj(), np.abs(etal), rng.uniform(0.5, 2.0, 3).astype(complex), mode))


@pytest.mark.parametrize("precision,tol", [("fp64", 1e-12), ("mixed", 1e-6)])
@pytest.mark.parametrize("packed", [True, False])
@pytest.mark.parametrize("kind", ["diag", "dense"])
@pytest.mark.parametrize("sizes", [[(2, 4)], [(2, 6)], [(3, 5)], [(5, 3)], [(2, 2), (3, 4), (4, 3), (2, 7), (8, 1)]])
def test_resident_equals_streamed(sizes, kind, packed, precision, tol):
    import torch
    from pyqed_amd.heom.engine import HeomEngine
    insts = [_inst(d, L, kind, 5) for d, L in sizes]
    field = torch.as_tensor(np.random.default_rng(1).normal(size=(20, 6)) * 0.3)
    field[:, 3:] = 0
    out = []
    for resident in (True, False):
        eng = HeomEngine(insts, resident=resident, **({} if packed else dict(packed=False)))
        assert eng.stats()["resident_instances"] == (len(insts) if resident else 0)
        traj = torch.zeros((5, eng.traj_stride), dtype=torch.complex128, device=eng.device)
        eng.advance(20, 0.01, precision, field.to(eng.device), traj, 4)
        torch.cuda.synchronize()
        out.append(traj.cpu().numpy())
    assert np.abs(out[0] - out[1]).max() <= tol
