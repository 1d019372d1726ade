"""Forms of the packed projector kernel for a class that holds one hierarchy: a block per item, and fewer
blocks that run through their items with one header and a prefetch across items; against the table-driven
kernel, which the hierarchy runs beside a second one of its class.  VALU, 16 x 16 and 2 x 2 MFMA classes, one
and several ADOs per wavefront, last items of every remainder.  The arithmetic of an ADO is the same in all
forms: mixed runs agree bit for bit, FP64 ones to 20 steps of rounding (1e-13 on O(1) states)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _inst(d, L, seed):
    from pyqed_amd.heom.bath import drude
    rng = np.random.default_rng(seed)
    A = rng.normal(size=(d, d)) + 1j * rng.normal(size=(d, d))
    Q = np.array([np.diag(np.eye(d)[j] * 0.8) for j in range(d)]).astype(complex)
    bath = tuple(np.tile(x, d) for x in drude(0.3, 0.8, 1.2, 1)) + (np.repeat(np.arange(d), 2),)
    v = rng.normal(size=d) + 1j * rng.normal(size=d)
    v /= np.linalg.norm(v)
    return dict(H=(A + A.conj().T) / 4, Q=Q, L=L, rho0=np.outer(v, v.conj()), bath=bath)


@pytest.mark.parametrize("precision", ["mixed", "fp64"])
@pytest.mark.parametrize("per,bpc", [(1, 16), (1, 1), (3, 1)])
@pytest.mark.parametrize("d,L,cls", [(7, 4, 1), (11, 3, 1), (12, 3, 2), (16, 3, 2), (17, 3, 3), (21, 3, 3)])
def test_single_forms_match_table_form(d, L, cls, per, bpc, precision):
    """(1, 1) and (3, 1): at most a block per CU and more than 256 items, the looping form; (1, 16): the form
    the launch has room for."""
    from pyqed_amd.heom.engine import HeomEngine
    a, b = _inst(d, L, 400 + d), _inst(d, L, 500 + d)
    out = []
    for insts in ([a], [a, b]):
        eng = HeomEngine(insts, resident=False)
        eng.autotune_cache = False
        eng.set_tiling(4 * per * d * d, bpc, 0)
        assert eng.packed and (eng.class_single()[cls] == 0) == (len(insts) == 1)
        if len(insts) == 1 and (per, bpc) == (1, 1):
            assert eng.classes()["items"][cls] > 256
        out.append(eng.run(0.01, 20, precision, save_every=5)[0])
    if precision == "mixed":
        assert np.array_equal(out[0], out[1])
    else:
        assert np.abs(out[0] - out[1]).max() <= 1e-13


@pytest.mark.parametrize("d,L,sites", [(6, 2, 3), (6, 5, 2), (8, 3, 8), (10, 2, 7), (11, 3, 5)])
@pytest.mark.parametrize("precision", ["mixed", "fp64"])
def test_small_sites_in_any_order(d, L, sites, precision):
    """d <= 11: exponentials that are not listed in site order, sites without a bath, complex H, a driven
    dipole, and ADO counts of every remainder modulo a block's four."""
    import torch
    from pyqed_amd.heom.engine import HeomEngine
    rng = np.random.default_rng(7 * d + L)
    insts = []
    for k in range(2):
        inst = _inst(d, L, 700 + d + k)
        where = rng.permutation(d)[:sites]
        inst["Q"] = inst["Q"][where]
        pick = rng.permutation(2 * sites)  # exponentials of coupling m // 2, in any order
        inst["bath"] = tuple(np.asarray(x)[pick] for x in inst["bath"][:4]) + (np.repeat(np.arange(sites), 2)[pick],)
        inst["sdip"] = np.eye(d, k=1) + np.eye(d, k=-1) + 0j
        insts.append(inst)
    field = torch.as_tensor(rng.normal(size=(20, 6)) * 0.3)
    field[:, 3:] = 0
    out = []
    for group in (insts[:1], insts):
        eng = HeomEngine(group, resident=False)
        assert eng.packed and (eng.class_single()[1] == 0) == (len(group) == 1)
        traj = torch.zeros((4, eng.traj_stride), dtype=torch.complex128, device=eng.device)
        eng.advance(20, 0.01, precision, field.to(eng.device), traj, 5)
        torch.cuda.synchronize()
        out.append(traj.cpu().numpy()[:, :d * d])
    if precision == "mixed":
        assert np.array_equal(out[0], out[1])
    else:
        assert np.abs(out[0] - out[1]).max() <= 1e-13
