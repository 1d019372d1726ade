"""Workloads of the open-system propagator, each through the entry points a program calls.

A case is a dict of plain values.  Its "kind" names the path:

  heom_run         DEOMSolver.run, the whole call (tables, plan, propagation, observable) of a d-level system
                   with one bath coupling: the spin-boson model and its few-level relatives
  heom             HeomEngine.advance of one exciton chain (one bath per site), from rho0, with trajectory rows
  heom_batch       the same for many uneven chains in one plan
  heom_gradient    HeomControl.gradient: forward run and streamed adjoint of a driven exciton chain
  lindblad_run     LindbladSolver.run of one small system: states and observables at every step
  lindblad_batch   LindbladSolver.run_batch: driven three-level systems, one field each
  lindblad_gradient  LindbladAdjoint.gradient of the driven three-level system
  redfield         RedfieldSolver.evolve of a damped oscillator
  cavity_batch     LindbladSolver.run_batch of a Kerr cavity, many coherent initial states (matrix form)
  cavity_emission  LindbladSolver.correlation_2op_1t of one Kerr cavity (matrix form)

Systems follow pyqed_amd/workloads.py: tridiagonal exciton chains with eps ~ N(0, 1), J ~ U(-0.5, 0.5),
Drude baths lambda ~ U(0.05, 0.5), gamma ~ U(0.2, 2), kT ~ U(0.5, 2) and one Pade pole; the driven
three-level Lambda system; the Kerr cavity of bench.py.
"""
import itertools
import math

import numpy as np
import torch

DT = 0.01
LAMBDA_DT = 0.05


def listed():
    return [
        # the smallest call: the textbook spin-boson run (21 ADOs of 2 x 2), 1000 steps, default precision
        dict(name="spin_boson_run", kind="heom_run", d=2, L=5, nt=1000, precision="fp64"),
        # a seven-site photosynthetic exciton (3060 ADOs of 7 x 7), the default precision, every 10th rho kept
        dict(name="exciton7_fp64", kind="heom", d=7, L=4, nt=200, precision="fp64", save_every=10, driven=False),
        # a sixteen-site aggregate (6545 ADOs of 16 x 16) in the default precision under a laser pulse
        dict(name="chain16_driven_fp64", kind="heom", d=16, L=3, nt=20, precision="fp64", save_every=1, driven=True),
        # one large hierarchy in mixed precision (20825 ADOs of 24 x 24)
        dict(name="chain24_mixed", kind="heom", d=24, L=3, nt=20, precision="mixed", save_every=5, driven=False),
        # ensemble average over static disorder: 512 uneven chains in one plan, mixed precision
        dict(name="batch512_mixed", kind="heom_batch", n=512, nt=6, precision="mixed", save_every=2),
        # optimal control: gradient with respect to site energies and 6 field amplitudes, 60 steps both ways
        dict(name="exciton7_gradient", kind="heom_gradient", d=7, L=3, nseg=6, sps=10, ckpt=20),
        # three coupled qubits with decay and dephasing, populations at every step
        dict(name="qubits3_run", kind="lindblad_run", d=8, nt=1000, driven=False),
        # a pulse-shape scan: 4096 fields on the three-level system, final states
        dict(name="lambda4096_driven", kind="lindblad_batch", n=4096, nt=1000),
        # optimal control of the three-level system: 50 amplitudes and 3 energies, 1000 steps both ways
        dict(name="lambda_gradient", kind="lindblad_gradient", nseg=50, sps=20, ckpt=50),
        # Bloch-Redfield relaxation of a 16-level oscillator (256 x 256 tensor)
        dict(name="redfield16", kind="redfield", d=16, nt=400),
        # 256 coherent initial states of a 64-level cavity
        dict(name="cavity64_batch", kind="cavity_batch", d=64, n=256, nt=40),
        # emission spectrum of one 96-level cavity: a single two-time correlation function
        dict(name="cavity96_emission", kind="cavity_emission", d=96, nt=100),
    ]


def draw(rng):
    def span(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["heom_run", "heom", "heom", "heom", "heom_batch", "heom_gradient", "lindblad_run", "lindblad_batch",
                       "lindblad_gradient", "redfield", "cavity_batch", "cavity_emission"])
    prec = rng.choice(["fp64", "mixed"])
    if kind == "heom_run":
        return dict(kind=kind, d=rng.randint(2, 4), L=rng.randint(2, 7), nt=span(150, 1500), precision=prec)
    if kind == "heom":
        d = rng.randint(2, 24)
        L = rng.randint(2, 5)
        while L > 2 and math.comb(2 * d + L, L) * d * d > 4e6:
            L -= 1
        cost = math.comb(2 * d + L, L) * d * d
        return dict(kind=kind, d=d, L=L, nt=max(3, min(span(20, 300), int(4e7 / cost))), precision=prec,
                    save_every=rng.choice([1, 2, 5]), driven=rng.random() < 0.3)
    if kind == "heom_batch":
        n = span(16, 256)
        return dict(kind=kind, n=n, nt=rng.randint(2, 6), precision=prec, save_every=rng.choice([1, 2]))
    if kind == "heom_gradient":
        return dict(kind=kind, d=rng.randint(3, 8), L=rng.randint(2, 3), nseg=rng.randint(2, 8), sps=rng.randint(3, 10),
                    ckpt=rng.choice([10, 20, 50]))
    if kind == "lindblad_run":
        return dict(kind=kind, d=span(2, 24), nt=span(100, 1000), driven=rng.random() < 0.4)
    if kind == "lindblad_batch":
        return dict(kind=kind, n=span(64, 4096), nt=span(200, 1000))
    if kind == "lindblad_gradient":
        return dict(kind=kind, nseg=span(5, 60), sps=rng.randint(5, 20), ckpt=rng.choice([20, 50, 100]))
    if kind == "redfield":
        return dict(kind=kind, d=span(3, 20), nt=span(50, 400))
    if kind == "cavity_batch":
        d = span(33, 80)
        return dict(kind=kind, d=d, n=max(8, min(span(16, 256), int(256 * (64 / d) ** 3))), nt=rng.randint(10, 40))
    return dict(kind=kind, d=span(33, 110), nt=rng.randint(20, 90))


# ------------------------------------------------------------------ inputs, from the seed alone
def _drude(lam, gam, beta):
    """Drude bath and one Pade pole: (etal, etar, etaa, expn)."""
    nu, r = 2.0 * math.sqrt(15.0), 2.5  # the [0/1] Pade pole and residue of the Bose function
    x = -1j * gam * beta
    bose = 1.0 / x + 0.5 + 2.0 * r * x / (x * x + nu * nu)
    nb = nu / beta
    etal = np.array([-2j * lam * gam * bose, 4.0 * r * lam * gam * nb / (beta * (nb * nb - gam * gam))], np.complex128)
    return etal, np.conj(etal), np.abs(etal), np.array([gam, nb], np.complex128)


def _ground(d):
    rho0 = np.zeros((d, d), np.complex128)
    rho0[0, 0] = 1.0
    return rho0


def _hop(d):
    return (np.diag(np.ones(d - 1), 1) + np.diag(np.ones(d - 1), -1)).astype(np.complex128)


def _chain(rng, d, L):
    """One exciton chain as an engine instance: d sites, one Drude bath per site (K = 2 d)."""
    H = np.diag(rng.normal(0.0, 1.0, d)).astype(np.complex128)
    J = rng.uniform(-0.5, 0.5, d - 1)
    H += np.diag(J, 1) + np.diag(J, -1)
    e = _drude(float(rng.uniform(0.05, 0.5)), float(rng.uniform(0.2, 2.0)), 1.0 / float(rng.uniform(0.5, 2.0)))
    Q = np.zeros((d, d, d), np.complex128)
    Q[np.arange(d), np.arange(d), np.arange(d)] = 1.0
    return dict(H=H, Q=Q, L=L, rho0=_ground(d), bath=tuple(np.tile(a, d) for a in e) + (np.repeat(np.arange(d), 2),))


def _pulse(rng, nt):
    """Field table [nt, 6] of a resonant pulse on the system dipole (columns: t, t + dt/2, t + dt)."""
    w, e0, t0 = rng.uniform(0.5, 2.0), rng.uniform(0.1, 0.5), 0.5 * nt * DT
    tab = np.zeros((nt, 6))
    for c, s in enumerate((0.0, 0.5, 1.0)):
        t = (np.arange(nt) + s) * DT
        tab[:, c] = e0 * np.exp(-((t - t0) / (0.3 * nt * DT)) ** 2) * np.cos(w * t)
    return tab


def _inputs(case, seed):
    rng = np.random.default_rng([seed, 77])
    kind = case["kind"]
    if kind == "heom_run":
        d = case["d"]
        H = rng.normal(0.0, 0.5, (d, d))
        return dict(H=(0.5 * (H + H.T)).astype(np.complex128), Q=np.diag(np.linspace(1.0, -1.0, d)).astype(np.complex128)[None],
                    bath=_drude(float(rng.uniform(0.05, 0.5)), float(rng.uniform(0.2, 2.0)), 1.0 / float(rng.uniform(0.5, 2.0)))
                    + (np.zeros(2, np.int64),), L=case["L"], rho0=_ground(d))
    if kind == "heom":
        inst = _chain(rng, case["d"], case["L"])
        field = None
        if case["driven"]:
            inst["sdip"] = _hop(case["d"])
            field = _pulse(rng, case["nt"])
        return dict(insts=[inst], field=field)
    if kind == "heom_batch":
        # shapes from the size alone, so that every seed costs the same; numbers from the seed
        shape = np.random.default_rng([case["n"], 5])
        return dict(insts=[_chain(rng, int(shape.integers(2, 17)), int(shape.integers(2, 5))) for _ in range(case["n"])],
                    field=None)
    if kind == "heom_gradient":
        d = case["d"]
        bar = np.zeros((d, d), np.complex128)
        bar[2, 2] = 1.0
        return dict(inst=_chain(rng, d, case["L"]), P=[np.diag(np.eye(d)[j]).astype(np.complex128) for j in range(d)],
                    mu=_hop(d), theta=rng.normal(0.0, 0.1, d), amps=rng.normal(0.0, 0.3, case["nseg"]), bar=bar)
    if kind == "lindblad_run":
        d = case["d"]
        H = rng.normal(0.0, 0.5, (d, d)) + 1j * rng.normal(0.0, 0.5, (d, d))
        H = 0.5 * (H + H.conj().T) / math.sqrt(d) * 2.0
        low = np.diag(np.sqrt(np.arange(1, d)), 1).astype(np.complex128)
        c_ops = [math.sqrt(rng.uniform(0.01, 0.1)) * low,
                 math.sqrt(rng.uniform(0.005, 0.05)) * np.diag(np.arange(d)).astype(np.complex128)]
        e_ops = [np.diag(np.eye(d)[0]).astype(np.complex128), np.diag(np.arange(d)).astype(np.complex128), low + low.T]
        return dict(H=H, H1=_hop(d), w=float(rng.uniform(0.5, 2.0)), c_ops=c_ops, e_ops=e_ops, rho0=_ground(d))
    if kind in ("lindblad_batch", "lindblad_gradient"):
        mu = np.array([[0, 1, 0], [1, 0, 0.7], [0, 0.7, 0]], np.complex128)
        c_ops = [math.sqrt(0.02) * np.diag(np.eye(3)[j]).astype(np.complex128) for j in range(3)]
        c_ops.append(np.zeros((3, 3), np.complex128))
        c_ops[3][0, 1] = math.sqrt(0.01)
        eps = np.array([0.0, 1.0, 2.5])
        if kind == "lindblad_gradient":
            bar = np.zeros((3, 3), np.complex128)
            bar[2, 2] = 1.0
            return dict(eps=eps, mu=mu, c_ops=c_ops, theta=eps + rng.normal(0.0, 0.05, 3),
                        amps=rng.normal(0.0, 0.1, (1, case["nseg"])), rho0=_ground(3), bar=bar)
        n, nt = case["n"], case["nt"]
        amps = rng.normal(0.0, 0.1, (n, -(-nt // 20)))
        return dict(H0=np.diag(eps).astype(np.complex128), mu=mu, c_ops=c_ops, rho0s=np.tile(_ground(3), (n, 1, 1)),
                    fields=np.ascontiguousarray(np.repeat(amps, 20, axis=1)[:, :nt, None]))
    if kind == "redfield":
        d = case["d"]
        a = np.diag(np.sqrt(np.arange(1, d)), 1)
        H = np.diag(0.5 * np.arange(d)) + 0.02 * (a + a.T) + np.diag(rng.normal(0.0, 0.02, d))
        v = rng.normal(size=d) + 1j * rng.normal(size=d)
        v /= np.linalg.norm(v)
        lam, gam, kT = float(rng.uniform(0.01, 0.05)), float(rng.uniform(0.5, 2.0)), float(rng.uniform(0.3, 1.0))
        return dict(H=H.astype(np.complex128), c_ops=[(a + a.T).astype(np.complex128) / math.sqrt(d)], bath=(lam, gam, kT),
                    rho0=np.outer(v, v.conj()), e_ops=[np.diag(np.arange(d)).astype(np.complex128), (a + a.T).astype(np.complex128)])
    d, n = case["d"], case.get("n", 1)
    a = np.diag(np.sqrt(np.arange(1, d)), 1).astype(np.complex128)
    num = a.conj().T @ a
    H = float(rng.uniform(0.5, 1.5)) * num + float(rng.uniform(0.002, 0.01)) * (num @ num)
    c_ops = [math.sqrt(float(rng.uniform(0.02, 0.08))) * a, math.sqrt(float(rng.uniform(0.001, 0.004))) * num]
    alpha = rng.uniform(1.0, 3.0, n) * np.exp(2j * np.pi * rng.uniform(size=n))
    k = np.arange(d)
    lg = np.array([math.lgamma(x + 1.0) for x in k])
    v = np.exp(k[None, :] * np.log(np.abs(alpha))[:, None] - 0.5 * lg[None, :]) * np.exp(1j * k[None, :] * np.angle(alpha)[:, None])
    v /= np.linalg.norm(v, axis=1, keepdims=True)
    return dict(H=H, c_ops=c_ops, a=a, rho0s=v[:, :, None] * v[:, None, :].conj())


CAVITY_DT = 0.002


def _spectrum(lam, gam, kT):
    """Quantum noise spectrum of a Drude bath, S(w) = 2 J(w) (n(w) + 1)."""
    def s(w):
        if abs(w) < 1e-9:
            return 4.0 * lam * kT / gam
        return 4.0 * lam * gam * w / (w * w + gam * gam) / (1.0 - math.exp(-w / kT))
    return s


def prepare(case, seed):
    x = _inputs(case, seed)
    kind = case["kind"]
    s = dict(case=case, x=x)
    if kind == "heom_run":
        from pyqed_amd.heom.deom import Bath, DEOMSolver
        s["solver"] = DEOMSolver(system=x["H"], bath=Bath.from_arrays(*x["bath"]), coupling=x["Q"], lmax=x["L"])
    elif kind in ("heom", "heom_batch"):
        from pyqed_amd.heom.engine import HeomEngine
        s["engine"] = eng = HeomEngine(x["insts"])
        s["field"] = None if x["field"] is None else torch.as_tensor(x["field"], device=eng.device)
        s["traj"] = torch.zeros((case["nt"] // case["save_every"], eng.traj_stride), dtype=torch.complex128, device=eng.device)
    elif kind == "heom_gradient":
        from pyqed_amd.heom.adjoint import HeomControl
        i = x["inst"]
        s["problem"] = HeomControl(i["H"], x["P"], x["mu"], i["Q"], i["bath"], i["L"], i["rho0"], DT, case["sps"],
                                   case["nseg"], ckpt_every=case["ckpt"])
    elif kind == "lindblad_run":
        from pyqed_amd.oqs import LindbladSolver
        w = x["w"]
        H = [x["H"], [x["H1"], lambda t: 0.2 * math.cos(w * t)]] if case["driven"] else x["H"]
        s["solver"] = LindbladSolver(H, x["c_ops"])
    elif kind == "lindblad_batch":
        from pyqed_amd.oqs import LindbladSolver
        s["solver"] = LindbladSolver([x["H0"], [x["mu"], None]], x["c_ops"])
    elif kind == "lindblad_gradient":
        from pyqed_amd.adjoint import lambda_system
        s["problem"] = lambda_system(x["eps"], x["mu"], x["c_ops"], LAMBDA_DT, case["sps"], case["nseg"], case["ckpt"])
    elif kind == "redfield":
        from pyqed_amd.oqs import RedfieldSolver
        s["solver"] = RedfieldSolver(x["H"], x["c_ops"], [_spectrum(*x["bath"])], x["e_ops"])
        s["solver"].redfield_tensor()
    else:
        from pyqed_amd.oqs import LindbladSolver
        s["solver"] = LindbladSolver(x["H"], x["c_ops"])
    return s


def run(s):
    case, x = s["case"], s["x"]
    kind = case["kind"]
    if kind == "heom_run":
        t, pop = s["solver"].run(x["rho0"], DT, case["nt"], p1=x["Q"][0], precision=case["precision"])
        return dict(t=t, pop=pop)
    if kind in ("heom", "heom_batch"):
        eng = s["engine"]
        eng.reset()
        eng.advance(case["nt"], DT, case["precision"], s["field"], s["traj"], case["save_every"])
        return dict(traj=s["traj"], state=eng.y)
    if kind == "heom_gradient":
        gt, ga, gr, _ = s["problem"].gradient(x["theta"], x["amps"], x["bar"])
        return dict(theta=gt, amps=ga, rho0=gr)
    if kind == "lindblad_run":
        r = s["solver"].run(x["rho0"], DT, case["nt"], e_ops=x["e_ops"])
        return dict(obs=r.observables, rho=np.array(r.rholist))
    if kind == "lindblad_batch":
        return dict(rho=s["solver"].run_batch(x["rho0s"], LAMBDA_DT, case["nt"], x["fields"]))
    if kind == "lindblad_gradient":
        gt, ga, gr = s["problem"].gradient(x["theta"], x["amps"], x["rho0"], x["bar"])
        return dict(theta=gt, amps=ga, rho0=gr)
    if kind == "redfield":
        r = s["solver"].evolve(x["rho0"], DT, case["nt"], e_ops=x["e_ops"])
        return dict(obs=r.observables, rho=np.array(r.rholist))
    if kind == "cavity_batch":
        return dict(rho=s["solver"].run_batch(x["rho0s"], CAVITY_DT, case["nt"]))
    return dict(cor=s["solver"].correlation_2op_1t(x["rho0s"][0], x["a"].conj().T, x["a"], CAVITY_DT, case["nt"], output=None))


# ------------------------------------------------------------------ what a pass cannot do without
def _heom_work(d, K, L, nt):
    """State (packed upper triangles, complex double) read and written once per step, or once in all where
    it fits the GPU's L2; per right-hand side one complex product H X (its adjoint is X H) and the row terms
    of every neighbour."""
    n = math.comb(K + L, L)
    nent = 2 * K * math.comb(K + L - 1, L - 1) if L else 0
    state = 16.0 * n * d * (d + 1) / 2
    return 2.0 * state * (nt if state > 32e6 else 1), 4.0 * nt * (8.0 * n * d ** 3 + 16.0 * nent * d)


def work(case):
    kind = case["kind"]
    b = f = 0.0
    if kind == "heom_run":
        d = case["d"]
        n = math.comb(2 + case["L"], 2)
        b, f = 16.0 * n * d * d + 24.0 * case["nt"], 4.0 * case["nt"] * n * (8.0 * d ** 3 + 4 * 16.0 * d * d)
    elif kind == "heom":
        b, f = _heom_work(case["d"], 2 * case["d"], case["L"], case["nt"])
    elif kind == "heom_batch":
        for i in _inputs(case, 0)["insts"]:
            d = i["H"].shape[0]
            b += 32.0 * math.comb(2 * d + i["L"], i["L"]) * d * (d + 1) / 2
            f += _heom_work(d, 2 * d, i["L"], case["nt"])[1]
        b *= case["nt"] if b > 64e6 else 1
    elif kind == "heom_gradient":
        db, df = _heom_work(case["d"], 2 * case["d"], case["L"], case["nseg"] * case["sps"])
        b, f = 2.0 * db, 3.0 * 2.0 * df  # full matrices; forward, recomputation, adjoint
    elif kind in ("lindblad_run", "redfield"):
        N, nt = case["d"] ** 2, case["nt"]
        b, f = 16.0 * (N * N + N * nt), 32.0 * N * N * nt
    elif kind == "lindblad_batch":
        b, f = case["n"] * (8.0 * case["nt"] + 2 * 144.0), 32.0 * 2 * 81 * case["n"] * case["nt"]
    elif kind == "lindblad_gradient":
        nt = case["nseg"] * case["sps"]
        b, f = 16.0 * nt, 4.0 * 32 * 2 * 81 * nt
    else:
        d, n, nt = case["d"], case.get("n", 1), case["nt"]
        b, f = 2 * 16.0 * n * d * d, 4.0 * 6 * 8 * d ** 3 * n * nt
    return dict(bytes=b, flops=f)


# ------------------------------------------------------------------ the same results in 64 bits, plain torch
_TABLES = {}


def _hierarchy(K, L):
    """(keys [n, K], entries): multi-indices in combinadic order (rank sum_i C(s_i + i, i + 1), s_i the prefix
    sums) and, as arrays, target ADO, neighbour ADO, exponential, sqrt factor and whether it is n + e_k."""
    if (K, L) in _TABLES:
        return _TABLES[K, L]
    comb = np.array([[math.comb(i, j) for j in range(K + 2)] for i in range(K + L + 2)], np.int64)

    def rank(keys):
        s = np.cumsum(keys, axis=1)
        i = np.arange(K)
        return comb[s + i, i + 1].sum(axis=1)

    keys = []
    for t in range(L + 1):
        for c in itertools.combinations_with_replacement(range(K), t):
            k = [0] * K
            for q in c:
                k[q] += 1
            keys.append(k)
    keys = np.array(keys, np.int64).reshape(-1, K)
    keys = keys[np.argsort(rank(keys))]
    tier = keys.sum(axis=1)
    cols = [[], [], [], [], []]
    for k in range(K):
        for plus, sel in ((0, np.nonzero(keys[:, k] > 0)[0]), (1, np.nonzero(tier < L)[0])):
            nb = keys[sel].copy()
            nb[:, k] += 1 if plus else -1
            for col, v in zip(cols, (sel, rank(nb), np.full(sel.size, k), np.sqrt(keys[sel, k] + plus), np.full(sel.size, plus))):
                col.append(v)
    _TABLES[K, L] = keys, [np.concatenate(c) for c in cols]
    return _TABLES[K, L]


class _Heom:
    """Right-hand side of one instance on torch complex128 (differentiable in H and X)."""

    def __init__(self, inst, dev):
        self.dev = dev
        etal, etar, etaa, expn, mode = inst["bath"]
        self.d = d = inst["H"].shape[0]
        keys, (tgt, nb, k, sq, plus) = _hierarchy(len(mode), inst["L"])
        self.n = keys.shape[0]
        t = lambda a: torch.as_tensor(np.ascontiguousarray(a), device=dev)  # noqa: E731
        self.damp = t(keys @ expn)[:, None, None]
        sa = np.sqrt(np.asarray(etaa, np.complex128))
        cl = np.where(plus == 1, -1j * sa[k], -1j * etal[k] / sa[k]) * sq
        cr = np.where(plus == 1, 1j * sa[k], 1j * etar[k] / sa[k]) * sq
        q = np.array([np.diag(m) for m in inst["Q"]])
        self.site = q.shape[0] == d and np.array_equal(q, np.eye(d))
        if self.site:  # a neighbour entering through site s adds to row s and column s
            s = np.asarray(mode)[k]
            self.at, self.of = t(tgt * d + s), t(nb * d + s)
            self.cl, self.cr = t(cl)[:, None], t(cr)[:, None]
        else:
            self.at, self.of = t(tgt), t(nb)
            qm = q[np.asarray(mode)[k]]
            self.w = t(cl[:, None, None] * qm[:, :, None] + cr[:, None, None] * qm[:, None, :])
        self.H = t(inst["H"])
        self.rho0 = t(inst["rho0"])

    def _add(self, out, at, v):
        n = out.shape[0]
        return torch.view_as_complex(torch.view_as_real(out).reshape(n, -1)
                                     .index_add(0, at, torch.view_as_real(v).reshape(v.shape[0], -1)).reshape(n, -1, 2))

    def rhs(self, H, X):
        n, d = self.n, self.d
        out = -1j * (torch.matmul(H, X.transpose(0, 1).reshape(d, n * d)).reshape(d, n, d).transpose(0, 1)
                     - torch.matmul(X.reshape(n * d, d), H).reshape(n, d, d)) - self.damp * X
        if self.site:
            out = self._add(out.reshape(n * d, d), self.at, self.cl * X.reshape(n * d, d)[self.of]).reshape(n, d, d)
            Xt = X.transpose(1, 2).reshape(n * d, d)
            col = self._add(torch.zeros_like(Xt), self.at, self.cr * Xt[self.of])
            return out + col.reshape(n, d, d).transpose(1, 2)
        v = (self.w * X[self.of]).reshape(-1, d * d)
        return self._add(out.reshape(n, d * d), self.at, v).reshape(n, d, d)

    def start(self, rho0=None):
        X = torch.zeros((self.n, self.d, self.d), dtype=torch.complex128, device=self.dev)
        return torch.cat([(self.rho0 if rho0 is None else rho0)[None], X[1:]])


def _rk4(f, y, dt):
    """One step of y' = f(c, y), c = 0, 1, 2 at t, t + dt/2, t + dt."""
    k1 = f(0, y)
    k2 = f(1, y + k1 * (dt / 2))
    k3 = f(1, y + k2 * (dt / 2))
    k4 = f(2, y + k3 * dt)
    return y + (k1 + 2 * k2 + 2 * k3 + k4) * (dt / 6)


def _exact_heom(inst, field, nt, save_every, dev):
    h = _Heom(inst, dev)
    mu = torch.as_tensor(inst["sdip"], device=dev) if field is not None else None
    y, rows = h.start(), []
    for s in range(nt):
        Hs = [h.H if field is None else h.H + mu * float(field[s, c]) for c in range(3)]
        y = _rk4(lambda c, X: h.rhs(Hs[c], X), y, DT)
        if (s + 1) % save_every == 0:
            rows.append(y[0].reshape(-1).clone())
    return rows, y


def _lindblad(H, c_ops):
    d = H.shape[0]
    eye = np.eye(d)
    A = -1j * (np.kron(H, eye) - np.kron(eye, H.T))
    for c in c_ops:
        cc = c.conj().T @ c
        A = A + np.kron(c, c.conj()) - 0.5 * (np.kron(cc, eye) + np.kron(eye, cc.T))
    return A


def _drive(H1):
    eye = np.eye(H1.shape[0])
    return 1j * (np.kron(H1, eye) - np.kron(eye, H1.T))


def _redfield(H, c_ops, spectrum):
    E, V = np.linalg.eigh(H)
    eye = np.eye(len(E))
    R = -1j * (np.kron(np.diag(E), eye) - np.kron(eye, np.diag(E)))
    for a in c_ops:
        A = V.conj().T @ a @ V
        C = np.array([[spectrum(-(p - q)) for q in E] for p in E])
        Lk = C * A
        R = R - (np.kron(A, eye) - np.kron(eye, A.T)) @ (np.kron(Lk, eye) - np.kron(eye, Lk.conj()))
    return R, V


def exact(case, seed):
    x = _inputs(case, seed)
    kind = case["kind"]
    dev = torch.device("cuda") if torch.cuda.is_available() else torch.device("cpu")
    if kind == "heom_run":
        rows, _ = _exact_heom(x, None, case["nt"], 1, dev)
        rho = np.concatenate([x["rho0"].reshape(1, -1), torch.stack(rows).cpu().numpy()]).reshape(-1, case["d"], case["d"])
        return dict(t=np.arange(case["nt"] + 1) * DT, pop=np.einsum("ij,tji->t", x["Q"][0], rho))
    if kind in ("heom", "heom_batch"):
        traj, state, at = [], [], 0
        for inst in x["insts"]:
            rows, y = _exact_heom(inst, x["field"], case["nt"], case["save_every"], dev)
            d = y.shape[1]
            traj.append(torch.stack(rows))
            pad = -at % 8  # instances start on 128-byte boundaries of the state
            iu = torch.triu_indices(d, d, device=dev)
            state += [torch.zeros(pad, dtype=y.dtype, device=dev), y[:, iu[0], iu[1]].reshape(-1)]
            at += pad + state[-1].numel()
        return dict(traj=torch.cat(traj, dim=1), state=torch.cat(state))
    if kind == "heom_gradient":
        h = _Heom(x["inst"], dev)
        d = case["d"]
        theta = torch.tensor(x["theta"], device=dev, requires_grad=True)
        amps = torch.tensor(x["amps"], device=dev, requires_grad=True)
        rho0 = torch.tensor(x["inst"]["rho0"], device=dev, requires_grad=True)
        mu = torch.as_tensor(x["mu"], device=dev)
        H = h.H + torch.diag(theta).to(torch.complex128)
        y = h.start(rho0)
        for s in range(case["nseg"]):
            Ht = H + amps[s] * mu
            for _ in range(case["sps"]):
                y = _rk4(lambda c, X: h.rhs(Ht, X), y, DT)
        y[0, 2, 2].real.backward()
        return dict(theta=theta.grad, amps=amps.grad, rho0=rho0.grad)
    if kind == "lindblad_run":
        nt, d = case["nt"], case["d"]
        A0 = torch.as_tensor(_lindblad(x["H"], x["c_ops"]), device=dev)
        A1 = torch.as_tensor(_drive(x["H1"]), device=dev)
        v = torch.as_tensor(x["rho0"].reshape(-1), device=dev)
        out = [v]
        for k in range(nt):
            A = A0 + 0.2 * math.cos(x["w"] * (k + 1) * DT) * A1 if case["driven"] else A0
            v = _rk4(lambda c, u: A @ u, v, DT)
            out.append(v)
        out = torch.stack(out).cpu().numpy().reshape(nt + 1, d, d)
        obs = np.stack([np.einsum("ij,tji->t", e, out) for e in x["e_ops"]], axis=1)
        return dict(obs=obs[1:] if case["driven"] else obs, rho=out[1:])
    if kind == "lindblad_batch":
        A0 = torch.as_tensor(_lindblad(x["H0"], x["c_ops"]).T.copy(), device=dev)
        A1 = torch.as_tensor(_drive(x["mu"]).T.copy(), device=dev)
        v = torch.as_tensor(x["rho0s"].reshape(-1, 9), device=dev)
        f = torch.as_tensor(x["fields"], device=dev)
        for k in range(case["nt"]):
            v = _rk4(lambda c, u: u @ A0 + f[:, k] * (u @ A1), v, LAMBDA_DT)
        return dict(rho=v.cpu().numpy().reshape(-1, 3, 3))
    if kind == "lindblad_gradient":
        base = torch.as_tensor(_lindblad(np.zeros((3, 3)), x["c_ops"]))
        G = torch.as_tensor(np.array([-_drive(np.diag(np.eye(3)[j])) for j in range(3)]))
        B = torch.as_tensor(_drive(x["mu"]))
        theta = torch.tensor(x["theta"], requires_grad=True)
        amps = torch.tensor(x["amps"], requires_grad=True)
        rho0 = torch.tensor(x["rho0"], requires_grad=True)
        A0 = base + torch.tensordot(theta.to(torch.complex128), G, dims=1)
        v = rho0.reshape(-1)
        for s in range(case["nseg"]):
            A = A0 + amps[0, s] * B
            for _ in range(case["sps"]):
                v = _rk4(lambda c, u: A @ u, v, LAMBDA_DT)
        v[8].real.backward()
        return dict(theta=theta.grad, amps=amps.grad, rho0=rho0.grad)
    if kind == "redfield":
        d = case["d"]
        R, V = _redfield(x["H"], x["c_ops"], _spectrum(*x["bath"]))
        R = torch.as_tensor(R, device=dev)
        v = torch.as_tensor((V.conj().T @ x["rho0"] @ V).reshape(-1), device=dev)
        out = []
        for _ in range(case["nt"]):
            v = _rk4(lambda c, u: R @ u, v, DT)
            out.append(v)
        out = torch.stack(out).cpu().numpy().reshape(-1, d, d)
        obs = np.stack([np.einsum("ij,tji->t", V.conj().T @ e @ V, out) for e in x["e_ops"]], axis=1)
        return dict(obs=obs, rho=V @ out @ V.conj().T)
    d = case["d"]
    H = torch.as_tensor(x["H"], device=dev)
    cs = [torch.as_tensor(c, device=dev) for c in x["c_ops"]]
    G = H - 0.5j * sum(c.conj().T @ c for c in cs)

    def rhs(_, r):
        n = r.shape[0]

        def left(m, r):
            return torch.matmul(m, r.transpose(0, 1).reshape(d, n * d)).reshape(d, n, d).transpose(0, 1)

        def right(r, m):
            return torch.matmul(r.reshape(n * d, d), m).reshape(n, d, d)

        out = -1j * left(G, r) + 1j * right(r, G.conj().T.contiguous())
        for c in cs:
            out = out + left(c, right(r, c.conj().T.contiguous()))
        return out

    if kind == "cavity_batch":
        r = torch.as_tensor(x["rho0s"], device=dev)
        for _ in range(case["nt"]):
            r = _rk4(rhs, r, CAVITY_DT)
        return dict(rho=r.cpu().numpy())
    a = torch.as_tensor(x["a"], device=dev)
    r = (a @ torch.as_tensor(x["rho0s"][0], device=dev))[None]
    cor = []
    for _ in range(case["nt"]):
        r = _rk4(rhs, r, CAVITY_DT)
        cor.append(torch.sum(a.conj().T.T * r[0]))  # Tr(a^dag r)
    return dict(cor=torch.stack(cor).cpu().numpy())
