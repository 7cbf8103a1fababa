"""Timed cases of the scattering operator: what a user's program has it do,
from the smallest evaluation to the largest that fits a quick preparation.

A case is a dict of plain values.  "kind" names the path:

  eval      one right-hand side dRho/dt|scatt, state and result on the GPU
  driver    evolve_driver with host arrays and an explicit 1 - rho: the call
            the reference's dm_dynamics makes, through a band window
  rk4       integrate_rk4 with observable reports, state on the GPU
  rkf45     one tstep of the adaptive integrator (the reference's default)
            from a host state, with the coherent term, and the spin measured
  batched   eval_batched: B trajectories share one pass over P
  adjoint   forward RK4, then the discrete adjoint of an observable loss with
            respect to the weights of P's components and the initial state
  ee        the Pee_update rebuild: P = base + P_ee(rho), then one right-hand
            side with it

Common keys: nb, nk, partners (drawn per k; 0: every pair k <= k', as a dense
window of k points gives), prec (0 complex128 P, 1 complex64, 2 BF16), steps.
P is drawn in the Gram form the initializer writes, energies over 0.1 eV at
300 K, states near equilibrium with a small spin imbalance.
"""
import math

import numpy as np
import torch

from denmat_dynm_development_amd import scatt

FS = 41.341373335182  # 1 fs in Hartree atomic time
T300 = 9.50043e-4     # k_B 300 K
EMAX = 3.67e-3        # 0.1 eV
RATE = 1e-4           # scattering rate of a k point, about 4 per ps
CHUNK = 1 << 19       # pairs of P generated at a time (nb = 2; fewer for nb = 4)


def listed():
    return [
        # one right-hand side of a tiny operator: latency and launches alone
        dict(name="eval_nb2_nk64", kind="eval", nb=2, nk=64, partners=8, prec=0),
        # the GaAs example's own shape: 941 k points, every pair of them, two
        # e-ph bands in a six-band density matrix, rkf45 over one tstep
        dict(name="rkf45_gaas_nk941", kind="rkf45", nb=2, nk=941, partners=0, prec=0, nb_dm=6),
        # the drop-in seam: host density matrix in and out, ragged nk
        dict(name="driver_host_nk10007", kind="driver", nb=2, nk=10007, partners=100, prec=0, nb_dm=4),
        # reference-size dynamics, reports every 5 steps
        dict(name="rk4_nb2_nk4096", kind="rk4", nb=2, nk=4096, partners=250, prec=0, steps=20, report=5, linear=0),
        # the linearized operator (alg_linearize) at an odd size
        dict(name="rk4_linear_nk8191", kind="rk4", nb=2, nk=8191, partners=120, prec=0, steps=5, report=5, linear=1),
        # a large one-GPU operator, bound by the stream of P
        dict(name="rk4_nb2_nk32768", kind="rk4", nb=2, nk=32768, partners=480, prec=0, steps=2, report=1, linear=0),
        # two spin pairs of bands, FP64
        dict(name="rk4_nb4_nk5003", kind="rk4", nb=4, nk=5003, partners=120, prec=0, steps=2, report=1, linear=0),
        # the BF16 store, one trajectory
        dict(name="rk4_nb4_bf16_nk9001", kind="rk4", nb=4, nk=9001, partners=180, prec=2, steps=2, report=1, linear=0),
        # trajectories in a batch on uneven rows (partners 10 .. 10 x this, power law)
        dict(name="batched_bf16_B16", kind="batched", nb=4, nk=6000, partners=250, prec=2, B=16),
        dict(name="batched_c64_B50", kind="batched", nb=4, nk=4001, partners=250, prec=1, B=50),
        # gradients: forward and backward through 8 steps, three components of P
        dict(name="adjoint_nb2_nk4096", kind="adjoint", nb=2, nk=4096, partners=120, prec=0, steps=8, comps=3,
             checkpoint=8),
        # the e-e P rebuilt at the state on a 12 x 12 x 12 mesh
        dict(name="ee_rebuild_mesh12", kind="ee", nb=2, nk=1728, partners=60, prec=0, mesh=12),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["eval", "eval", "rkf45", "driver", "rk4", "rk4", "rk4", "batched", "adjoint", "ee"])
    if kind == "eval":
        nb = rng.choice([2, 2, 4])
        nk = _log(rng, 40, 20000 if nb == 2 else 2000)
        return dict(kind=kind, nb=nb, nk=nk, partners=min(nk // 3, _log(rng, 4, 250)), prec=0)
    if kind == "rkf45":
        dense = rng.random() < 0.5
        nk = _log(rng, 60, 1200) if dense else _log(rng, 300, 12000)
        return dict(kind=kind, nb=2, nk=nk, partners=0 if dense else min(nk // 3, _log(rng, 20, 200)), prec=0,
                    nb_dm=rng.choice([2, 4, 6]))
    if kind == "driver":
        nk = _log(rng, 200, 12000)
        return dict(kind=kind, nb=2, nk=nk, partners=min(nk // 3, _log(rng, 20, 150)), prec=0,
                    nb_dm=rng.choice([2, 4, 6]))
    if kind == "rk4":
        nb = rng.choice([2, 2, 4])
        prec = 0 if nb == 2 else rng.choice([0, 1, 2])
        nk = _log(rng, 100, 25000 if nb == 2 else 6000)
        case = dict(kind=kind, nb=nb, nk=nk, partners=min(nk // 3, _log(rng, 15, 300 if nb == 2 else 120)), prec=prec,
                    steps=rng.randint(1, 10), report=rng.choice([0, 1, 5]),
                    linear=int(prec == 0 and rng.random() < 0.25))
        while case["steps"] > 1 and work(case)["bytes"] > 5e10:
            case["steps"] -= 1
        return case
    if kind == "batched":
        nk = _log(rng, 200, 5000)
        return dict(kind=kind, nb=4, nk=nk, partners=min(nk // 5, _log(rng, 15, 200)), prec=rng.choice([1, 2]),
                    B=_log(rng, 2, 64))
    if kind == "adjoint":
        nk, steps = _log(rng, 100, 4000), rng.randint(2, 9)
        return dict(kind=kind, nb=2, nk=nk, partners=min(nk // 3, _log(rng, 20, 110)), prec=0, steps=steps,
                    comps=rng.randint(1, 3), checkpoint=rng.choice([steps, max(1, steps // 2)]))
    m = rng.randint(5, 11)
    return dict(kind="ee", nb=2, nk=m ** 3, partners=rng.randint(10, 50), prec=0, mesh=m)


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _gen(seed, tag):
    g = torch.Generator(device="cuda")
    g.manual_seed((int(seed) * 1000003 + tag) % (1 << 62))
    return g


def _pairs(case, seed):
    """Stored pairs k1 <= k2, sorted, on the GPU."""
    nk, c = case["nk"], case["partners"]
    if c == 0:
        ij = torch.triu_indices(nk, nk, device="cuda")
        return ij[0].contiguous(), ij[1].contiguous()
    g = _gen(seed, 1)
    k = torch.arange(nk, device="cuda")
    if case["kind"] == "batched":  # rows of 10 .. 10 c partners, density ~ 1 / count
        lo, hi = min(10.0, c / 2.0), min(10.0 * c, nk / 2.0)
        cnt = lo * torch.exp(torch.rand(nk, generator=g, device="cuda", dtype=torch.float64) * math.log(hi / lo))
        k = torch.repeat_interleave(k, cnt.long())
    else:
        k = k.repeat_interleave(c)
    q = torch.randint(0, nk, k.shape, generator=g, device="cuda")
    code = torch.minimum(k, q) * nk + torch.maximum(k, q)
    if case.get("linear"):  # the linearized operator keeps a row's own term in its (k, k) pair
        code = torch.cat([code, torch.arange(nk, device="cuda") * (nk + 1)])
    code = torch.unique(code)
    return code // nk, code % nk


def _p_chunks(case, seed, n_pairs, tag=100):
    """(first, P1, P2) of the stored pairs in chunks, Gram form, sized so that
    every k point scatters at about RATE."""
    nb, nk = case["nb"], case["nk"]
    step = CHUNK if nb <= 2 else CHUNK // 8
    amp = math.sqrt(RATE * nk / (2 * math.pi) * nk / (2.0 * n_pairs) / nb)
    for c, first in enumerate(range(0, n_pairs, step)):
        n = min(step, n_pairs - first)
        g = _gen(seed, tag * 100003 + c)
        w = amp * torch.exp(-(2 * torch.rand(n, 1, 1, generator=g, device="cuda", dtype=torch.float64)) ** 2)
        P1 = P2 = 0
        for _ in range(2):
            A = torch.randn(n, nb, nb, generator=g, device="cuda", dtype=torch.complex128) * w
            B = torch.randn(n, nb, nb, generator=g, device="cuda", dtype=torch.complex128) * w
            # P1[(i1 i2),(i3 i4)] = A[i1,i3] conj(A[i2,i4]), P2 = B[i3,i1] conj(B[i4,i2])
            P1 = P1 + A[:, :, None, :, None] * A.conj()[:, None, :, None, :]
            Bt = B.transpose(1, 2)
            P2 = P2 + Bt[:, :, None, :, None] * Bt.conj()[:, None, :, None, :]
        yield first, P1.reshape(n, nb ** 4), P2.reshape(n, nb ** 4)


def _energies(nk, nb, rng):
    """Kramers pairs: band edge over EMAX, splitting up to 5 meV, second pair above."""
    e = np.empty((nk, nb))
    for b in range(0, nb, 2):
        base = rng.uniform(0, EMAX, nk) if b == 0 else e[:, b - 2] + rng.uniform(7e-4, 2.2e-3, nk)
        e[:, b] = base
        if b + 1 < nb:
            e[:, b + 1] = base + rng.uniform(0, 1.8e-4, nk)
    return e


def _herm(nk, nb, rng):
    A = rng.normal(size=(nk, nb, nb)) + 1j * rng.normal(size=(nk, nb, nb))
    return (A + A.conj().transpose(0, 2, 1)) / 2


def _state(e, mu, rng, amp):
    """diag f plus a Hermitian imbalance of amp f (1 - f)."""
    nk, nb = e.shape
    f = 1 / (np.exp((e - mu) / T300) + 1)
    w = np.sqrt((f * (1 - f))[:, :, None] * (f * (1 - f))[:, None, :])
    rho = f[:, :, None] * np.eye(nb) + amp * w * _herm(nk, nb, rng)
    return rho.reshape(nk, nb * nb), f


def _host_inputs(case, seed):
    """Everything but P and the pairs, as numpy arrays."""
    rng = np.random.default_rng(int(seed) * 7919 + 17)
    nk, nb = case["nk"], case["nb"]
    nbd = case.get("nb_dm", nb)
    b0 = nbd - nb
    e = _energies(nk, nb, rng)
    edm = np.empty((nk, nbd))
    edm[:, b0:] = e
    edm[:, :b0] = -0.05 + rng.uniform(-2e-3, 0, (nk, b0))
    mu = 0.5 * EMAX if case["kind"] == "ee" else 0.1 * EMAX
    rho, f = _state(edm, mu, rng, 0.02)
    s = _herm(nk, nbd, rng)
    s[:, :b0, b0:] = 0  # no valence-conduction elements (alg_set_scv_zero)
    s[:, b0:, :b0] = 0
    s = s.reshape(nk, nbd * nbd)
    d = dict(e=e, edm=edm, rho=rho, f=f, s=s, b0=b0, nbd=nbd)
    if case["kind"] == "rkf45":  # a small field on the spin: the coherent term
        d["H"] = 2e-6 * s
    if case["kind"] == "batched":
        states = [_state(e, mu, rng, 0.002 * 10 ** rng.uniform(0, 1.5))[0] for _ in range(case["B"])]
        d["rho"] = np.stack(states)
    if case["kind"] == "ee":
        m = case["mesh"]
        g = np.stack(np.meshgrid(*[np.arange(m)] * 3, indexing="ij"), -1).reshape(-1, 3)
        d["kvec"] = g / float(m)
        nw = 4
        d["U"] = (rng.normal(size=(nk, nw, nb)) + 1j * rng.normal(size=(nk, nw, nb))) / 2
    if case["kind"] == "adjoint":
        d["target"] = rng.normal(size=case["steps"] + 1) * 1e-3
    return d


EE_R = np.array([[0.0, 5.34145, 5.34145], [5.34145, 0.0, 5.34145], [5.34145, 5.34145, 0.0]])
EE_DEGAUSS, EE_ETHR, EE_EPS = 1.84e-4, 1e-3, 12.9


def _ee_model(case, d):
    V = abs(np.linalg.det(EE_R))
    n_free = d["f"].sum() / (case["nk"] * V)
    return scatt.eimp_model("debye", n_free, T300, V, scatt.reciprocal_metric(EE_R), d["U"].shape[1], n_ionized=1.0,
                            epsilon_background=EE_EPS, degauss=EE_DEGAUSS, ethr=EE_ETHR,
                            kmesh=(case["mesh"],) * 3, nk_full=float(case["nk"]))


def _operator(case, seed, k1, k2, e, tag=100):
    op = scatt.ScatteringOperator(case["nk"], case["nb"], k1, k2, e, nk_full=case["nk"], precision=case["prec"])
    for first, P1, P2 in _p_chunks(case, seed, len(k1), tag):
        torch.cuda.synchronize()  # the handle copies on its own stream
        op.upload_P_range(first, P1, P2)
    return op


def prepare(case, seed):
    d = _host_inputs(case, seed)
    g1, g2 = _pairs(case, seed)
    k1, k2 = g1.cpu().numpy().astype(np.uint64), g2.cpu().numpy().astype(np.uint64)
    kind, nk, nb = case["kind"], case["nk"], case["nb"]
    s = dict(case=dict(case), kind=kind, d=d, t=17 * FS)
    if kind == "adjoint":
        s["comps"] = [_operator(case, seed, k1, k2, d["e"], 100 + c) for c in range(case["comps"])]
        op = scatt.ScatteringOperator(nk, nb, k1, k2, d["e"], nk_full=nk)
        op.combine_P(s["comps"], np.ones(case["comps"]))
    else:
        op = _operator(case, seed, k1, k2, d["e"])
    if d["nbd"] != nb:
        op.set_window(d["nbd"], d["b0"], d["edm"])
    if case["prec"]:
        op.set_split(d["f"])
    if case.get("linear"):
        op.set_Lsc(d["f"])
    if kind in ("rk4", "rkf45", "adjoint"):
        op.set_observable(d["s"], d["f"], d["b0"], d["nbd"], 1.0 / nk)
    if kind == "rkf45":
        op.set_coherent(d["H"])
    if kind == "ee":
        s["base"] = op
        op = scatt.ScatteringOperator(nk, nb, k1, k2, d["e"], nk_full=nk)
        s["model"], s["k1"], s["k2"] = _ee_model(case, d), k1, k2
        s["dm1"] = np.eye(nb).reshape(-1) - d["rho"]
    if kind == "driver":
        s["dm1"] = np.eye(d["nbd"]).reshape(-1) - d["rho"]
    if kind in ("eval", "rk4", "batched", "ee"):
        s["rho"] = torch.from_numpy(d["rho"]).cuda()
        s["out"] = torch.empty_like(s["rho"])
    else:
        s["rho"] = d["rho"]
    s["op"] = op
    torch.cuda.synchronize()
    return s


def run(s):
    op, case, kind = s["op"], s["case"], s["kind"]
    if kind == "eval":
        return op.eval(s["t"], s["rho"], out=s["out"])
    if kind == "driver":
        return op.evolve_driver(s["t"], s["rho"], s["dm1"])
    if kind == "batched":
        return op.eval_batched(s["t"], s["rho"], out=s["out"])
    if kind == "rk4":
        return op.integrate_rk4(s["rho"], s["t"], FS, case["steps"], case["report"])
    if kind == "rkf45":
        rho, t, _, _ = op.rkf45_apply(s["rho"], s["t"], s["t"] + FS, FS, hmin=0.0, hmax=FS, eps_abs=1e-8)
        return rho, op.measure(t, rho)
    if kind == "adjoint":
        n = case["steps"]
        rho, obs = op.integrate_rk4(s["rho"], s["t"], FS, n, 1)
        dth, drho = op.adjoint_rk4(s["rho"], s["t"], FS, n, 1, case["checkpoint"], obs - s["d"]["target"], s["comps"])
        return rho, obs, dth, drho
    d = s["d"]
    op.copy_P_from(s["base"])
    op.add_ee_model_state(s["k1"], s["k2"], d["U"], d["kvec"], d["f"], s["model"], dm=d["rho"], dm1=s["dm1"], add=True)
    return op.eval(s["t"], s["rho"], out=s["out"])


def _n_pairs(case):
    """Stored pairs of the case, in the mean over seeds."""
    nk, c = case["nk"], float(case["partners"])
    if c == 0:
        return nk * (nk + 1) // 2
    if case["kind"] == "batched":
        lo, hi = min(10.0, c / 2.0), min(10.0 * c, nk / 2.0)
        c = (hi - lo) / math.log(hi / lo)
    m = nk * (nk + 1) / 2.0
    return int(m * (1 - math.exp(-nk * c / m)))


def work(case):
    """P once per right-hand side (the stages depend on one another), the
    states read and written once each; per pair and trajectory 32 nb^4 flops."""
    np_, nb, nk, kind = _n_pairs(case), case["nb"], case["nk"], case["kind"]
    pair = 2 * nb ** 4 * (16, 8, 4)[case["prec"]] + 8
    state = nk * case.get("nb_dm", nb) ** 2 * 16
    steps = case.get("steps", 1)
    rhs = {"rk4": 4 * steps, "rkf45": 6, "adjoint": 12 * steps}.get(kind, 1)
    B = case.get("B", 1)
    fl = 32.0 * nb ** 4 * np_ * rhs * B
    if kind == "adjoint":
        fl *= 1.7  # a VJP forms the right-hand side's sums and their transposes
    by = rhs * np_ * pair + 2.0 * B * state
    if kind == "ee":
        # base P read, P written and read; per (pair, k3) inside the window (about
        # half) 16 Gaussians of ~20 flops and two 4 x 4 complex forms
        by = 3.0 * np_ * pair
        fl += np_ * nk * 0.5 * (16 * 20 + 2 * 400)
    return {"bytes": float(by), "flops": float(fl)}


# ---------------------------------------------------------------------------
# the same results from plain torch in 64 bits
# ---------------------------------------------------------------------------
def _rhs_S(P, k1, k2, rho, prefac):
    """prefac/2 (C + C^+) at the Schroedinger-picture state rho (nk, nb, nb).
    P: list of (first, P1, P2)."""
    nk, nb = rho.shape[0], rho.shape[1]
    n2 = nb * nb
    eye = torch.eye(nb, dtype=rho.dtype, device=rho.device)
    one = (eye - rho).reshape(nk, n2)
    r = rho.reshape(nk, n2)
    F1 = torch.zeros(nk, n2, dtype=rho.dtype, device=rho.device)
    F2 = torch.zeros_like(F1)
    for first, P1, P2 in P:
        a, b = k1[first:first + len(P1)], k2[first:first + len(P1)]
        A1, A2 = P1.reshape(-1, n2, n2), P2.reshape(-1, n2, n2)
        rev = (a < b).to(r.real.dtype)[:, None]
        F1 = F1.index_add(0, a, (A1 * r[b][:, None, :]).sum(2))
        F2 = F2.index_add(0, a, (A2 * one[b][:, :, None]).sum(1))
        F1 = F1.index_add(0, b, (A2.conj() * r[a][:, None, :]).sum(2) * rev)
        F2 = F2.index_add(0, b, (A1.conj() * one[a][:, :, None]).sum(1) * rev)
    F1, F2 = F1.reshape(nk, nb, nb), F2.reshape(nk, nb, nb)
    C = _mm(eye - rho, F1) - _mm(F2, rho)
    return 0.5 * prefac * (C + C.mH)


def _mm(a, b):
    return (a[:, :, :, None] * b[:, None, :, :]).sum(2)


def _lin_rhs_S(P, k1, k2, rho, f, prefac):
    """The linearized right-hand side: the derivative of _rhs_S at diag f
    along rho - diag f (evolve_linear: no product with the imbalance itself)."""
    D = torch.diag_embed(f).to(rho.dtype)
    h = rho - D
    # _rhs_S is quadratic in the state: (f(D + h) - f(D - h)) / 2 is its linear part
    return 0.5 * (_rhs_S(P, k1, k2, D + h, prefac) - _rhs_S(P, k1, k2, D - h, prefac))


class _Plain:
    """The case's operator in torch: the right-hand side in the interaction
    picture with the band window and the coherent term."""

    def __init__(self, case, seed):
        self.case, self.d = case, _host_inputs(case, seed)
        self.k1, self.k2 = _pairs(case, seed)
        self.nk, self.nb, self.nbd, self.b0 = case["nk"], case["nb"], self.d["nbd"], self.d["b0"]
        self.prefac = 2 * math.pi / case["nk"]
        self.e = torch.from_numpy(self.d["edm"]).cuda()
        self.w = self.e[:, :, None] - self.e[:, None, :]
        self.H = torch.from_numpy(self.d["H"]).cuda().reshape(self.nk, self.nbd, self.nbd) if "H" in self.d else None
        self.f = torch.from_numpy(self.d["f"]).cuda()
        self.s = torch.from_numpy(self.d["s"]).cuda().reshape(self.nk, self.nbd, self.nbd)

    def load(self, seed, tag=100):
        return list(_p_chunks(self.case, seed, len(self.k1), tag))

    def rhs(self, P, t, y):
        ph = torch.exp(1j * self.w * t)
        r = y * ph.conj()
        a, b = self.b0, self.nbd
        if self.case.get("linear"):
            c = _lin_rhs_S(P, self.k1, self.k2, r[:, a:b, a:b], self.f[:, a:b], self.prefac)
        else:
            c = _rhs_S(P, self.k1, self.k2, r[:, a:b, a:b], self.prefac)
        c = c * ph[:, a:b, a:b]
        if a:
            full = torch.zeros_like(y)
            full[:, a:b, a:b] = c
            c = full
        if self.H is not None:
            Ht = self.H * ph
            c = c - 1j * (_mm(Ht, y) - _mm(y, Ht))
        return c

    def obs(self, t, y):
        d = y - torch.diag_embed(self.f).to(y.dtype)
        st = self.s * torch.exp(1j * self.w * t)
        a, b = self.b0, self.nbd
        return (st * d.transpose(1, 2))[:, a:b].real.sum() / self.nk

    def rk4(self, rhs, y, t0, steps, report):
        got = [self.obs(t0, y)] if report else []
        for j in range(steps):
            t = t0 + j * FS
            K1 = rhs(t, y)
            K2 = rhs(t + 0.5 * FS, y + 0.5 * FS * K1)
            K3 = rhs(t + 0.5 * FS, y + 0.5 * FS * K2)
            K4 = rhs(t + FS, y + FS * K3)
            y = y + FS / 6 * (K1 + 2 * K2 + 2 * K3 + K4)
            y = 0.5 * (y + y.mH)
            if report and (j + 1) % report == 0:
                got.append(self.obs(t + FS, y))
        return y, torch.stack(got) if got else torch.zeros(0, dtype=torch.float64)


def _fehlberg(rhs, y, t, h):
    """Fourth-order solution of one Fehlberg 4(5) step."""
    c = (0, 1 / 4, 3 / 8, 12 / 13, 1, 1 / 2)
    a = ((), (1 / 4,), (3 / 32, 9 / 32), (1932 / 2197, -7200 / 2197, 7296 / 2197),
         (439 / 216, -8, 3680 / 513, -845 / 4104), (-8 / 27, 2, -3544 / 2565, 1859 / 4104, -11 / 40))
    b = (25 / 216, 0, 1408 / 2565, 2197 / 4104, -1 / 5, 0)
    K = []
    for s in range(6):
        K.append(rhs(t + c[s] * h, y + h * sum((a[s][j] * K[j] for j in range(s)), torch.zeros_like(y))))
    return y + h * sum(b[j] * K[j] for j in range(6))


def _ee_P(case, d, k1, k2):
    """P_ee at the state for every stored pair (unexchanged, Lindblad form)."""
    nk, m = case["nk"], case["mesh"]
    V = abs(np.linalg.det(EE_R))
    qscr2 = 4 * math.pi * d["f"].sum() / (nk * V) / (EE_EPS * T300)
    Ri = np.linalg.inv(EE_R)
    GGT = torch.from_numpy(4 * math.pi ** 2 * Ri @ Ri.T).cuda()
    kv, e = torch.from_numpy(d["kvec"]).cuda(), torch.from_numpy(d["e"]).cuda()
    U = torch.from_numpy(d["U"]).cuda()
    cell = torch.round(kv * m).long()
    dm = torch.from_numpy(d["rho"]).cuda().reshape(nk, 2, 2)
    dm1 = torch.eye(2, device="cuda", dtype=dm.dtype) - dm
    pfac = 1 / (EE_DEGAUSS * math.sqrt(2 * math.pi)) / nk
    out1, out2 = [], []
    step = max(1, (1 << 20) // nk)
    for a0 in range(0, len(k1), step):
        A, B = k1[a0:a0 + step], k2[a0:a0 + step]
        dk = kv[A] - kv[B]
        dk = dk - torch.floor(0.5 + dk)
        q2 = ((dk[:, :, None] * GGT).sum(1) * dk).sum(1)
        v = 4 * math.pi / EE_EPS / V / (q2 + qscr2)
        v = torch.where(A == B, torch.zeros_like(v), v)
        o12 = (U[A].conj()[:, :, :, None] * U[B][:, :, None, :]).sum(1) * v[:, None, None]  # [n, p, q]
        c4 = (cell[A][:, None, :] + cell[None] - cell[B][:, None, :]) % m
        k4 = (c4[..., 0] * m + c4[..., 1]) * m + c4[..., 2]  # [n, k3]
        o34 = (U.conj()[None, :, :, :, None] * U[k4][:, :, :, None, :]).sum(2)  # [n, k3, x, y]
        de = (e[A][:, :, None] - e[B][:, None, :])[:, None, :, :, None, None] + \
            (e[None, :, :, None] - e[k4][:, :, None, :])[:, :, None, None]
        G = torch.exp(-0.25 * (de / EE_DEGAUSS) ** 2) * (de.abs() < EE_ETHR)
        A2 = o12[:, None, :, :, None, None] * o34[:, :, None, None] * G  # [n, k3, p, q, x, y]
        n = len(A)

        def form(L, R):  # sum over k3, x, y of (L A(p q) R)_xy conj(A(r s)_xy): [n, p, q, r, s]
            res = torch.empty(n, 2, 2, 2, 2, dtype=A2.dtype, device="cuda")
            for p in range(2):
                for q in range(2):
                    t = (L[:, :, :, :, None] * A2[:, :, p, q][:, :, None]).sum(3)
                    t = (t[..., None] * R[:, :, None]).sum(3)
                    for r in range(2):
                        for s_ in range(2):
                            res[:, p, q, r, s_] = (t * A2[:, :, r, s_].conj()).sum((1, 2, 3))
            return res

        S1 = form(dm1[None], dm[k4])
        S2 = form(dm[None], dm1[k4])
        # P1[(i1 i2),(i3 i4)]: A(i1 i3), A(i2 i4); P2: A(i3 i1), A(i4 i2)
        out1.append(S1.permute(0, 1, 3, 2, 4).reshape(n, 16) * pfac)
        out2.append(S2.permute(0, 2, 4, 1, 3).reshape(n, 16) * pfac)
    return torch.cat(out1), torch.cat(out2)


def exact(case, seed):
    kind, nk, nb = case["kind"], case["nk"], case["nb"]
    X = _Plain(case, seed)
    t = 17 * FS
    n = X.nbd
    if kind == "adjoint":
        return _exact_adjoint(X, case, seed, t)
    P = X.load(seed)
    if kind == "batched":
        rho = torch.from_numpy(X.d["rho"]).cuda().reshape(-1, nk, nb, nb)
        return torch.stack([X.rhs(P, t, r).reshape(nk, nb * nb) for r in rho])
    rho = torch.from_numpy(X.d["rho"]).cuda().reshape(nk, n, n)
    if kind in ("eval", "driver"):
        return X.rhs(P, t, rho).reshape(nk, n * n)
    if kind == "rk4":
        y, obs = X.rk4(lambda u, z: X.rhs(P, u, z), rho, t, case["steps"], case["report"])
        return y.reshape(nk, n * n), obs
    if kind == "rkf45":
        y = _fehlberg(lambda u, z: X.rhs(P, u, z), rho, t, FS)
        return y.reshape(nk, n * n), float(X.obs(t + FS, y))
    P1, P2 = _ee_P(case, X.d, X.k1, X.k2)
    P = [(a, p + P1[a:a + len(p)], q + P2[a:a + len(p)]) for a, p, q in P]
    return X.rhs(P, t, rho).reshape(nk, nb * nb)


def _exact_adjoint(X, case, seed, t):
    from torch.utils.checkpoint import checkpoint

    nk, nb = case["nk"], case["nb"]
    comps = [X.load(seed, 100 + c) for c in range(case["comps"])]
    theta = torch.ones(len(comps), dtype=torch.float64, device="cuda", requires_grad=True)
    rho = torch.from_numpy(X.d["rho"]).cuda().reshape(nk, nb, nb).requires_grad_(True)

    def one(th, u, z):
        P = [(c[0][0], sum(th[i] * c[i][1] for i in range(len(c))), sum(th[i] * c[i][2] for i in range(len(c))))
             for c in zip(*comps)]
        return X.rhs(P, u, z)

    y, obs = X.rk4(lambda u, z: checkpoint(one, theta, u, z, use_reentrant=False), 0.5 * (rho + rho.mH), t,
                   case["steps"], 1)
    w = obs.detach() - torch.from_numpy(X.d["target"]).cuda()
    gth, gr = torch.autograd.grad((obs * w).sum(), [theta, rho])
    return (y.detach().reshape(nk, nb * nb), obs.detach(), gth, (0.5 * (gr + gr.mH)).reshape(nk, nb * nb))
