"""Workloads of the per-(E,k) Green's-function engine, one case per kind of call.

Each case is one call of a public entry point of ``libnegf_amd.hip`` on a
block-tridiagonal device with semi-infinite contacts: coherent transmission
(two contacts, several contacts, several k-points, mixed precision), the local
density of states beside it, the density-matrix integrands on the complex
contour and on the real axis, the elastic-dephasing SCBA and the inelastic
polar-optical SCBA.  Sizes are those of ``libnegf_amd.workloads`` and of the
tests, or generic ones beside them (orders that fit no tile, few energies).

Two families of devices stand for what users bring: ``ribbon`` -- disordered
nearest-neighbour ribbons (orthogonal basis, sparse blocks, as workloads.C1,
C2, C4 and CI) -- and ``slab`` -- dense Bloch blocks with an overlap matrix
(as workloads.KSlab).

``exact`` restates the algorithms on torch complex128 batches: Sancho-Rubio
surface functions, the block recursions and, for the inelastic loop, whole
dense inverses.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from libnegf_amd import hip
from libnegf_amd.structure import BlockStructure, Contact
from libnegf_amd.workloads import CI, KB_EV, energy_grid

_CASES = [
    # One short energy sweep over a thin chain: the smallest call, a few ms of
    # device time at most (workloads.C1 with weak disorder).
    dict(name="chain_sweep", kind="T", model="ribbon", n=10, nbl=20, nE=200, nk=1, delta=1e-5,
         mirror=True, lanes=1, mixed=False),
    # A handful of energies at a time, as an adaptive energy grid or a bias
    # loop asks for them: launches and latency.
    dict(name="few_points", kind="T", model="slab", n=40, nbl=12, nE=5, nk=1, delta=1e-4,
         mirror=False, lanes=1, mixed=False),
    # Full transmission curve of a disordered ribbon (workloads.C2 at the
    # wrappers' default eta: at 1e-6 two FP64 evaluations differ by 1e-3 of T at
    # the resonances).
    dict(name="ribbon_sweep", kind="T", model="ribbon", n=64, nbl=100, nE=2000, nk=1, delta=1e-4,
         mirror=True, lanes=1, mixed=False),
    # One transverse k-point of a slab with overlap (workloads.C3's sizes), the
    # item groups left to the library.
    dict(name="slab_sweep", kind="T", model="slab", n=256, nbl=40, nE=500, nk=1, delta=1e-4,
         mirror=True, lanes=0, mixed=False),
    # k-resolved transmission between two different leads, orders that fit no
    # tile, every (E,k) of three slots in one call.
    dict(name="slab_kpoints", kind="T", model="slab", n=150, nbl=9, nE=33, nk=3, delta=1e-5,
         mirror=False, lanes=1, mixed=False),
    # The mixed-precision mode the serving loop uses (FP32 block inverses, two
    # FP64 Newton-Schulz steps).
    dict(name="slab_mixed", kind="T", model="slab", n=128, nbl=30, nE=200, nk=1, delta=1e-4,
         mirror=True, lanes=1, mixed=True),
    # Three-terminal device, all pairs.
    dict(name="three_terminal", kind="multi", model="slab", n=48, nbl=10, nE=101, delta=1e-4),
    # Transmission and layer-resolved local density of states.
    dict(name="slab_ldos", kind="ldos", model="slab", n=200, nbl=16, nE=128, delta=1e-5, dos_delta=1e-4,
         lanes=0),
    # Equilibrium density matrix: G^r on the complex contour.
    dict(name="dm_contour", kind="dm0", model="slab", n=128, nbl=20, npts=120),
    # Non-equilibrium part of the density matrix: G^n on the real axis under bias.
    dict(name="dm_bias", kind="dm1", model="slab", n=72, nbl=10, npts=101, delta=1e-4),
    # Elastic-dephasing SCBA with Meir-Wingreen currents (workloads.C4, a
    # quarter of its energies).
    dict(name="dephasing_scba", kind="scba", n=128, nbl=30, nE=250, delta=1e-5, coupling=0.1, tol=1e-8,
         lanes=0),
    # Inelastic polar-optical SCBA over an (E,k) grid (workloads.CI, half its
    # layers, fewer energies, a fixed number of outer passes).
    dict(name="optical_phonons", kind="inel", n=64, nbl=10, nE=160, nk=2, delta=1e-5, passes=10, lanes=0),
]


def listed():
    return [dict(c) for c in _CASES]


def _logint(rng, a, b):
    return int(round(math.exp(rng.uniform(math.log(a), math.log(b)))))


def draw(rng):
    """One more case of the listed kinds; sizes log-uniform over the ranges
    the listed cases span, redrawn while it would cost more than the largest."""
    top = max(work(c)["flops"] for c in _CASES)
    while True:
        kind = rng.choice(["T", "T", "T", "multi", "ldos", "dm0", "dm1", "scba", "inel"])
        delta = rng.choice([1e-4, 1e-5])
        if kind == "T":
            model = rng.choice(["ribbon", "slab"])
            mixed = model == "slab" and rng.random() < 0.2
            c = dict(kind="T", model=model, n=_logint(rng, 10, 256), nbl=_logint(rng, 8, 100),
                     nE=_logint(rng, 5, 2000), nk=rng.choice([1, 1, 2, 3]) if model == "slab" else 1,
                     delta=1e-4 if mixed or model == "ribbon" else delta, mirror=rng.random() < 0.6, lanes=rng.choice([0, 1]),
                     mixed=mixed)
        elif kind == "multi":
            c = dict(kind="multi", model="slab", n=_logint(rng, 10, 128), nbl=_logint(rng, 5, 24),
                     nE=_logint(rng, 5, 200), delta=delta)
        elif kind == "ldos":
            c = dict(kind="ldos", model="slab", n=_logint(rng, 10, 256), nbl=_logint(rng, 5, 40),
                     nE=_logint(rng, 5, 300), delta=delta, dos_delta=1e-4, lanes=rng.choice([0, 1]))
        elif kind == "dm0":
            c = dict(kind="dm0", model="slab", n=_logint(rng, 10, 256), nbl=_logint(rng, 5, 40),
                     npts=_logint(rng, 20, 200))
        elif kind == "dm1":
            c = dict(kind="dm1", model="slab", n=_logint(rng, 10, 128), nbl=_logint(rng, 4, 20),
                     npts=_logint(rng, 11, 201), delta=1e-4)
        elif kind == "scba":
            c = dict(kind="scba", n=_logint(rng, 16, 128), nbl=_logint(rng, 6, 30), nE=_logint(rng, 20, 250),
                     delta=1e-5, coupling=0.1, tol=1e-8, lanes=rng.choice([0, 1]))
        else:
            c = dict(kind="inel", n=_logint(rng, 16, 64), nbl=_logint(rng, 4, 10), nE=_logint(rng, 40, 160),
                     nk=rng.choice([2, 3]), delta=1e-5, passes=rng.choice([5, 8, 10]),
                     lanes=rng.choice([0, 1]))
        items = c.get("nE", c.get("npts", 1)) * c.get("nk", 1)
        blocks = 16.0 * c["n"] ** 2 * c["nbl"] * items
        if work(c)["flops"] <= top and blocks <= 2e10:
            return c


# ---- devices -----------------------------------------------------------------

def _rng(seed, salt):
    return np.random.Generator(np.random.PCG64([int(seed) & 0x7FFFFFFF, salt]))


def _ribbon(n, nbl, disorder, seed, shift=0.0, weak_lead=False):
    """Square-lattice ribbon of n sites across, seeded on-site disorder in the
    device; the second lead is the first one's mirror image unless weak_lead
    (hopping 0.9)."""
    rng = _rng(seed, 1)
    pl = -(np.eye(n, k=1) + np.eye(n, k=-1)) + shift * np.eye(n)
    t = -np.eye(n)
    hd = [pl + np.diag(rng.uniform(-disorder, disorder, n)) for _ in range(nbl)]
    t2 = 0.9 * t if weak_lead else t
    return BlockStructure(Hd=hd, Hu=[t] * (nbl - 1), Hl=[t.T] * (nbl - 1),
                          contacts=[Contact(cblk=nbl, H00=pl, H01=t, HMC=t),
                                    Contact(cblk=1, H00=pl, H01=t2.T, HMC=t.T)])


def _sym(rng, n, sigma):
    a = rng.normal(0.0, sigma, (n, n))
    return (a + a.T) / math.sqrt(2.0)


def _slab(n, nbl, seed, nk=1, mirror=True, side=False):
    """Dense slab with overlap at nk transverse k-points (workloads.KSlab's
    construction; the overlap's scale from the norm of a Gaussian matrix).
    side: a third contact on a middle layer."""
    rng = _rng(seed, 2)
    sc = 0.5 / (14.0 * math.sqrt(n))

    def onsite():
        return _sym(rng, n, 0.3), sc * _sym(rng, n, 1.0)

    def hop():
        return rng.normal(0.0, 0.1, (n, n)), sc * rng.normal(0.0, 1.0, (n, n))

    on = [onsite() for _ in range(nbl)]
    off = [hop() for _ in range(nbl - 1)]
    bx, by = hop(), hop()
    lead, leadhop = onsite(), hop()
    lead2, leadhop2 = (lead, leadhop) if mirror else (onsite(), hop())
    lead3, leadhop3 = (onsite(), hop()) if side else (None, None)
    ks = rng.uniform(-math.pi, math.pi, (nk, 2))
    out = []
    for kx, ky in ks:
        def bloch(a, j, eye):
            b = (a + bx[j] * np.exp(1j * kx) + bx[j].T * np.exp(-1j * kx)
                 + by[j] * np.exp(1j * ky) + by[j].T * np.exp(-1j * ky))
            return b + np.eye(n) if eye else b

        def contact(cblk, l, h, conj):
            a, s = (h[0].T, h[1].T) if conj else h
            return Contact(cblk=cblk, H00=bloch(l[0], 0, False), H01=a, HMC=a, S00=bloch(l[1], 1, True),
                           S01=s, SMC=s)

        cs = [contact(nbl, lead, leadhop, False), contact(1, lead2, leadhop2, True)]
        if side:
            cs.append(contact((nbl + 1) // 2, lead3, leadhop3, False))
        out.append(BlockStructure(Hd=[bloch(a, 0, False) for a, _ in on], Hu=[a for a, _ in off],
                                  Hl=[a.T for a, _ in off], contacts=cs,
                                  Sd=[bloch(s, 1, True) for _, s in on], Su=[s for _, s in off],
                                  Sl=[s.T for _, s in off]))
    return out


# Centre of the bias window of the SCBA cases: off the band centre, where the
# layers of a clean lead of odd width have a zero eigenvalue and E = 0 on the
# grid makes every evaluation ill-conditioned.
_MU0 = 0.0137


def _fermi(E, mu, kT):
    return 1.0 / (1.0 + np.exp(np.clip((E - mu) / kT, -500.0, 500.0)))


def _inputs(case, seed):
    """Structures (one per slot) and the call's host arrays."""
    k = case["kind"]
    n, nbl = case["n"], case["nbl"]
    r = _rng(seed, 3)
    x = {}
    if k == "T" and case["model"] == "ribbon":
        s = [_ribbon(n, nbl, 0.5 if n >= 32 else 0.1, seed, weak_lead=not case["mirror"])]
        E = energy_grid(case["nE"], -3.5, 3.47)  # off E = 0: see _MU0
    elif k in ("T", "multi", "ldos"):
        s = _slab(n, nbl, seed, case.get("nk", 1), case.get("mirror", True), side=(k == "multi"))
        E = energy_grid(case["nE"], -2.0, 2.0)
    if k in ("T", "multi", "ldos"):
        nk = len(s)
        x["E"] = np.tile(E, nk)
        x["slot"] = np.repeat(np.arange(nk, dtype=np.int32), len(E))
        if k == "ldos":
            x["proj"] = [list(range(i * n + 1, (i + 1) * n + 1)) for i in range(nbl)]
        return s, x
    if k in ("dm0", "dm1"):
        s = _slab(n, nbl, seed)
        m = case["npts"]
        t, w = np.polynomial.legendre.leggauss(m)
        if k == "dm0":  # upper half circle from below the spectrum to mu
            lo, mu = -6.0, 0.1 * r.uniform(-1.0, 1.0)
            c, R = 0.5 * (lo + mu), 0.5 * (mu - lo)
            th = 0.5 * math.pi * (1.0 - t)
            x["z"] = c + R * np.exp(1j * th) + 1e-3j
            x["w"] = -2.0 / math.pi * (-0.5 * math.pi * w) * (1j * R * np.exp(1j * th))
        else:
            kT, bias = KB_EV * 300.0, 0.2
            E = 0.5 * (bias + 20 * kT) * t
            x["z"] = E + 0j
            x["w"] = 0.5 * (bias + 20 * kT) * w / math.pi + 0j
            x["frm"] = np.stack([_fermi(E, bias / 2, kT), _fermi(E, -bias / 2, kT), np.zeros(m)], axis=1)
        return s, x
    kT, bias = KB_EV * 300.0, 0.2
    E = energy_grid(case["nE"], _MU0 - bias / 2 - 10 * kT, _MU0 + bias / 2 + 10 * kT)
    x["E"] = E
    x["frm"] = np.stack([_fermi(E, _MU0 + bias / 2, kT), _fermi(E, _MU0 - bias / 2, kT), np.zeros_like(E)], axis=1)
    if k == "scba":
        s = [_ribbon(n, nbl, 0.2, seed)]
        x["coupling"] = np.full(n * nbl, case["coupling"])
        return s, x
    nk = case["nk"]
    ky = (np.arange(nk) + 0.5) / (2 * nk)
    s = [_ribbon(n, nbl, CI["disorder"], seed, shift=2.0 * CI["ty"] * math.cos(2 * math.pi * y)) for y in ky]
    x["kw"] = np.full(nk, 1.0 / nk)
    kfrac = np.stack([np.zeros(nk), ky, np.zeros(nk)], axis=1)
    x["K"] = hip.inel_kmat_po(nbl, 1.0, kfrac, x["kw"], CI["coupling"], CI["wq"], CI["area"], CI["eps0"],
                              CI["eps_inf"], CI["q0"], latt=np.eye(3))
    x["iz"] = np.repeat(np.arange(nbl, dtype=np.int32), n)
    x["shift"] = int(round(CI["wq"] / (E[1] - E[0])))
    x["Nq"] = 1.0 / (math.exp(CI["wq"] / (KB_EV * CI["Tph"])) - 1.0)
    return s, x


def prepare(case, seed):
    """The engine, the device copy of the structure and the call's arrays."""
    s, x = _inputs(case, seed)
    return dict(case=case, x=x, eng=hip.Engine(0), ds=hip.DeviceStructure(s))


def run(state):
    """One call of the case's entry point."""
    c, x, eng, ds = state["case"], state["x"], state["eng"], state["ds"]
    k = c["kind"]
    if k == "T":
        return hip.solve_transmission(eng, ds, x["E"], slot=x["slot"], delta=c["delta"], lanes=c["lanes"],
                                      precision=hip.MIXED if c["mixed"] else hip.FP64,
                                      ns_steps=2 if c["mixed"] else 0)
    if k == "multi":
        return hip.solve_transmission_pairs(eng, ds, x["E"], [(1, 2), (1, 3), (2, 3)], slot=x["slot"],
                                            delta=c["delta"])
    if k == "ldos":
        return hip.solve_transmission_dos(eng, ds, x["E"], proj=x["proj"], dos_delta=c["dos_delta"],
                                          slot=x["slot"], delta=c["delta"], lanes=c["lanes"])
    if k == "dm0":
        return hip.density_accumulate(eng, ds, x["z"], x["w"], mode=0)
    if k == "dm1":
        return hip.density_accumulate(eng, ds, x["z"], x["w"], mode=1, frm=x["frm"], ref=2, delta=c["delta"])
    if k == "scba":
        r = hip.solve_scba_mw(eng, ds, x["E"], x["coupling"], 100, c["tol"], x["frm"], 3, delta=c["delta"],
                              want_diag=True, lanes=c["lanes"])
        return r["curr"], r["gn_diag"], r["gr_diag"], r["iters"], r["status"]
    r = hip.solve_inelastic_mw(eng, ds, x["E"], x["kw"], x["frm"], 3, x["K"], x["iz"], x["shift"], x["Nq"],
                               True, c["passes"] - 1, 0.0, delta=c["delta"], lanes=c["lanes"])
    return r["curr_mat"], r["currents"], r["passes"], r["status"], r["iters"]


# SCBA passes a dephasing solve at coupling 0.1 and tol 1e-8 takes.
_SCBA_PASSES = 9


def work(case):
    """Block products (8 m n k flops) and block inverses (8 n^3) of the
    recursions, with log2(1/eta) + 3 decimation iterations per contact (one
    recursion for a mirror-image pair); bytes are the structure and the outputs."""
    k, n, nbl = case["kind"], case["n"], case["nbl"]
    items = case.get("nE", case.get("npts", 1)) * case.get("nk", 1)
    nc = 3 if k == "multi" else 2
    nit = math.log2(1.0 / case.get("delta", 1e-3)) + 3.0
    dec = 56.0 * nit * (1 if case.get("mirror", k in ("scba", "inel", "ldos", "dm0", "dm1")) else nc) + 24.0 * nc
    per = {"T": 24 * nbl + 24, "multi": 24 * nbl + 32 * nbl + 3 * 16 * nbl / 2, "ldos": 56 * nbl + 24,
           "dm0": 64 * nbl + 64, "dm1": 64 * nbl + 80 * nbl + 80, "scba": _SCBA_PASSES * 112 * nbl,
           "inel": case.get("passes", 0) * 112 * nbl}[k]
    slab = case.get("model") == "slab"
    struct = 16.0 * n * n * (3 * nbl + 3 * nc) * (2 if slab else 1) * case.get("nk", 1)
    outs = {"T": 8.0 * items, "multi": 24.0 * items, "ldos": 8.0 * items * (nbl + 1),
            "dm0": 16.0 * n * n * (3 * nbl + 2), "dm1": 16.0 * n * n * (3 * nbl + 2),
            "scba": 32.0 * items * n * nbl, "inel": 16.0 * items}[k]
    return {"bytes": struct + outs, "flops": items * (dec + per) * float(n) ** 3}


def tolerance(case):
    """Relative bars from FP64 runs against ``exact`` over several seeds: the
    blocks E S - H - Sigma at real E have condition numbers up to 1/eta, so a
    few energies of each grid carry most of the difference and it varies by a
    factor of 30 from seed to seed (T: 4e-9 .. 2e-7; SCBA: 2e-8 .. 3e-6, its own
    stopping tolerance amplified; contour points are well conditioned).  ``differ``:
    decimation and SCBA counts whose test value falls on the threshold."""
    rel = {"T": 2e-6 if case["n"] >= 32 else 1e-7, "multi": 2e-7, "ldos": 2e-7, "dm0": 1e-12, "dm1": 2e-7,
           "scba": 2e-5, "inel": 5e-8}[case["kind"]]
    return {"rel": rel, "differ": 0.02}


# ---- the same quantities in torch complex128 ------------------------------------

def _dag(a):
    return a.conj().transpose(-1, -2)


class _Dev:
    """Blocks of the slots on the GPU, expanded per item on request."""

    def __init__(self, structs, slot):
            self.s, self.slot = structs, torch.as_tensor(np.asarray(slot), dtype=torch.int64).cuda()

    def stack(self, get):
        a = np.stack([np.ascontiguousarray(get(s)) for s in self.s])
        return torch.from_numpy(a).cuda()[self.slot]

    def esh(self, z, h, s, eye=False):
        H = self.stack(h)
        if s is not None and s(self.s[0]) is not None:
            S = self.stack(s)
        else:
            S = torch.eye(H.shape[1], dtype=H.dtype, device="cuda") if eye else 0.0
        return z[:, None, None] * S - H

    def diag(self, z, i):
        return self.esh(z, lambda s: s.Hd[i], (lambda s: s.Sd[i] if s.Sd else None), True)

    def up(self, z, i):
        return self.esh(z, lambda s: s.Hu[i], (lambda s: s.Su[i] if s.Su else None))

    def lo(self, z, i):
        return self.esh(z, lambda s: s.Hl[i], (lambda s: s.Sl[i] if s.Sl else None))


def _inv(a):
    # in parts: the batched LU's workspace grows with batch * order
    return torch.cat([torch.linalg.inv(p.contiguous()) for p in a.split(max(1, 8192 // a.shape[-1]))])


def _surface(dev, c, z):
    """(g_s, Tlc, Sigma) of contact c at the complex energies z."""
    ct = lambda s: s.contacts[c]
    Ao = dev.esh(z, lambda s: ct(s).H00, lambda s: ct(s).S00, True)
    Bo = dev.esh(z, lambda s: ct(s).H01, lambda s: ct(s).S01)
    Co = _dag(dev.esh(z.conj(), lambda s: ct(s).H01, lambda s: ct(s).S01))
    As, ok = Ao.clone(), 0
    for _ in range(200):
        g = _inv(Ao)
        gc, gb = g @ Co, g @ Bo
        c1, b1 = Co @ gc, Bo @ gb
        self_ = Bo @ gc
        As = As - self_
        Ao = Ao - self_ - Co @ gb
        ok = ok + 1 if float(c1.abs().max()) <= 1e-9 and float(b1.abs().max()) <= 1e-9 else 0
        Bo, Co = b1, c1
        if ok == 2:
            break
    gs = _inv(As)
    tl = dev.esh(z, lambda s: ct(s).HMC, lambda s: ct(s).SMC)
    tp = dev.esh(z.conj(), lambda s: ct(s).HMC, lambda s: ct(s).SMC)
    return gs, tl, tl @ gs @ _dag(tp)


def _gsmr(D, U, L):
    g = [None] * len(D)
    g[-1] = _inv(D[-1])
    for i in range(len(D) - 2, -1, -1):
        g[i] = _inv(D[i] - U[i] @ g[i + 1] @ L[i])
    return g


def _gr(D, U, L):
    """gsmr blocks and the tridiagonal G^r blocks."""
    g = _gsmr(D, U, L)
    Gd, Gu, Gl = [g[0]], [], []
    for i in range(1, len(D)):
        Gl.append(-g[i] @ L[i - 1] @ Gd[-1])
        ug = U[i - 1] @ g[i]
        Gu.append(-Gd[-1] @ ug)
        Gd.append(g[i] - Gl[-1] @ ug)
    return g, Gd, Gu, Gl


def _gn(g, Gd, Gu, U, L, S):
    """G^n blocks (diagonal, upper) for block-diagonal inflow S."""
    N = len(Gd)
    S = list(S)
    for i in range(N - 2, -1, -1):
        ug = U[i] @ g[i + 1]
        S[i] = S[i] + ug @ S[i + 1] @ _dag(ug)
    Nd, Nu = [Gd[0] @ S[0] @ _dag(Gd[0])], []
    for i in range(N - 1):
        lo = g[i + 1] @ (S[i + 1] @ _dag(Gu[i]) - L[i] @ Nd[i])
        Nu.append(_dag(lo))
        Nd.append(g[i + 1] @ (S[i + 1] @ _dag(Gd[i + 1]) - L[i] @ Nu[-1]))
    return Nd, Nu


def _tr(a, b):
    return (a * b.transpose(-1, -2)).sum((-1, -2)).real


def _gamma(s):
    return 1j * (s - _dag(s))


def _exact_T(case, s, x):
    nbl, k = case["nbl"], case["kind"]
    out_T, out_L = [], []
    chunk = max(1, int(3e9 / (16 * case["n"] ** 2 * (nbl + 24))))
    for a in range(0, len(x["E"]), chunk):
        E = torch.as_tensor(x["E"][a:a + chunk], dtype=torch.complex128).cuda()
        dev = _Dev(s, x["slot"][a:a + chunk])
        sig = [_surface(dev, c, E + 1j * case["delta"])[2] for c in range(s[0].ncont)]
        zd = E + 1j * case.get("dos_delta", 0.0)
        D = [dev.diag(zd, i) for i in range(nbl)]
        for c, ct in enumerate(s[0].contacts):
            D[ct.cblk - 1] = D[ct.cblk - 1] - sig[c]
        U = [dev.up(zd, i) for i in range(nbl - 1)]
        L = [dev.lo(zd, i) for i in range(nbl - 1)]
        gam = [_gamma(v) for v in sig]
        if k == "T":
            G = _gsmr(D, U, L)[0]
            out_T.append((_tr(gam[1], _gamma(G)) - _tr(gam[1] @ G @ gam[1], _dag(G))).abs())
            continue
        g, Gd, Gu, Gl = _gr(D, U, L)
        if k == "ldos":
            out_T.append((_tr(gam[1], _gamma(Gd[0])) - _tr(gam[1] @ Gd[0] @ gam[1], _dag(Gd[0]))).abs()[:, None])
            out_L.append(torch.stack([-torch.diagonal(v, dim1=-2, dim2=-1).imag.sum(-1) / math.pi for v in Gd], 1))
            continue
        cb = [ct.cblk for ct in s[0].contacts]
        ts = []
        for p, q in ((0, 1), (0, 2), (1, 2)):
            lo, hi = (p, q) if cb[p] < cb[q] else (q, p)
            cur = Gd[cb[lo] - 1]
            for i in range(cb[lo], cb[hi]):
                cur = -g[i] @ L[i - 1] @ cur
            ts.append(_tr(gam[hi] @ cur @ gam[lo], _dag(cur)).abs())
        out_T.append(torch.stack(ts, 1))
    cat = lambda v: torch.cat(v).cpu().numpy()
    if k == "ldos":
        return cat(out_T), cat(out_L), None, None
    return cat(out_T), None, None


def _exact_dm(case, s, x):
    nbl, gn = case["nbl"], case["kind"] == "dm1"
    acc = None
    chunk = max(1, int(3e9 / (16 * case["n"] ** 2 * (10 * nbl + 24))))
    for a in range(0, len(x["z"]), chunk):
        z = torch.as_tensor(x["z"][a:a + chunk], dtype=torch.complex128).cuda()
        w = torch.as_tensor(x["w"][a:a + chunk], dtype=torch.complex128).cuda()
        dev = _Dev(s, np.zeros(len(z), dtype=np.int64))
        zc = z + 1j * case["delta"] if gn else z
        con = [_surface(dev, c, zc) for c in range(2)]
        D = [dev.diag(z, i) for i in range(nbl)]
        U = [dev.up(z, i) for i in range(nbl - 1)]
        L = [dev.lo(z, i) for i in range(nbl - 1)]
        cb = [ct.cblk - 1 for ct in s[0].contacts]
        for c in range(2):
            D[cb[c]] = D[cb[c]] - con[c][2]
        g, Gd, Gu, Gl = _gr(D, U, L)
        if not gn:
            tc = [_dag(dev.esh(zc.conj(), lambda q: q.contacts[c].HMC, lambda q: q.contacts[c].SMC))
                  for c in range(2)]
            blocks = Gd + Gu + Gl + [-Gd[cb[c]] @ con[c][1] @ con[c][0] for c in range(2)] + \
                [-con[c][0] @ tc[c] @ Gd[cb[c]] for c in range(2)]
        else:
            f = torch.as_tensor(x["frm"][a:a + chunk]).cuda()
            S = [torch.zeros_like(v) for v in D]
            S[cb[0]] = S[cb[0]] + (f[:, 0] - f[:, 1])[:, None, None] * _gamma(con[0][2])  # contact 2 is the reference
            Nd, Nu = _gn(g, Gd, Gu, U, L, S)
            lc = []
            for c in range(2):
                gs, tl, _ = con[c]
                df = (f[:, 1] - f[:, c])[:, None, None]
                lc.append(-Nd[cb[c]] @ tl @ _dag(gs) + df * (Gd[cb[c]] @ tl @ _gamma(gs)))
            blocks = Nd + Nu + [_dag(v) for v in Nu] + lc + [_dag(v) for v in lc]
        part = torch.cat([(w[:, None, None] * b).sum(0).transpose(0, 1).reshape(-1) for b in blocks])
        acc = part if acc is None else acc + part
    return acc.cpu().numpy(), None


def _exact_scba(case, s, x):
    nbl, n = case["nbl"], case["n"]
    E = torch.as_tensor(x["E"], dtype=torch.complex128).cuda()
    f = torch.as_tensor(x["frm"]).cuda()
    B = len(E)
    dev = _Dev(s, np.zeros(B, dtype=np.int64))
    sig = [_surface(dev, c, E + 1j * case["delta"])[2] for c in range(2)]
    gam = [_gamma(v) for v in sig]
    cb = [ct.cblk - 1 for ct in s[0].contacts]
    c2 = case["coupling"] ** 2
    dr = torch.zeros(B, nbl, n, dtype=torch.complex128, device="cuda")
    dn = torch.zeros_like(dr)
    diag = lambda v: torch.diagonal(v, dim1=-2, dim2=-1)
    act = torch.arange(B, device="cuda")
    curr = torch.zeros(B, 2, dtype=torch.float64, device="cuda")
    for it in range(101):
        da = _Dev(s, np.zeros(len(act), dtype=np.int64))
        Ea = E[act]
        D = [da.diag(Ea, i) - torch.diag_embed(c2 * dr[act, i]) for i in range(nbl)]
        U = [da.up(Ea, i) for i in range(nbl - 1)]
        L = [da.lo(Ea, i) for i in range(nbl - 1)]
        S = [torch.diag_embed(c2 * dn[act, i]) for i in range(nbl)]
        for c in range(2):
            D[cb[c]] = D[cb[c]] - sig[c][act]
            S[cb[c]] = S[cb[c]] + f[act, c][:, None, None] * gam[c][act]  # no reference contact
        g, Gd, Gu, Gl = _gr(D, U, L)
        Nd, _ = _gn(g, Gd, Gu, U, L, S)
        new = torch.stack([diag(v) for v in Nd], 1)
        err = (new - dn[act]).abs().amax((1, 2))
        dr[act] = torch.stack([diag(v) for v in Gd], 1)
        dn[act] = new
        for c in range(2):
            tg = _tr(gam[c][act], Nd[cb[c]])
            ta = _tr(gam[c][act], _gamma(Gd[cb[c]]))
            curr[act, c] = -(tg - f[act, c] * ta)
        if it > 0:
            act = act[err >= case["tol"]]
        if len(act) == 0:
            break
    h = lambda v: v.reshape(B, -1).cpu().numpy()
    return curr.cpu().numpy(), h(dn), h(dr), None, None


def _exact_inel(case, s, x):
    nbl, n, ne, nk = case["nbl"], case["n"], case["nE"], case["nk"]
    N = nbl * n
    dt = torch.complex128
    E = torch.as_tensor(np.tile(x["E"], nk), dtype=dt).cuda()
    f = torch.as_tensor(np.tile(x["frm"], (nk, 1))).cuda()
    dev = _Dev(s, np.repeat(np.arange(nk), ne))
    sig = [_surface(dev, c, E + 1j * case["delta"])[2] for c in range(2)]
    gam = [_gamma(v) for v in sig]
    sl = [slice((ct.cblk - 1) * n, ct.cblk * n) for ct in s[0].contacts]
    A0 = dev.stack(lambda q: q.dense_device(0.0)) + E[:, None, None] * torch.eye(N, dtype=dt, device="cuda")
    S0 = torch.zeros_like(A0)
    for c in range(2):
        A0[:, sl[c], sl[c]] -= sig[c]
        S0[:, sl[c], sl[c]] += f[:, c][:, None, None] * gam[c]
    iz = torch.as_tensor(x["iz"].astype(np.int64)).cuda()
    dz = (iz[:, None] - iz[None, :]).abs()
    band = dz <= 1  # one z bin per layer: the tridiagonal blocks
    upper = iz[:, None] <= iz[None, :]
    K = torch.as_tensor(np.ascontiguousarray(x["K"])).cuda()
    sh, Nq = x["shift"], x["Nq"]
    Sr = Sn = None
    for _ in range(case["passes"]):
        cur = torch.zeros(nk * ne, 2, dtype=torch.float64, device="cuda")
        Gr, Gn = torch.empty_like(A0), torch.empty_like(A0)
        for a in range(0, nk * ne, 32):
            b = slice(a, min(a + 32, nk * ne))
            G = _inv(A0[b] - Sr[b] if Sr is not None else A0[b])
            Gr[b] = G
            Gn[b] = G @ (S0[b] + Sn[b] if Sn is not None else S0[b]) @ _dag(G)
            for c in range(2):
                A = _gamma(G[:, sl[c], sl[c]])
                cur[b, c] = -(_tr(gam[c][b], Gn[b][:, sl[c], sl[c]]) - f[b, c] * _tr(gam[c][b], A))
        Sr, Sn = torch.zeros_like(A0), torch.zeros_like(A0)
        v = lambda t, q: t[q * ne:(q + 1) * ne]
        for k in range(nk):
            for q in range(nk):
                Kq = K[:, k, q][dz] * band
                for dst, up, dn_ in ((v(Sn, k), v(Gn, q) * Nq, v(Gn, q) * (Nq + 1)),
                                     (v(Sr, k), v(Gr, q) * (Nq + 1) + 0.5j * v(Gn, q),
                                      v(Gr, q) * Nq - 0.5j * v(Gn, q))):
                    dst[sh:] += Kq * up[:ne - sh]
                    dst[:ne - sh] += Kq * dn_[sh:]
        Sn = Sn * upper
        off = iz[:, None] < iz[None, :]
        Sn = Sn + _dag(Sn * off)
    w = torch.as_tensor(np.repeat(x["kw"], ne)).cuda()
    cm = (cur * w[:, None]).reshape(nk, ne, 2).sum(0).cpu().numpy()
    de = x["E"][1] - x["E"][0]
    tw = np.full(ne, de)
    tw[0] = tw[-1] = 0.5 * de
    return cm, 2.0 * (tw[:, None] * cm).sum(0), None, None, None


def exact(case, seed):
    """What ``run`` returns, in torch complex128 (None for counts and status words)."""
    s, x = _inputs(case, seed)
    k = case["kind"]
    if k in ("T", "multi", "ldos"):
        return _exact_T(case, s, x)
    if k in ("dm0", "dm1"):
        return _exact_dm(case, s, x)
    return _exact_scba(case, s, x) if k == "scba" else _exact_inel(case, s, x)
