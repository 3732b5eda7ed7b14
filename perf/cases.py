"""Performance cases of the engine: the work a CHAMP-style program has it do,
through the public entry points of ``champ_amd.engine``.

A case is a dict of plain values.  ``op`` names the call sequence of one pass:

sweep   one VMC sweep of a population (``metrop1`` or CHAMP's default mover
        ``metrop6``): every electron of every walker moved, then the local
        energies; returns the walkers and their energies
hpsi    the local energies of a population at given positions and quadrature
drive   the calls of CHAMP's own metropolis loop, one electron at a time
        (drift, psie, drift at the proposal, accept), then hpsi
dmc     one DMC step with T-moves of the reference's butadiene case
batch   one sweep of eight molecules together (``metrop1_batch``)
deriv   the derivatives of ln psi and the sums of stochastic reconfiguration

Systems are the named ones of ``champ_amd.system.config``, the reference
inputs under ``tests/golden/champ_inputs``, or ("molecule") a chain of heavy
atoms and hydrogens from ``make_system`` with the c160 basis recipe.
"""
from __future__ import annotations

import functools
import math
import os

import numpy as np
import torch

from champ_amd import champ_io, optwf
from champ_amd import system as S
from champ_amd.engine import (DERIV_CI, DERIV_JAS_EE, DERIV_JAS_EEN, DERIV_JAS_EN, DERIV_ORB, PREC_FP64, PREC_MIXED,
                              Engine, metrop1_batch)

DEVICE = "cuda" if torch.cuda.is_available() else "cpu"
ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
INPUTS = {
    "C4H6_dmc": ("C4H6_dmc", "dmc.inp", None),
    "C4H6_500": ("C4H6_500", "vmc_optimization_500.inp", 280),
}


def listed():
    return [
        # the smallest call: one short test sweep of four walkers of a 10-electron
        # molecule, where launches and latency count
        dict(name="sweep_small_4w", op="sweep", system="small", walkers=4, mover=1, graphs=False),
        # an all-electron molecule of the size of butadiene with one walker per
        # CU, CHAMP's default mover, the sweep replayed as a captured graph
        dict(name="sweep_c22_256w_m6_graph", op="sweep", system="c22", walkers=256, mover=6, graphs=True),
        # an ordinary production run: 60 electrons, pseudopotential
        dict(name="sweep_c60_768w", op="sweep", system="c60", walkers=768, mover=1, graphs=False),
        # odd sizes: 97 electrons, unequal spins, a walker count that no tile divides,
        # order-5 electron-electron-nucleus terms, the default mover
        dict(name="sweep_ragged97_611w_m6", op="sweep", system="molecule", heavy=13, hydrogens=7, electrons=97,
             ecp=True, order=5, walkers=611, mover=6, graphs=False),
        # the largest: 160 electrons and 4096 walkers, the workload of bench.py
        dict(name="sweep_c160_4096w", op="sweep", system="c160", walkers=4096, mover=1, graphs=False),
        # a multideterminant trial function: 256 electrons, 5000 determinants
        dict(name="sweep_md256_384w", op="sweep", system="md256", walkers=384, mover=1, graphs=False),
        # local energies of the largest population on the mixed-precision path
        dict(name="hpsi_c160_4096w_mixed", op="hpsi", system="c160", walkers=4096, mixed=True),
        # local energies of an ordinary population (correlated sampling, restarts)
        dict(name="hpsi_c60_1000w", op="hpsi", system="c60", walkers=1000, mixed=False),
        # CHAMP's own driver calling the engine one electron at a time, mixed precision
        dict(name="drive_c160_1024w_mixed", op="drive", system="c160", walkers=1024, mixed=True),
        # a DMC step of the reference's 500-determinant butadiene input with T-moves
        dict(name="dmc_c4h6_1536w", op="dmc", walkers=1536),
        # eight molecules of 20 to 300 electrons swept together
        dict(name="batch_hetero_quarter", op="batch", scale=0.25),
        # an optimisation sample: 500 determinants with orbital terms
        dict(name="deriv_c4h6_500_2048w", op="deriv", system="C4H6_500", walkers=2048, orbital_terms=300),
    ]


def _logint(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["sweep", "sweep", "sweep", "sweep", "hpsi", "hpsi", "drive", "dmc", "deriv"])
    if op == "dmc":
        return dict(op="dmc", walkers=_logint(rng, 16, 1536))
    if op == "deriv":
        if rng.random() < 0.5:
            return dict(op="deriv", system="C4H6_500", walkers=_logint(rng, 32, 2048),
                        orbital_terms=_logint(rng, 1, 300))
        return dict(op="deriv", system="c22_md", walkers=_logint(rng, 32, 4096), orbital_terms=0)
    if rng.random() < 0.2:  # a multideterminant molecule
        case = dict(op=op, system=rng.choice(["small_md", "small_ae_md", "c22_md"]), walkers=_logint(rng, 3, 4096))
    else:
        heavy = _logint(rng, 2, 38)
        electrons = int(heavy * rng.uniform(4.0, 8.0)) + rng.randrange(2)
        hydrogens = rng.randrange(0, heavy + 1)
        # no dearer than the largest listed case: walkers x electrons^2 x centres
        most = 0.9 * 4096 * 160 * 160 * 40 / (electrons ** 2 * (heavy + hydrogens))
        case = dict(op=op, system="molecule", heavy=heavy, hydrogens=hydrogens, electrons=electrons,
                    ecp=rng.random() < 0.75, order=rng.choice([3, 4, 4, 4, 5]),
                    walkers=_logint(rng, 1, min(4096, int(most))))
    if op == "sweep":
        case.update(mover=rng.choice([1, 6]), graphs=rng.random() < 0.25)
    else:
        case.update(mixed=rng.random() < 0.5)
        if op == "drive":
            case.update(walkers=min(case["walkers"], 1024))
    return case


# --------------------------------------------------------------------------
@functools.lru_cache(maxsize=None)
def _system(name, heavy, hydrogens, electrons, ecp, order):
    if name == "molecule":
        return S.make_system("molecule", heavy, hydrogens, electrons, "sssspppdd", "ssp", nloc=4 if ecp else 0,
                             nordc=order)
    if name in INPUTS:
        d, inp, nadorb = INPUTS[name]
        return champ_io.load_input(os.path.join(ROOT, "tests", "golden", "champ_inputs", d, inp), name=name,
                                   **({} if nadorb is None else dict(nadorb=nadorb)))
    return S.config(name)


def system_of(case):
    return _system(case.get("system", "C4H6_dmc"), case.get("heavy"), case.get("hydrogens"), case.get("electrons"),
                   case.get("ecp"), case.get("order"))


@functools.lru_cache(maxsize=None)
def _orb_terms(n):
    sy = _system("C4H6_500", None, None, None, None, None)
    irrep = champ_io.read_symmetry(os.path.join(ROOT, "tests", "golden", "champ_inputs", "C4H6_500",
                                                "ci1010_pVTZ_1_symmetry.sym"), sy.coef.shape[0])
    return np.asarray(optwf.optorb_define(sy.iworbd, sy.nup, irrep, nadorb=280))[:n]


def _streams(nwalk, seed):
    return np.random.default_rng([seed, 1]).integers(1, 2 ** 63 - 1, size=(nwalk, 4), dtype=np.uint64)


def _rotations(nwalk, seed):
    """A random rotation per walker (unit quaternions)."""
    q = np.random.default_rng([seed, 2]).normal(size=(nwalk, 4))
    a, b, c, d = (q / np.linalg.norm(q, axis=1, keepdims=True)).T
    return np.stack([np.stack([1 - 2 * (c * c + d * d), 2 * (b * c - a * d), 2 * (b * d + a * c)], -1),
                     np.stack([2 * (b * c + a * d), 1 - 2 * (b * b + d * d), 2 * (c * d - a * b)], -1),
                     np.stack([2 * (b * d - a * c), 2 * (c * d + a * b), 1 - 2 * (b * b + c * c)], -1)], 1)


def _quadrature(sy, nwalk, seed):
    """Rotated quadrature points [nwalk][nquad][3]."""
    return np.einsum("wij,qj->wqi", _rotations(nwalk, seed), np.stack([sy.xq0, sy.yq0, sy.zq0], -1))


def _engine(sy, nwalk, seed, mixed=False):
    eng = Engine(sy, nwalk, precision=PREC_MIXED if mixed else PREC_FP64)
    eng.set_walkers(sy.initial_walkers(nwalk, seed=seed))
    eng.set_rng(_streams(nwalk, seed))
    return eng


def _drive_plan(sy, nwalk, seed):
    """Proposals of two sweeps (alternating passes) and the walkers that take
    them: steps of 0.3 bohr about the starting positions, 40% accepted."""
    rng = np.random.default_rng([seed, 3])
    x0 = sy.initial_walkers(nwalk, seed=seed)
    return x0, [(np.ascontiguousarray((x0 + 0.3 * rng.standard_normal(x0.shape)).transpose(1, 0, 2)),
                 rng.random((sy.nelec, nwalk)) < 0.4) for _ in range(2)]


def _kinds(case, sy):
    k = DERIV_JAS_EN | DERIV_JAS_EE | DERIV_CI
    if sy.nordc > 1:
        k |= DERIV_JAS_EEN
    if case["orbital_terms"]:
        k |= DERIV_ORB
    return k


def prepare(case, seed):
    op = case["op"]
    if op == "batch":
        engs = []
        for sy, w in _batch(case["scale"]):
            eng = _engine(sy, w, seed)
            eng.hpsi()
            engs.append(eng)
        return dict(op=op, engines=engs)
    sy, w = system_of(case), case["walkers"]
    if op == "dmc":
        eng = _engine(sy, 2 * w, seed)
        eng.hpsi()
        eng.metrop1(10, 0.2)
        eng.dmc_init(w, 0.05, -26.3, _streams(1, seed + 1)[0])
        eng.dmc_set_icasula(-1)
        return dict(op=op, engine=eng)
    eng = _engine(sy, w, seed, case.get("mixed", False))
    state = dict(op=op, engine=eng, mixed=case.get("mixed", False))
    if sy.nloc and op in ("hpsi", "drive"):
        q = _quadrature(sy, w, seed)
        eng.set_quadrature(q[..., 0], q[..., 1], q[..., 2])
    if op == "hpsi":
        return state
    eng.hpsi()
    if op == "sweep":
        eng.set_graphs(case["graphs"])
        state.update(mover=case["mover"])
    elif op == "drive":
        state.update(plan=_drive_plan(sy, w, seed)[1], passes=0)
    elif op == "deriv":
        if case["orbital_terms"]:
            eng.set_orb_terms(_orb_terms(case["orbital_terms"]))
        state.update(kinds=_kinds(case, sy))
    return state


@functools.lru_cache(maxsize=None)
def _batch(scale):
    return S.hetero_batch(scale=scale)


def _result(state, values):
    """What a mixed-precision program keeps of a result: that path forms the
    Jastrow and the moves' orbitals in FP32 and its results are FP32 numbers."""
    return {k: v.astype(np.float32) for k, v in values.items()} if state["mixed"] else values


def _log_psi(psid, psij):
    return np.log(np.abs(psid)) + psij


def run(state):
    op = state["op"]
    if op == "batch":
        stats = metrop1_batch(state["engines"], 1, 0.3)
        sc = [e.scalars() for e in state["engines"]]
        return dict(walkers=[e.get_walkers() for e in state["engines"]],
                    stats={k: np.array([st[k] for st in stats]) for k in stats[0]},
                    scalars={k: np.concatenate([v[k] for v in sc]) for k in sc[0]})
    eng = state["engine"]
    if op == "sweep":
        st = eng.metrop1(1, 0.3) if state["mover"] == 1 else eng.metrop6(1)
        return dict(st, walkers=eng.get_walkers(), **eng.scalars())
    if op == "hpsi":
        h = eng.hpsi()
        return _result(state, dict(logpsi=_log_psi(h["psid"], h["psij"]), psij=h["psij"], ekin=h["ekin"],
                                   energy=h["energy"]))
    if op == "drive":
        xnew, mask = state["plan"][state["passes"] % 2]
        state["passes"] += 1
        logpsi, drift = [], []
        for iel in range(eng.nelec):
            vold = eng.compute_determinante_grad(iel, 1)
            pd, pj = eng.psie(iel, xnew[iel])
            vnew = eng.compute_determinante_grad(iel, 0)
            eng.accept(iel, mask[iel])
            logpsi.append(_log_psi(pd, pj))
            drift.append(np.stack([vold, vnew]))
        h = eng.hpsi()
        return _result(state, dict(logpsi_moves=np.stack(logpsi), drift=np.stack(drift),
                                   logpsi=_log_psi(h["psid"], h["psij"]), ekin=h["ekin"], energy=h["energy"]))
    if op == "dmc":
        st = eng.dmc_step()
        wt, x, e = eng.dmc_population()
        return dict(st, weights=wt, walkers=x, energies=e)
    o = eng.deriv_psi(state["kinds"])
    s, osum, eosum, esum = eng.sr_sums(state["kinds"])
    return dict(o=o, s=s, osum=osum, eosum=eosum, esum=esum)


# --------------------------------------------------------------------------
def _sweep_work(sy, w, hpsi_only=False):
    """Floating operations of one sweep: per move the electron-electron-nucleus
    sums of one electron against its partners (value and both gradients, about
    26 multiply-adds per pair and centre), its orbitals and the update of the
    inverse; per hpsi all pairs, the orbitals and inverse of every electron and
    the quadrature (a quarter of the electrons within the range of a
    pseudopotential).  Bytes: the walkers in and out, their streams, psi and
    energies, and the orbital coefficients."""
    ne, nc, nb, no = sy.nelec, sy.ncent, sy.nbasis, sy.norb
    ns = (ne + 1) // 2
    een = 52.0 * nc if sy.nordc > 1 else 0.0
    move = (ne - 1) * (een + 60.0) + 8.0 * nb * no + 30.0 * nb + 1.6 * ns * ns
    h = 0.5 * ne * (ne - 1) * (2.0 * een + 120.0) + 10.0 * ne * nb * no + 4.0 * ns ** 3
    if sy.nloc:
        npt = 0.25 * ne * len(sy.wq)
        h += npt * ((ne - 1) * (een / 4 + 40.0) + 8.0 * nb) + 4.0 * ns * ns * nb
    flops = h if hpsi_only else ne * move + h
    return 8.0 * (w * (3 * ne * (1 if hpsi_only else 2) + 12) + no * nb), w * flops


def work(case):
    op = case["op"]
    if op == "batch":
        parts = [_sweep_work(sy, w) for sy, w in _batch(case["scale"])]
        return dict(bytes=sum(p[0] for p in parts), flops=sum(p[1] for p in parts))
    sy, w = system_of(case), case["walkers"]
    if op == "deriv":
        n = sy.nctype * (sy.norda + 1) + sy.nspin2b * (sy.nordb + 1) + sy.iworbd.shape[0] + case["orbital_terms"]
        if sy.nordc > 1:
            n += sy.nctype * sy.c.shape[1]
        pairs = 0.5 * sy.nelec * (sy.nelec - 1)
        return dict(bytes=8.0 * (n * w + n * n), flops=1.0 * n * n * w + w * pairs * (40.0 + 40.0 * sy.ncent) +
                    2.0 * w * n * sy.nelec)
    b, f = _sweep_work(sy, w, hpsi_only=op == "hpsi")
    return dict(bytes=b, flops=f)


# --------------------------------------------------------------------------
# The quantities in 64 bits by torch: single Slater determinants with their
# local energies, and the parameter derivatives of a determinant expansion.
def _t(a):
    return torch.as_tensor(np.ascontiguousarray(a), dtype=torch.float64, device=DEVICE)


class _Exact:
    def __init__(self, sy):
        self.sy = sy
        self.cent, self.coef = _t(sy.cent), _t(sy.coef)
        self.type = [int(t) for t in sy.iwctype]
        self.of_type = [torch.as_tensor([c for c, t in enumerate(self.type) if t == it], device=DEVICE)
                        for it in range(sy.nctype)]
        self.rwf, self.d2 = _t(sy.rwf), _t(sy.d2rwf)
        self.kap, self.ainf = sy.scalek, 1.0 / sy.scalek
        self.terms = S.een_terms(sy.nordc) if sy.nordc > 1 else []
        like = 0.5 if (sy.nspin2b == 1 and sy.nocuspb == 0) else 1.0
        spin = torch.as_tensor([0] * sy.nup + [1] * sy.ndn, device=DEVICE)
        self.like = (spin[:, None] == spin[None, :])
        self.scale = torch.where(self.like, like, 1.0).double()

    def radial(self, it, irb, r):
        """R, R', R'' of a shell on the shifted exponential grid."""
        sy = self.sy
        xr = torch.log((r + sy.grid_r0) / sy.grid_r0) / math.log(sy.grid_arg) + 1.0
        j = xr.long().clamp(1, sy.nr - 1)
        lo = sy.grid_r0 * torch.pow(torch.tensor(sy.grid_arg, dtype=torch.float64, device=DEVICE), (j - 1).double()) - sy.grid_r0
        hi = (lo + sy.grid_r0) * sy.grid_arg - sy.grid_r0
        h = hi - lo
        y, d = self.rwf[it, irb], self.d2[it, irb]
        y0, y1, s0, s1 = y[j - 1], y[j], d[j - 1], d[j]
        b, a = (r - lo) / h, (hi - r) / h
        f = a * y0 + b * y1 + (a * (a * a - 1) * s0 + b * (b * b - 1) * s1) * h * h / 6
        f1 = (y1 - y0) / h + ((3 * b * b - 1) * s1 - (3 * a * a - 1) * s0) * h / 6
        f2 = a * s0 + b * s1
        tail = xr >= sy.nr
        ae = sy.ae[it, irb]
        t = ae[0] * torch.exp(-ae[1] * r)
        f, f1, f2 = (torch.where(tail, v, u) for u, v in ((f, t), (f1, -ae[1] * t), (f2, ae[1] ** 2 * t)))
        off = r > sy.rmaxwf[it, irb]
        return tuple(torch.where(off, 0.0, v) for v in (f, f1, f2))

    MONOMIALS = ["", "x", "y", "z", "xx", "xy", "xz", "yy", "yz", "zz", "xxx", "xxy", "xxz", "yyx", "xyz", "zzx",
                 "yyy", "yyz", "zzy", "zzz"]
    CS, CP, CD1, CD2 = 0.28209479177387814, 0.48860251190291992, 0.630783130505040, 1.092548430592079
    CF, CF2, CF3 = 0.74635266518023078, 1.66889529453113635, 2.89061144264055405
    NORMS = [CS] + [CP] * 3 + [CD1, CD2, CD2, CD1, CD2, CD1] + [CF, CF2, CF2, CF2, CF3, CF2, CF, CF2, CF2, CF]

    def shells(self, p, derivs):
        """For each AO of each centre type: its columns and its values
        [n][centres of the type] at points p [n][3], with derivs also gradients
        [n][centres][3] and Laplacians."""
        sy = self.sy
        first = np.concatenate([[0], np.cumsum([int(sy.nbastyp[t]) for t in self.type])])
        for it, idx in enumerate(self.of_type):
            if not len(idx):
                continue
            off = torch.as_tensor(first[idx.cpu().numpy()], device=DEVICE)
            v = p[:, None] - self.cent[idx]
            r = v.norm(dim=-1)
            pw = [[torch.ones_like(r), v[..., k], v[..., k] ** 2, v[..., k] ** 3] for k in range(3)]
            rad = {}
            for m in range(int(sy.nbastyp[it])):
                irb, code = int(sy.iwrwf[it, m]), int(sy.iwlbas[it, m]) - 1
                if irb not in rad:
                    rad = {irb: self.radial(it, irb, r)}
                f, f1, f2 = rad[irb]
                e, nc = [self.MONOMIALS[code].count(ch) for ch in "xyz"], self.NORMS[code]
                y = nc * pw[0][e[0]] * pw[1][e[1]] * pw[2][e[2]]
                if not derivs:
                    yield off + m, y * f
                    continue
                dy, ly = [], 0.0
                for k in range(3):
                    a, b = (k + 1) % 3, (k + 2) % 3
                    rest = nc * pw[a][e[a]] * pw[b][e[b]]
                    dy.append(e[k] * pw[k][e[k] - 1] * rest if e[k] else torch.zeros_like(r))
                    if e[k] > 1:
                        ly = ly + e[k] * (e[k] - 1) * pw[k][e[k] - 2] * rest
                u = [v[..., k] / r for k in range(3)]
                yield (off + m, y * f, torch.stack([y * u[k] * f1 + dy[k] * f for k in range(3)], -1),
                       y * f2 + 2 * y * f1 / r + ly * f + 2 * sum(dy[k] * u[k] for k in range(3)) * f1)

    def ao(self, p, derivs):
        """AO values [n][nb], with derivs also gradients and Laplacians [5][n][nb]"""
        out = torch.zeros(5 if derivs else 1, len(p), self.sy.nbasis, dtype=torch.float64, device=DEVICE)
        for got in self.shells(p, derivs):
            out[0][:, got[0]] = got[1]
            if derivs:
                for k in range(3):
                    out[1 + k][:, got[0]] = got[2][..., k]
                out[4][:, got[0]] = got[3]
        return out if derivs else out[0]

    # ------------------------------------------------------------- Jastrow
    def pade(self, p, scale, r):
        """value minus asymptote, first and second derivative of the Pade and
        polynomial form in the scaled distance r"""
        def val(s):
            return scale * p[0] * s / (1 + p[1] * s) + sum(p[o] * s ** o for o in range(2, len(p)))
        bot = 1 + p[1] * r
        d1 = scale * p[0] / bot ** 2 + sum(o * p[o] * r ** (o - 1) for o in range(2, len(p)))
        d2 = -2 * scale * p[0] * p[1] / bot ** 3 + sum(o * (o - 1) * p[o] * r ** (o - 2) for o in range(2, len(p)))
        return val(r) - val(torch.full((), self.ainf, dtype=torch.float64, device=DEVICE)), d1, d2

    def scaled(self, r):
        return (1 - torch.exp(-self.kap * r)) / self.kap

    def jastrow(self, x):
        """ln J, gradients [w][ne][3] and the sum of Laplacians; x [w][ne][3]."""
        sy, kap = self.sy, self.kap
        w, ne = x.shape[:2]
        eye = torch.eye(ne, dtype=torch.bool, device=DEVICE)
        rv = x[:, :, None] - x[:, None]
        r = torch.where(eye, 1.0, rv.norm(dim=-1))
        u = torch.exp(-kap * r)  # the switched distance 1 - kap R
        lnj = torch.zeros(w, dtype=torch.float64, device=DEVICE)
        grad, lap = torch.zeros_like(x), torch.zeros_like(lnj)

        def radial_pair(f, f1, f2):  # a function of R(r_ij): f, df/dR, d2f/dR2
            nonlocal lnj, grad, lap
            d1, d2 = f1 * u, f2 * u * u - kap * f1 * u
            f, d1, d2 = (torch.where(eye, 0.0, v) for v in (f, d1, d2))
            lnj = lnj + 0.5 * f.sum((1, 2))
            grad = grad + ((d1 / r)[..., None] * rv).sum(2)
            lap = lap + (d2 + 2 * d1 / r).sum((1, 2))

        R = self.scaled(r)
        if sy.nspin2b == 1:
            radial_pair(*self.pade(sy.b[0], self.scale, R))
        else:
            a, b = self.pade(sy.b[0], 1.0, R), self.pade(sy.b[1], 1.0, R)
            radial_pair(*(torch.where(self.like, q, p) for p, q in zip(a, b)))
        ev = x[:, :, None] - self.cent[None, None]
        er = ev.norm(dim=-1)
        X = torch.exp(-kap * er)
        for it, idx in enumerate(self.of_type):
            f, f1, f2 = self.pade(sy.a4[it], 1.0, self.scaled(er[..., idx]))
            d1 = f1 * X[..., idx]
            d2 = f2 * X[..., idx] ** 2 - kap * f1 * X[..., idx]
            lnj = lnj + f.sum((1, 2))
            grad = grad + ((d1 / er[..., idx])[..., None] * ev[..., idx, :]).sum(2)
            lap = lap + (d2 + 2 * d1 / er[..., idx]).sum((1, 2))
        # e-e-n: sum_k u^k M_k(i, j) with M_k bilinear in powers of the switched
        # electron-centre distances
        n = sy.nordc
        if self.terms:
            unit = rv / r[..., None]
            for k in range(0, n + 1):
                pairs = [(c, l, m) for c, (kk, l, m) in enumerate(self.terms) if kk == k]
                if not pairs:
                    continue
                M = torch.zeros(w, ne, ne, dtype=torch.float64, device=DEVICE)
                G = torch.zeros(w, ne, ne, 3, dtype=torch.float64, device=DEVICE)
                L = torch.zeros_like(M)
                for it, idx in enumerate(self.of_type):
                    Xi, evi, eri = X[..., idx], ev[..., idx, :], er[..., idx]
                    pw = [Xi ** p for p in range(n + 1)]
                    # gradient and Laplacian of x^p = exp(-p kap r)
                    gp = [(-p * kap * pw[p] / eri)[..., None] * evi for p in range(n + 1)]
                    lp = [p * kap * pw[p] * (p * kap - 2 / eri) for p in range(n + 1)]
                    for c, l, m in pairs:
                        cf = float(sy.c[it, c])
                        for p, q in ((l + m, m), (m, l + m)):
                            right = pw[q].transpose(1, 2).contiguous()
                            M = M + cf * (pw[p] @ right)
                            L = L + cf * (lp[p] @ right)
                            G = G + cf * torch.stack([gp[p][..., d].contiguous() @ right for d in range(3)], -1)
                uk = u ** k
                fr = torch.where(eye, 0.0, uk)
                lnj = lnj + 0.5 * (fr * M).sum((1, 2))
                du = torch.where(eye, 0.0, -k * kap * uk)  # d u^k / d r
                d2u = torch.where(eye, 0.0, k * kap * uk * (k * kap - 2 / r))  # Laplacian of u^k
                grad = grad + ((du * M)[..., None] * unit + fr[..., None] * G).sum(2)
                lap = lap + (d2u * M + 2 * du * (unit * G).sum(-1) + fr * L).sum((1, 2))
        return lnj, grad, lap

    def jastrow_at(self, x, xq, e):
        """sum of the terms of ln J that hold electron e [w][p] moved to xq
        [w][p][3] in the configurations x [w][ne][3]."""
        sy, kap = self.sy, self.kap
        keep = torch.arange(sy.nelec, device=DEVICE) != e[..., None]
        r = (xq[:, :, None] - x[:, None]).norm(dim=-1)
        u = torch.exp(-kap * r)
        R = self.scaled(r)
        if sy.nspin2b == 1:
            f = self.pade(sy.b[0], self.scale[e], R)[0]
        else:
            f = torch.where(self.like[e], self.pade(sy.b[1], 1.0, R)[0], self.pade(sy.b[0], 1.0, R)[0])
        eq, ej = (xq[:, :, None] - self.cent).norm(dim=-1), (x[:, :, None] - self.cent).norm(dim=-1)
        s = torch.zeros_like(eq[..., 0])
        for it, idx in enumerate(self.of_type):
            s = s + self.pade(sy.a4[it], 1.0, self.scaled(eq[..., idx]))[0].sum(-1)
        Xq, Xj = torch.exp(-kap * eq), torch.exp(-kap * ej)
        for k in sorted({t[0] for t in self.terms}):
            M = torch.zeros_like(r)
            for it, idx in enumerate(self.of_type):
                a, b = Xq[..., idx], Xj[..., idx].transpose(1, 2).contiguous()
                for c, (kk, l, m) in enumerate(self.terms):
                    if kk == k:
                        M = M + float(sy.c[it, c]) * (a ** (l + m) @ b ** m + a ** m @ b ** (l + m))
            f = f + u ** k * M
        return s + torch.where(keep, f, 0.0).sum(-1)

    # --------------------------------------------------------- local energy
    def ecp(self, it, l, r):
        sy, v = self.sy, 0.0
        for g in range(int(sy.necp_term[it, l])):
            ex = sy.ecp_exponent[it, l, g] * r * r
            v = v + r ** (int(sy.necp_power[it, l, g]) - 2) * torch.where(ex > 700, 0.0, sy.ecp_coef[it, l, g] * torch.exp(-ex))
        return v

    def hpsi(self, x, quad):
        """ln|psi|, ln J, kinetic and local energy of one determinant; x
        [w][ne][3], quad [w][nq][3]."""
        sy = self.sy
        w, ne = x.shape[:2]
        ao = self.ao(x.reshape(-1, 3), True)
        orb = [(ao[k] @ self.coef.T).reshape(w, ne, -1) for k in range(5)]
        phi, dphi, lphi = orb[0], torch.stack(orb[1:4], -1), orb[4]
        lnj, gj, lapj = self.jastrow(x)
        logpsi, drift, ld = lnj.clone(), torch.zeros_like(x), torch.zeros(w, ne, dtype=torch.float64, device=DEVICE)
        rows = torch.zeros(w, ne, self.coef.shape[1], dtype=torch.float64, device=DEVICE)
        for lo, hi in ((0, sy.nup), (sy.nup, ne)):
            if hi == lo:
                continue
            occ = torch.as_tensor(sy.iworbd[0, lo:hi].astype(np.int64), device=DEVICE)
            A = phi[:, lo:hi][:, :, occ].contiguous()
            logpsi = logpsi + torch.linalg.slogdet(A)[1]
            inv = torch.linalg.inv(A).transpose(1, 2).contiguous()  # [w][electron][slot]
            drift[:, lo:hi] = (inv[..., None] * dphi[:, lo:hi][:, :, occ]).sum(2)
            ld[:, lo:hi] = (inv * lphi[:, lo:hi][:, :, occ]).sum(2)
            rows[:, lo:hi] = inv @ self.coef[occ]
        ekin = -0.5 * (ld.sum(1) + 2 * (gj * drift).sum((1, 2)) + lapj + (gj * gj).sum((1, 2)))
        z = _t(sy.znuc)[torch.as_tensor(self.type, device=DEVICE)]
        iu = torch.triu_indices(ne, ne, 1, device=DEVICE)
        pot = (1 / (x[:, iu[0]] - x[:, iu[1]]).norm(dim=-1)).sum(1)
        cu = torch.triu_indices(len(self.type), len(self.type), 1, device=DEVICE)
        pot = pot + (z[cu[0]] * z[cu[1]] / (self.cent[cu[0]] - self.cent[cu[1]]).norm(dim=-1)).sum()
        er = (x[:, :, None] - self.cent).norm(dim=-1)
        pot = pot - (z / er).sum((1, 2))
        if sy.nloc:
            wq = _t(sy.wq)
            V = torch.zeros(w, ne, len(self.type), 5, dtype=torch.float64, device=DEVICE)
            active = torch.zeros(w, ne, len(self.type), dtype=torch.bool, device=DEVICE)
            for c, it in enumerate(self.type):
                pot = pot + torch.as_tensor(self.ecp(it, int(sy.lpot[it]) - 1, er[..., c])).sum(-1)
                for l in range(int(sy.lpot[it]) - 1):
                    V[:, :, c, l] = self.ecp(it, l, er[..., c])
                    active[:, :, c] |= V[:, :, c, l].abs() > 1e-4
            kw, e, c = active.nonzero(as_tuple=True)
            count = active.sum((1, 2))
            slot = torch.arange(len(kw), device=DEVICE) - (torch.cumsum(count, 0) - count)[kw]
            nq = len(wq)
            rec = er[kw, e, c]
            xq = rec[:, None, None] * quad[kw] + self.cent[c][:, None]  # [pair][nq][3]
            ratio = torch.zeros(len(kw), nq, dtype=torch.float64, device=DEVICE)
            for s in _chunks(len(kw), 8000):
                row = rows[kw[s], e[s]].repeat_interleave(nq, 0)
                for cols, v in self.shells(xq[s].reshape(-1, 3), False):
                    ratio[s] += (v * row[:, cols]).sum(1).reshape(-1, nq)
            old = self.jastrow_at(x, x, torch.arange(ne, device=DEVICE).expand(w, ne))
            new = torch.zeros_like(ratio)
            for s in _chunks(int(count.max()), max(1, int(2e8 / (w * nq * ne * 8)))):  # pairs of all walkers, padded
                on = (slot >= s.start) & (slot < s.stop)
                pe = torch.zeros(w, s.stop - s.start, dtype=torch.long, device=DEVICE)
                px = torch.ones(w, s.stop - s.start, nq, 3, dtype=torch.float64, device=DEVICE)
                pe[kw[on], slot[on] - s.start] = e[on]
                px[kw[on], slot[on] - s.start] = xq[on]
                j = self.jastrow_at(x, px.reshape(w, -1, 3), pe.repeat_interleave(nq, 1))
                new[on] = j.reshape(w, -1, nq)[kw[on], slot[on] - s.start]
            ratio = ratio * torch.exp(new - old[kw, e][:, None])
            cos = ((x[kw, e] - self.cent[c])[:, None] * quad[kw]).sum(-1) / rec[:, None]
            yl = [torch.ones_like(cos), 3 * cos, 2.5 * (3 * cos ** 2 - 1), 3.5 * (5 * cos ** 3 - 3 * cos)]
            term = sum(yl[l] * V[kw, e, c, l][:, None] for l in range(4))
            pot = pot.index_add(0, kw, (term * wq * ratio).sum(1))
        return logpsi, lnj, ekin, ekin + pot

    # ------------------------------------------------------ derivatives
    def deriv(self, x, case):
        """d ln psi / dp [w][n] of the raw parameters, in the order of the
        system's arrays, and the determinant coefficients and orbital terms."""
        sy, out = self.sy, []
        w, ne = x.shape[:2]
        iu, ju = torch.triu_indices(ne, ne, 1, device=DEVICE)
        er = (x[:, :, None] - self.cent).norm(dim=-1)

        def form(p, o, s):
            if o == 0:
                return s / (1 + p[1] * s)
            return -p[0] * s ** 2 / (1 + p[1] * s) ** 2 if o == 1 else s ** o

        inf = torch.full((), self.ainf, dtype=torch.float64, device=DEVICE)
        for it, idx in enumerate(self.of_type):
            R = self.scaled(er[..., idx])
            for o in range(sy.norda + 1):
                out.append((form(sy.a4[it], o, R) - form(sy.a4[it], o, inf)).sum((1, 2)))
        rij = (x[:, iu] - x[:, ju]).norm(dim=-1)
        R, like, scale = self.scaled(rij), self.like[iu, ju], self.scale[iu, ju]
        for b in range(sy.nspin2b):
            for o in range(sy.nordb + 1):
                g = (form(sy.b[b], o, R) - form(sy.b[b], o, inf)) * (scale if o < 2 else 1.0)
                out.append((g if sy.nspin2b == 1 else torch.where(like == bool(b), g, 0.0)).sum(1))
        if self.terms:
            u, X = torch.exp(-self.kap * rij), torch.exp(-self.kap * er)
            for it, idx in enumerate(self.of_type):
                a, b = X[:, iu][..., idx], X[:, ju][..., idx]
                for k, l, m in self.terms:
                    out.append((u ** k * ((a ** l + b ** l) * (a * b) ** m).sum(-1)).sum(1))
        phi = (self.ao(x.reshape(-1, 3), False) @ self.coef.T).reshape(w, ne, -1)
        dets, slots, invs = [], [], []
        for lo, hi in ((0, sy.nup), (sy.nup, ne)):
            rows, which = np.unique(sy.iworbd[:, lo:hi], axis=0, return_inverse=True)
            slot = torch.as_tensor(rows.astype(np.int64), device=DEVICE)
            A = phi[:, lo:hi][:, :, slot].permute(0, 2, 1, 3).contiguous()  # [w][det][electron][slot]
            inv = torch.linalg.inv(A)
            dets.append(torch.linalg.det(A)[:, torch.as_tensor(which.reshape(-1), device=DEVICE)])
            slots.append((slot, torch.as_tensor(which.reshape(-1), device=DEVICE)))
            invs.append(inv)
        prod = dets[0] * dets[1]
        cd = _t(sy.cdet)
        psi = prod @ cd
        out += list((prod / psi[:, None]).T)
        if case["orbital_terms"]:
            V = torch.zeros_like(phi)
            for s, (lo, hi) in enumerate(((0, sy.nup), (sy.nup, ne))):
                slot, which = slots[s]
                wt = torch.zeros(w, len(slot), dtype=torch.float64, device=DEVICE)
                wt.index_add_(1, which, cd * prod / psi[:, None])
                for d in range(len(slot)):
                    V[:, lo:hi].index_add_(2, slot[d], wt[:, d, None, None] * invs[s][:, d].transpose(1, 2))
            for io, jo in _orb_terms(case["orbital_terms"]):
                out.append((V[..., int(io)] * phi[..., int(jo)]).sum(1))
        return torch.stack(out, 1)


def _chunks(n, size):
    return [slice(a, min(n, a + size)) for a in range(0, n, size)]


def exact(case, seed):
    """The 64-bit values for one determinant's energies and for the
    derivatives; None for trajectories, whose random numbers and decisions are
    the program's own, and for energies of determinant expansions."""
    op = case["op"]
    if op not in ("hpsi", "drive", "deriv"):
        return None
    sy = system_of(case)
    if op != "deriv" and sy.iworbd.shape[0] > 1:
        return None
    ex, w = _Exact(sy), case["walkers"]
    if op == "deriv":
        x = _t(sy.initial_walkers(w, seed=seed))
        o = torch.cat([ex.deriv(x[c], case) for c in _chunks(w, 128)])
        # the local energies that weigh the sums are this repository's own
        return dict(o=o.cpu().numpy(), s=(o.T.contiguous() @ o).cpu().numpy(), osum=o.sum(0).cpu().numpy(), eosum=None,
                    esum=None)
    x = sy.initial_walkers(w, seed=seed)
    if op == "drive":
        x0, plan = _drive_plan(sy, w, seed)
        xn, mask = plan[0]
        x = np.where(mask.T[..., None], xn.transpose(1, 0, 2), x0)
    quad = _t(_quadrature(sy, w, seed)) if sy.nloc else torch.zeros(w, 1, 3, dtype=torch.float64, device=DEVICE)
    x = _t(x)
    per = max(1, int(2.0e8 / (sy.nelec * max(sy.nbasis * 12, 8 * sy.nelec * (6 + 3 * sy.nordc)))))
    got = [ex.hpsi(x[c], quad[c]) for c in _chunks(w, per)]
    logpsi, lnj, ekin, energy = (torch.cat(v).cpu().numpy() for v in zip(*got))
    if op == "drive":
        return dict(logpsi_moves=None, drift=None, logpsi=logpsi, ekin=ekin, energy=energy)
    return dict(logpsi=logpsi, psij=lnj, ekin=ekin, energy=energy)
