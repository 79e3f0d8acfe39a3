"""Timed cases of the excited-state core, through the package's public entry points.

Each case is one pass of a user's program over data that it holds on the host
(the library takes the Fortran driver's host arrays): the molecule's boundary
arrays go in, spectra or response tensors come out.

Kinds:

* ``spectrum``: ``StdaHip.setup`` + ``csf`` + ``solve_tda`` on one molecule, the
  drop-in for the reference's sTDA run; ``precision`` "fp64" or "mixed";
  ``roots`` 0 asks for every root below the threshold, as the reference does.
* ``rpa``: the same with ``solve_rpa`` (sTD-DFT).
* ``alpha``: ``setup`` + ``lresp``, the frequency-dependent polarizability.
* ``series``: ``spectrum`` on molecules of mixed sizes, one after the other on one
  context (the benchmark's plain pass).
* ``prepare``: ``prep.prepare`` on the device, from a molecule with its basis and
  MO coefficients to the core's inputs (AO integrals, Loewdin, moments).
* ``curves``: ``StdaHip.gspec_curves``, the broadened curves of many spectra.

Molecules are those of the repository's benchmark: random organic-like clusters
(C:H:N:O = 45:45:5:5, 0.1 atoms per cubic Angstrom, pairs at least 1 Angstrom
apart) or a planar polyene chain, random orthogonal orbitals, occupied energies
uniform in [-20, -5] eV and virtual ones in [-1, 15] eV, with the frontier pair within
half an eV of the ends so that small molecules too have excitations below the
threshold.  The boundary arrays are drawn in the Loewdin basis directly, so that
making them needs no integrals.
"""

from __future__ import annotations

import functools
import math

import numpy as np
import torch

from stda_amd.basis import shells_for
from stda_amd.core import StdaHip
from stda_amd.molden import build_ao_basis
from stda_amd.prep import CoreInputs, prepare as prepare_core

EV = 27.211385050
BOHR = 0.52917721092
THRP = 1e-4


def listed():
    return [
        # the smallest request of a mixed stream: latency of one solve
        dict(name="spectrum_10", kind="spectrum", shape="cluster", atoms=10, basis="minimal",
             thr=7.0, ax=0.25, roots=20, precision="fp64", triplet=False),
        # the reference's default run: every root below the threshold, of a small molecule
        dict(name="window_21", kind="spectrum", shape="cluster", atoms=21, basis="minimal",
             thr=7.0, ax=0.5, roots=0, precision="fp64", triplet=False),
        # a conjugated chain, C14H16, with the ten lowest roots
        dict(name="spectrum_polyene30", kind="spectrum", shape="polyene", atoms=30,
             basis="minimal", thr=7.0, ax=0.25, roots=10, precision="fp64", triplet=False),
        # an ordinary molecule of an odd size, plain FP64
        dict(name="spectrum_79", kind="spectrum", shape="cluster", atoms=79, basis="minimal",
             thr=7.0, ax=0.25, roots=20, precision="fp64", triplet=False),
        # the upper end of the mixed sizes, plain FP64
        dict(name="spectrum_200", kind="spectrum", shape="cluster", atoms=200, basis="minimal",
             thr=7.0, ax=0.25, roots=20, precision="fp64", triplet=False),
        # a large molecule in mixed precision
        dict(name="spectrum_mixed_133", kind="spectrum", shape="cluster", atoms=133,
             basis="minimal", thr=7.0, ax=0.25, roots=20, precision="mixed", triplet=False),
        # a split-valence basis, a wide window, many roots
        dict(name="spectrum_split_180", kind="spectrum", shape="cluster", atoms=180,
             basis="split", thr=10.0, ax=0.25, roots=50, precision="fp64", triplet=False),
        # sTD-DFT on a medium molecule
        dict(name="rpa_60", kind="rpa", shape="cluster", atoms=60, basis="minimal", thr=7.0,
             ax=0.25, roots=20, precision="fp64", triplet=False),
        # static and dynamic polarizability
        dict(name="alpha_85", kind="alpha", shape="cluster", atoms=85, basis="minimal", thr=7.0,
             ax=0.25, precision="fp64", nfreq=3),
        # molecules of mixed sizes one after the other, as a screening program runs them
        dict(name="series_16", kind="series", molecules=16, low=10, high=200, thr=7.0, ax=0.25,
             roots=20, precision="fp64"),
        # upstream preparation of a large molecule on the device
        dict(name="prepare_240", kind="prepare", atoms=240, basis="minimal", thr=10.0, ax=0.25),
        # the broadened curves of many spectra
        dict(name="curves_512", kind="curves", spectra=512, lines=20, points=2000, uv=False),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["spectrum"] * 6 + ["rpa"] * 2 + ["alpha"] * 2 + ["series"] * 2 +
                      ["prepare", "curves"])
    ax = rng.choice([0.25, 0.25, 0.5])
    if kind == "spectrum":
        precision = rng.choice(["fp64", "fp64", "mixed"])
        triplet = rng.random() < 0.1
        if rng.random() < 0.2:
            return dict(kind=kind, shape="cluster", atoms=_log_int(rng, 10, 170), basis="split",
                        thr=10.0, ax=ax, roots=rng.choice([20, 50]), precision=precision,
                        triplet=triplet)
        if rng.random() < 0.15:
            return dict(kind=kind, shape="cluster", atoms=_log_int(rng, 12, 30), basis="minimal",
                        thr=7.0, ax=ax, roots=0, precision="fp64", triplet=triplet)
        if rng.random() < 0.15:
            return dict(kind=kind, shape="polyene", atoms=2 * rng.randint(6, 40) + 2,
                        basis="minimal", thr=7.0, ax=ax, roots=rng.choice([10, 20]),
                        precision=precision, triplet=triplet)
        return dict(kind=kind, shape="cluster", atoms=_log_int(rng, 10, 200), basis="minimal",
                    thr=7.0, ax=ax, roots=rng.choice([10, 20, 20, 30]), precision=precision,
                    triplet=triplet)
    if kind == "rpa":
        return dict(kind=kind, shape="cluster", atoms=_log_int(rng, 12, 90), basis="minimal",
                    thr=7.0, ax=ax, roots=rng.choice([10, 20]),
                    precision=rng.choice(["fp64", "mixed"]), triplet=False)
    if kind == "alpha":
        return dict(kind=kind, shape="cluster", atoms=_log_int(rng, 12, 110), basis="minimal",
                    thr=7.0, ax=ax, precision=rng.choice(["fp64", "fp64", "mixed"]),
                    nfreq=rng.choice([1, 3, 4]))
    if kind == "series":
        low = _log_int(rng, 10, 20)
        return dict(kind=kind, molecules=_log_int(rng, 4, 16), low=low,
                    high=low + _log_int(rng, 20, 160), thr=7.0, ax=ax,
                    roots=rng.choice([10, 20, 20]), precision=rng.choice(["fp64", "mixed"]))
    if kind == "prepare":
        return dict(kind=kind, atoms=_log_int(rng, 10, 200), basis="minimal",
                    thr=rng.choice([7.0, 10.0]), ax=ax)
    return dict(kind=kind, spectra=_log_int(rng, 1, 512), lines=_log_int(rng, 5, 60),
                points=rng.choice([2000, 2501]), uv=rng.random() < 0.5)


# ------------------------------------------------------------------------- inputs
def _geometry(rng, shape, atoms):
    """Nuclear charges and positions (Bohr)."""
    if shape == "polyene":   # C_n H_{n+2} zig-zag in the plane, C-H pointing outwards
        nc = (atoms - 2) // 2
        step = 1.40 + rng.uniform(-0.05, 0.05, nc - 1)
        ang = np.radians(np.where(np.arange(1, nc) % 2, 30.0, -30.0))
        carbon = np.zeros((nc, 3))
        carbon[1:, 0] = np.cumsum(step * np.cos(ang))
        carbon[1:, 1] = np.cumsum(step * np.sin(ang))
        side = np.where(np.arange(nc) % 2, 1.0, -1.0)
        hyd = carbon + np.stack([np.zeros(nc), 1.08 * side, np.zeros(nc)], axis=1)
        ends = np.stack([carbon[0] + [-0.94, 0.54, 0.0],
                         carbon[-1] + [0.94, -0.54 * side[-1], 0.0]])
        return (np.r_[np.full(nc, 6), np.full(nc + 2, 1)],
                np.vstack([carbon, hyd, ends]) / BOHR)
    counts = np.floor(np.array([0.45, 0.45, 0.05, 0.05]) * atoms).astype(int)
    counts[0] += atoms - counts.sum()
    Z = np.repeat([6, 1, 7, 8], counts)[rng.permutation(atoms)]
    side = (atoms / 0.1) ** (1.0 / 3.0)
    pts = np.empty((atoms, 3))
    n = 0
    while n < atoms:
        p = rng.uniform(0.0, side, 3)
        if n == 0 or ((pts[:n] - p) ** 2).sum(1).min() >= 1.0:
            pts[n] = p
            n += 1
    return Z, pts / BOHR


def _haar(rng, n):
    q, r = np.linalg.qr(rng.standard_normal((n, n)))
    return q * np.sign(np.diag(r))[None, :]


def _energies(rng, nocc, nvir):
    """Occupied and virtual orbital energies (Hartree), ascending."""
    occ, vir = rng.uniform(-20.0, -5.0, nocc), rng.uniform(-1.0, 15.0, nvir)
    occ[0], vir[0] = rng.uniform(-5.5, -5.0), rng.uniform(-1.0, -0.5)
    return np.sort(occ) / EV, np.sort(vir) / EV


def _core_inputs(rng, shape, atoms, basis, thr, ax):
    """The core's boundary arrays of one molecule."""
    Z, xyz = _geometry(rng, shape, atoms)
    heavy = 5 if basis == "minimal" else 9
    per = np.where(Z == 1, 1 if basis == "minimal" else 2, heavy)
    atom = np.repeat(np.arange(atoms), per)
    nao, nocc = len(atom), int(Z.sum()) // 2
    U = _haar(rng, nao)
    eo, ev = _energies(rng, nocc, nao - nocc)
    deps = 2.0 * (1.0 + 0.8 * ax) * thr / EV      # the driver's orbital window
    osel = np.nonzero(eo > ev[0] - deps)[0]
    vsel = nocc + np.nonzero(ev < eo[-1] + deps)[0]
    clow = U[:, np.r_[osel, vsel]]
    # one-electron operators in the Loewdin basis: a local overlap-like weight times
    # the pair's midpoint (dipole), times its separation (gradient), and r x gradient
    pos = xyz[atom] - xyz.mean(axis=0)
    diff = pos[:, None, :] - pos[None, :, :]
    mid = 0.5 * (pos[:, None, :] + pos[None, :, :])
    g = rng.uniform(-0.5, 0.5, (nao, nao))
    wt = np.tril(g, -1) + np.tril(g, -1).T
    wt *= np.exp(-0.25 * (diff ** 2).sum(-1))
    onsite = wt * (atom[:, None] == atom[None, :])
    sgn = np.sign(np.arange(nao)[:, None] - np.arange(nao)[None, :])
    grad = [0.5 * wt * diff[:, :, k] + 0.5 * onsite * sgn for k in range(3)]
    ops = [-(np.eye(nao) * pos[:, k] + wt * mid[:, :, k] + onsite) for k in range(3)]
    for k in range(3):
        a, b = (k + 1) % 3, (k + 2) % 3
        ops.append(mid[:, :, a] * grad[b] - mid[:, :, b] * grad[a])
    ops += [-m for m in grad]
    low = np.tril_indices(clow.shape[1])
    mom = np.empty((9, len(low[0])))
    for q in range(9):
        mom[q] = (clow.T @ ops[q] @ clow).T[low]
    pack = np.zeros((4, atoms))
    pack[:3], pack[3] = xyz.T, Z
    return CoreInputs(ncent=atoms, nao=nao, no=len(osel), nv=len(vsel),
                      clow=np.asfortranarray(clow),
                      epsi=np.r_[eo[osel], ev[vsel - nocc]],
                      iaoat=(atom + 1).astype(np.int32), xyz=np.asfortranarray(pack),
                      moments=mom)


def _frequencies(case):
    return [0.0, 0.05, 0.1, 0.075][:case["nfreq"]]


@functools.lru_cache(maxsize=None)
def _context(precision):
    """The context that a program keeps for all its molecules."""
    h = StdaHip(0)
    h.set_precision(precision)
    return h


def _rng(case, seed):
    return np.random.Generator(np.random.PCG64([int(seed) & 0x7FFFFFFF, 77]))


def prepare(case, seed):
    rng = _rng(case, seed)
    kind = case["kind"]
    if kind == "series":
        sizes = np.rint(np.exp(rng.uniform(math.log(case["low"]), math.log(case["high"]),
                                           case["molecules"]))).astype(int)
        return {"case": case, "h": _context(case["precision"]),
                "mols": [_core_inputs(rng, "cluster", int(n), "minimal", case["thr"], case["ax"])
                         for n in sizes]}
    if kind == "prepare":
        Z, xyz = _geometry(rng, "cluster", case["atoms"])
        mol = build_ao_basis(Z.tolist(), xyz, [shells_for(int(z), case["basis"]) for z in Z])
        h = _context("fp64")
        e, V = np.linalg.eigh(h.ao_ints(mol)["S"])
        nocc = int(Z.sum()) // 2
        mol.C = (V / np.sqrt(e)) @ (V.T @ _haar(rng, mol.nao))
        mol.eps = np.concatenate(_energies(rng, nocc, mol.nao - nocc))
        mol.occ = np.r_[np.full(nocc, 2.0), np.zeros(mol.nao - nocc)]
        return {"case": case, "h": h, "mol": mol}
    if kind == "curves":
        n, L = case["spectra"], case["lines"]
        x = np.sort(rng.uniform(2.5, 7.0, (n, L)), axis=1)
        y = rng.exponential(0.05, (n, L)) if case["uv"] else 20.0 * rng.standard_normal((n, L))
        lo = np.maximum(x[:, 0] - 0.2 * (x[:, -1] - x[:, 0]), 0.5)
        hi = x[:, -1] + 0.2 * (x[:, -1] - x[:, 0])
        return {"case": case, "h": _context("fp64"), "off": L * np.arange(n + 1, dtype=np.int64),
                "x": x.ravel(), "y": y.ravel(), "w": np.full(n * L, 0.4), "emin": lo,
                "step": (hi - lo) / case["points"]}
    return {"case": case, "h": _context(case["precision"]),
            "ci": _core_inputs(rng, case["shape"], case["atoms"], case["basis"], case["thr"],
                               case["ax"])}


def _fill(a, shape):
    """`a` at the head of a zeroed array: tables of a fixed size, as the Fortran driver
    holds them, whatever the number of CSFs and roots of a molecule."""
    out = np.zeros(shape, dtype=a.dtype)
    out[tuple(slice(n) for n in a.shape)] = a
    return out


def _capacity(case):
    """Largest numbers of CSFs and of roots: all occupied x virtual pairs."""
    if case["shape"] == "polyene":
        nc = (case["atoms"] - 2) // 2
        nao = 6 * nc + 2 if case["basis"] == "minimal" else 11 * nc + 4
        nocc = (7 * nc + 2) // 2
    else:
        n = [int(f * case["atoms"]) for f in (0.45, 0.45, 0.05, 0.05)]
        n[0] += case["atoms"] - sum(n)
        heavy, hyd = (5, 1) if case["basis"] == "minimal" else (9, 2)
        nao = heavy * (n[0] + n[2] + n[3]) + hyd * n[1]
        nocc = (6 * n[0] + n[1] + 7 * n[2] + 8 * n[3]) // 2
    pairs = nocc * (nao - nocc)
    return pairs, case["roots"] or pairs


def run(state):
    case, h = state["case"], state["h"]
    kind = case["kind"]
    if kind == "series":
        res = []
        for ci in state["mols"]:
            h.setup(ci, case["thr"], case["ax"])
            res.append(h.solve_tda(case["roots"], vectors=False))
        return {"omega": np.stack([_fill(r.omega, case["roots"]) for r in res]),
                "props": np.stack([_fill(r.props, (case["roots"], 4)) for r in res]),
                "alpha": np.stack([r.alpha_sos for r in res])}
    if kind == "prepare":
        ci = prepare_core(state["mol"], case["thr"], case["ax"], device=h)
        return {"clow": ci.clow, "moments": ci.moments, "epsi": ci.epsi}
    if kind == "curves":
        e, r = h.gspec_curves(state["off"], state["x"], state["y"], state["w"], state["emin"],
                              state["step"], case["points"], 1 if case["uv"] else 0, 1.0)
        return {"e": e, "r": r}
    ci = state["ci"]
    if kind == "alpha":
        h.setup(ci, case["thr"], case["ax"])
        return {"alpha": np.stack([a for _, a in h.lresp(_frequencies(case))])}
    h.setup(ci, case["thr"], case["ax"], triplet=case["triplet"])
    conf, ed = h.csf()
    solve = h.solve_rpa if kind == "rpa" else h.solve_tda
    sol = solve(case["roots"] or None, vectors=False)
    pairs, roots = _capacity(case)
    return {"conf": _fill(conf, (pairs, 2)), "ed": _fill(ed, pairs),
            "omega": _fill(sol.omega, roots), "props": _fill(sol.props, (roots, 4)),
            "alpha": sol.alpha_sos}


# ------------------------------------------------------------------------- work
def _sizes(atoms, basis, thr, ax):
    """Expected sizes of a molecule: AOs, window, pairs, primaries, secondaries."""
    nao = atoms * (3.2 if basis == "minimal" else 5.85)
    nocc = 1.95 * atoms
    nvir = nao - nocc
    deps = 2.0 * (1.0 + 0.8 * ax) * thr
    no, nv = nocc * min(1.0, (deps - 4.0) / 15.0), nvir * min(1.0, (deps - 4.0) / 16.0)
    prim = nocc * nvir * (thr + 1.0 - 4.0) ** 2 / 480.0
    return nao, no, nv, prim, max(no * nv - prim, 0.0)


def _molecule_work(atoms, basis, thr, ax, vectors):
    """Inputs, couplings of the PT2 selection, p = gamma q, and `vectors` products with A."""
    nao, no, nv, prim, sec = _sizes(atoms, basis, thr, ax)
    m = no + nv
    flops = (4.0 * atoms * sec * prim + 2.0 * atoms ** 2 * (no * nv + no * no / 2) +
             vectors * 4.0 * (nao * no * nv + nao * nao * no))
    return 8.0 * (nao * m + 4.5 * m * m) + 20.0 * (prim + sec), flops


def work(case):
    kind = case["kind"]
    if kind == "curves":
        n = case["spectra"]
        return {"bytes": 8.0 * n * (3 * case["lines"] + 2 * case["points"]),
                "flops": 25.0 * n * case["lines"] * case["points"]}
    if kind == "prepare":
        nao, no, nv, _, _ = _sizes(case["atoms"], case["basis"], case["thr"], case["ax"])
        m = no + nv
        return {"bytes": 8.0 * (2 * nao * m + 4.5 * m * m),
                "flops": 9.0 * 2 * (nao * nao * m + nao * m * m) + 9.0 * nao ** 3}
    if kind == "series":
        r = math.log(case["high"] / case["low"])
        sizes = [case["low"] * math.exp(r * (i + 0.5) / case["molecules"])
                 for i in range(case["molecules"])]
        each = [_molecule_work(n, "minimal", case["thr"], case["ax"], 8 * case["roots"])
                for n in sizes]
        return {"bytes": sum(b for b, _ in each), "flops": sum(f for _, f in each)}
    vectors = {"rpa": 24, "spectrum": 8}.get(kind, 0) * (case.get("roots") or 2 * case["atoms"])
    if kind == "alpha":
        vectors = 60 * case["nfreq"]
    b, f = _molecule_work(case["atoms"], case["basis"], case["thr"], case["ax"], vectors)
    return {"bytes": b, "flops": f}


# ------------------------------------------------------------------------- 64-bit values
_ETA = {1: 0.472592880, 6: 0.421954120, 7: 0.504381930, 8: 0.586918630}
_ROT = 235.7220


class _Core:
    """The method on explicit matrices in 64 bits."""

    def __init__(self, ci, thr, ax, triplet=False):
        self.dev = torch.device("cuda" if torch.cuda.is_available() else "cpu")
        t = self.t = lambda a: torch.as_tensor(np.ascontiguousarray(a), dtype=torch.float64,
                                               device=self.dev)
        na, no, nv = ci.ncent, ci.no, ci.nv
        self.ci, self.no, self.nv, self.ax, self.ak = ci, no, nv, ax, 0.0 if triplet else 2.0
        eta = t([_ETA[int(z)] for z in ci.xyz[3]])
        r = t(ci.xyz[:3].T)
        d = (r[:, None, :] - r[None, :, :]).square().sum(-1).sqrt()
        hard = 0.5 * (eta[:, None] + eta[None, :])
        bj, bk = 0.20 + 1.830 * ax, 1.420 + 0.480 * ax
        gj = (d ** bj + (hard * ax) ** -bj) ** (-1.0 / bj)
        gk = (d ** bk + hard ** -bk) ** (-1.0 / bk)
        C = t(ci.clow)
        ind = torch.zeros((na, ci.nao), dtype=torch.float64, device=self.dev)
        ind[torch.as_tensor(ci.iaoat.astype(np.int64) - 1), torch.arange(ci.nao)] = 1.0
        Co, Cv = C[:, :no], C[:, no:]

        def charges(a, b):   # (atoms, n_a, n_b), a few orbitals at a time
            out = torch.empty((na, a.shape[1], b.shape[1]), dtype=torch.float64, device=self.dev)
            for i in range(a.shape[1]):
                out[:, i] = ind @ (a[:, i:i + 1] * b)
            return out

        self.qia, self.qab, qij = charges(Co, Cv), charges(Cv, Cv), charges(Co, Co)
        self.pia = (gk @ self.qia.reshape(na, -1)).reshape(na, no, nv)
        self.pij = (gj @ qij.reshape(na, -1)).reshape(na, no, no)
        del qij
        at = torch.as_tensor(ci.iaoat.astype(np.int64) - 1, device=self.dev)
        self.Co, self.Cv, self.gj_ao = Co, Cv, gj[at][:, at]
        diag = torch.arange(nv, device=self.dev)
        occ = torch.arange(no, device=self.dev)
        J = self.pij[:, occ, occ].T @ self.qab[:, diag, diag]
        eps = t(ci.epsi)
        K = (self.pia * self.qia).sum(0)
        de = (eps[None, no:] - eps[:no, None] - J + self.ak * K).reshape(-1)
        lim = thr / EV
        prim = torch.nonzero(de <= lim)[:, 0]
        prim = prim[torch.argsort(de[prim], stable=True)]
        sec = torch.nonzero(de > lim)[:, 0]
        pert, lower = torch.zeros_like(de), torch.zeros(len(prim), dtype=torch.float64,
                                                        device=self.dev)
        take = torch.zeros(len(de), dtype=torch.bool, device=self.dev)
        for k in range(no):
            rows = sec[sec // nv == k]
            if not len(rows) or not len(prim):
                continue
            pt = self.coupling(rows, prim).square() / (de[rows, None] - de[None, prim] + 1e-10)
            pert[rows] = pt.sum(1)
            take[rows] = pert[rows] > THRP
            lower += pt[~take[rows]].sum(0)
        sec = sec[take[sec]]
        self.idx = torch.cat([prim, sec])
        self.ed = torch.cat([de[prim] - lower, de[sec]])
        self.n = len(self.idx)
        self.K, self.J = K.reshape(-1)[self.idx], J.reshape(-1)[self.idx]
        i, a = self.idx // nv, self.idx % nv
        hi, lo = no + a, i
        mom = t(ci.moments)
        self.mom = mom[:, lo + hi * (hi + 1) // 2]          # (9, n)
        self.conf = torch.stack([i + 1, no + a + 1], 1).cpu().numpy()

    def coupling(self, rows, cols, ak=None, aj=1.0, aexc=0.0):
        """ak K - aj J + aexc (exchange of the B block) for rows of ONE occupied orbital."""
        nv, na = self.nv, self.qia.shape[0]
        ak = self.ak if ak is None else ak
        k, c = int(rows[0]) // nv, rows % nv
        j, b = cols // nv, cols % nv
        q = self.qia.reshape(na, -1)
        out = ak * (self.pia[:, k, :][:, c].T @ q[:, cols])
        if aj:
            jo, inv = torch.unique(j, return_inverse=True)
            m = self.pij[:, k, jo].T @ self.qab.reshape(na, -1)      # (no', nv nv)
            out -= aj * m.reshape(len(jo), nv, nv)[inv[None, :], c[:, None], b[None, :]]
        if aexc:   # (kb|jc)
            jo, inv = torch.unique(j, return_inverse=True)
            m = (self.pia[:, k, :].T @ self.qia[:, jo].reshape(na, -1)).reshape(nv, len(jo), nv)
            out += aexc * m[b[None, :], inv[None, :], c[:, None]]
        return out

    def matrix(self, diag, **kw):
        M = torch.empty((self.n, self.n), dtype=torch.float64, device=self.dev)
        occ = self.idx // self.nv
        for k in torch.unique(occ).tolist():
            at = torch.nonzero(occ == k)[:, 0]
            M[at] = self.coupling(self.idx[at], self.idx, **kw)
        if diag is not None:
            M.diagonal().copy_(diag)
        return M

    def tda(self):
        return self.matrix(self.ed)

    def tda_times(self, X):
        """A X without the matrix, through the transition densities Co x Cv^T."""
        out = torch.empty_like(X)
        na, q = self.qia.shape[0], self.qia.reshape(self.qia.shape[0], -1)
        full = torch.zeros(q.shape[1], dtype=X.dtype, device=X.device)
        for v in range(X.shape[1]):
            full[self.idx] = X[:, v]
            y = self.ak * (self.pia.reshape(na, -1).T @ (q @ full))
            G = self.gj_ao * (self.Co @ full.reshape(self.no, self.nv) @ self.Cv.T)
            y -= (self.Co.T @ G @ self.Cv).reshape(-1)
            out[:, v] = y[self.idx]
        return out + (self.ed - self.ak * self.K + self.J)[:, None] * X

    def apb(self):
        return self.matrix(self.ed + self.ak * self.K - self.ax * self.K, ak=2.0 * self.ak,
                           aexc=-self.ax)

    def amb(self):
        return self.matrix(self.ed - self.ak * self.K + self.ax * self.K, ak=0.0, aexc=self.ax)

    def bhalf_times(self, X):
        out = torch.empty_like(X)
        occ = self.idx // self.nv
        for k in torch.unique(occ).tolist():
            at = torch.nonzero(occ == k)[:, 0]
            out[at] = self.coupling(self.idx[at], self.idx, ak=0.5 * self.ak, aj=0.0,
                                    aexc=-0.5 * self.ax) @ X
        return out


def _orth(V, W):
    for _ in range(3):
        W = W / W.norm(dim=0).clamp_min(1e-300)
        W = W - V @ (V.T @ W)
        W = W[:, W.norm(dim=0) > 1e-8]
        if not W.shape[1]:
            return W
        U, s, _ = torch.linalg.svd(W, full_matrices=False)
        W = U[:, s > 1e-8 * s[0]]
    return W


def _lowest(A, k):
    """The k lowest eigenpairs of a symmetric matrix."""
    if A.shape[0] <= 3000:
        w, X = torch.linalg.eigh(A)
        return w[:k], X[:, :k]
    return _davidson(lambda V: A @ V, A.diagonal(), k)


def _davidson(times, d, k):
    V = torch.zeros((len(d), 2 * k), dtype=d.dtype, device=d.device)
    V[torch.argsort(d)[:2 * k], torch.arange(2 * k, device=d.device)] = 1.0
    AV = times(V)
    for _ in range(150):
        H = V.T @ AV
        w, Y = torch.linalg.eigh(0.5 * (H + H.T))
        X, AX = V @ Y[:, :k], AV @ Y[:, :k]
        R = AX - X * w[:k]
        bad = R.norm(dim=0) > 1e-12
        if not bad.any():
            break
        if V.shape[1] > 10 * k:
            m = 3 * k
            V, AV = V @ Y[:, :m], AV @ Y[:, :m]
        den = w[:k][bad][None, :] - d[:, None]
        W = _orth(V, R[:, bad] / torch.where(den.abs() < 1e-3, den.sign() * 1e-3 + 1e-30, den))
        if not W.shape[1]:
            break
        V, AV = torch.cat([V, W], 1), torch.cat([AV, times(W)], 1)
    return w[:k], X


def _lowest_rpa(P, M, k):
    """w, X+Y, X-Y of the k lowest roots of (A-B)(A+B), P = A+B, M = A-B."""
    L = torch.linalg.cholesky(M)
    w2, Z = _lowest(L.T @ P @ L, k)
    w = w2.sqrt()
    xpy = L @ Z / w.sqrt()                      # (A-B)^1/2-like factor, normalised below
    xmy = torch.linalg.solve_triangular(L.T, Z, upper=True) * w.sqrt()
    return w, xpy, xmy


def _props(c, w, xpy, xmy, bx=None):
    l, m, v = c.mom[0:3] @ xpy, c.mom[3:6] @ xmy, c.mom[6:9] @ xmy
    ef = 1.0 / (w + 1e-8)
    fl = w * (2.0 / 3.0) * c.ak * (l * l).sum(0)
    fv = ef * (2.0 / 3.0) * c.ak * (v * v).sum(0)
    rl = -_ROT * c.ak * (l * m).sum(0)
    rv = -_ROT * c.ak * (v * m).sum(0) * ef
    if bx is not None:
        bx = bx * ef
        v2, m2 = c.mom[6:9] @ bx, c.mom[3:6] @ bx
        scale = 1.0 / (w ** (1.0 - torch.exp(-150.0 * w * w)) + 1e-8)
        rv = -_ROT * c.ak * ((v * m).sum(0) + (v2 * m).sum(0) + (v * m2).sum(0)) * scale
    return torch.stack([fl, fv, rl, rv], 1), 2.0 * c.ak * (l * ef) @ l.T


def _spectrum(c, roots, thr):
    if roots and c.n > 12000:
        w, X = _davidson(c.tda_times, c.ed, roots)
        return w, *_props(c, w, X, X, c.bhalf_times(X))
    A = c.tda()
    if roots:
        w, X = _lowest(A, min(roots, c.n))
    else:
        w, X = torch.linalg.eigh(A)
        keep = (w > 0.0) & (w <= thr / EV)
        w, X = w[keep], X[:, keep]
    del A
    return w, *_props(c, w, X, X, c.bhalf_times(X))


def exact(case, seed):
    kind = case["kind"]
    if kind == "prepare":
        return None
    if kind == "curves":
        s = prepare(case, seed)
        n, L, m = case["spectra"], case["lines"], case["points"]
        x, y, w = (s[q].reshape(n, L) for q in "xyw")
        if case["uv"]:   # the reference's single-precision constants
            y = float(np.float32(np.float32(6.4607) * np.float32(1.5))) * y / (3.67493e-2 * x)
        f1 = 9.186e-3 if case["uv"] else float(np.float32(22.97))
        amp = x * y / (f1 * float(np.float32(1.7724539)) * w)
        e = s["emin"][:, None] + np.arange(1, m + 1)[None, :] * s["step"][:, None]
        r = sum(amp[:, q:q + 1] * np.exp(-((e - x[:, q:q + 1]) / w[:, q:q + 1]) ** 2)
                for q in range(L))
        return {"e": e, "r": r}
    if kind == "series":
        parts = []
        for ci in prepare(case, seed)["mols"]:
            c = _Core(ci, case["thr"], case["ax"])
            w, pr, al = (v.cpu().numpy() for v in _spectrum(c, case["roots"], case["thr"]))
            parts.append((_fill(w, case["roots"]), _fill(pr, (case["roots"], 4)), al))
        return {q: np.stack([p[i] for p in parts])
                for i, q in enumerate(("omega", "props", "alpha"))}
    _, _, _, prim, sec = _sizes(case["atoms"], case["basis"], case["thr"], case["ax"])
    if kind != "spectrum" and prim + sec > 16000:
        return None
    ci = prepare(case, seed)["ci"]
    c = _Core(ci, case["thr"], case["ax"], case.get("triplet", False))
    if kind == "alpha":
        P, M = c.apb(), c.amb()
        mu = c.mom[0:3].T
        inv = torch.cholesky_inverse(torch.linalg.cholesky(M))
        out = [4.0 * mu.T @ torch.linalg.solve(P - f * f * inv, mu) for f in _frequencies(case)]
        return {"alpha": torch.stack(out).cpu().numpy()}
    if kind == "rpa":
        w, xpy, xmy = _lowest_rpa(c.apb(), c.amb(), min(case["roots"], c.n))
        props, alpha = _props(c, w, xpy, xmy)
    else:
        w, props, alpha = _spectrum(c, case["roots"], case["thr"])
    pairs, roots = _capacity(case)
    return {"conf": None, "ed": _fill(c.ed.cpu().numpy(), pairs),
            "omega": _fill(w.cpu().numpy(), roots),
            "props": _fill(props.cpu().numpy(), (roots, 4)), "alpha": alpha.cpu().numpy()}
