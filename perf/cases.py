"""The calls that users of this package make, with their sizes, inputs, work and
tolerances.

Kinds of call (each through the package's public classes):

* force      one ForceField call of a driver with its own integrator: positions
             in, the skin check, forces, energy and virial out (host arrays)
* nvt        NVT(T, dt).run and the atoms' positions and velocities after it
* nst        NST(S, T, dt).run, the same with the box
* muvt       MuVT(mu, T, dt, gas, seed).run, the same with the exchanged atoms
* min        MinLBFGS().run from given positions
* dmd        AtomsDMD.derivative(): free energy and its gradient
* newton     one implicit step of the DMD concentrations
* gcmc       attempts of a batch of cells
* replica    minimisation of a batch of cells, from the cells to their positions

Sizes are those of the package's benchmark and tests, and odd boxes between
them. Positions start a quarter of a lattice constant inside the box, so that
no atom sits on a face.
"""
import functools
import math

import numpy as np
import torch

import mapp4py_amd as M
from mapp4py_amd import potentials as pot

KB = pot.KB_EV
A_CU, A_FE, A_NI = 3.615, 2.86, 3.52


def listed():
    return [
        # a driver's single force call on the smallest box that is used in earnest: launches and copies
        {"name": "force_cu_256", "kind": "force", "n0": 4, "n1": 4, "n2": 4, "nr": 2000},
        # an ordinary box of one element, as a user runs most of the time
        {"name": "nvt_cu_32k", "kind": "nvt", "alloy": "cu", "n0": 20, "n1": 20, "n2": 20, "T": 300.0, "steps": 100},
        # the largest: the benchmark's 8.4 million atoms
        {"name": "nvt_cu_8m", "kind": "nvt", "alloy": "cu", "n0": 128, "n1": 128, "n2": 128, "T": 300.0,
         "steps": 100},
        # a binary alloy with its own density per pair (eam/fs)
        {"name": "nvt_feni_1m", "kind": "nvt", "alloy": "feni", "n0": 128, "n1": 64, "n2": 64, "T": 600.0,
         "steps": 50},
        # a barostat run, which needs the stress of every step, in a box of odd sides
        {"name": "nst_cu_260k", "kind": "nst", "n0": 37, "n1": 41, "n2": 43, "T": 300.0, "steps": 50},
        # molecular dynamics with exchanges of a gas element, three elements in the table
        {"name": "muvt_nih_11k", "kind": "muvt", "n0": 14, "gas": 200, "steps": 100, "nevery": 50, "attempts": 500},
        # relaxation of a large cell with vacancies
        {"name": "min_cu_1m", "kind": "min", "n0": 64, "n1": 64, "n2": 64, "steps": 10},
        # diffusive MD: the quadrature at the benchmark's size, FP32 pair splines
        {"name": "dmd_cuh_262k", "kind": "dmd", "n0": 32, "n1": 32, "n2": 64, "nquad": 3, "fp32": True},
        # the same in full FP64 with five points, at the size of the diffusion example
        {"name": "dmd_cuh_16k_fp64", "kind": "dmd", "n0": 16, "n1": 16, "n2": 16, "nquad": 5, "fp32": False},
        # an implicit step of the concentrations: rates, Jacobian products and GMRES; odd sides
        {"name": "newton_cuh_60k", "kind": "newton", "n0": 23, "n1": 25, "n2": 26, "nquad": 3},
        # thousands of small cells with a gas reservoir
        {"name": "gcmc_nih_4096", "kind": "gcmc", "cells": 4096, "attempts": 64},
        # many small cells relaxed together
        {"name": "replica_nih_1024", "kind": "replica", "cells": 1024, "steps": 20},
    ]


def _sides(rng, per_cell, lo, hi, kmin):
    """sides of a box of about exp(U(log lo, log hi)) atoms, up to 1.5 : 1 apart"""
    n = math.exp(rng.uniform(math.log(lo), math.log(hi))) / per_cell
    a, b = rng.uniform(0.8, 1.25), rng.uniform(0.8, 1.25)
    k = n ** (1.0 / 3.0)
    return {"n0": max(kmin, round(k * a)), "n1": max(kmin, round(k * b)), "n2": max(kmin, round(k / (a * b)))}


def draw(rng):
    kind = rng.choice(["force", "nvt", "nvt", "nst", "muvt", "min", "dmd", "dmd", "newton", "gcmc", "replica"])
    if kind == "force":
        return {"kind": kind, **_sides(rng, 4, 256, 1_000_000, 4), "nr": rng.choice([2000, 10000])}
    if kind == "nvt":
        alloy = rng.choice(["cu", "feni"])
        s = _sides(rng, 4, 256, 2_000_000, 4) if alloy == "cu" else _sides(rng, 2, 432, 1_200_000, 6)
        return {"kind": kind, "alloy": alloy, **s, "T": round(rng.uniform(200.0, 700.0), 1), "steps": 50}
    if kind == "nst":
        return {"kind": kind, **_sides(rng, 4, 500, 1_000_000, 5), "T": round(rng.uniform(200.0, 500.0), 1),
                "steps": 30}
    if kind == "muvt":
        n0 = rng.randint(5, 15)
        return {"kind": kind, "n0": n0, "gas": max(4, 4 * n0 ** 3 // rng.randint(40, 80)), "steps": 100,
                "nevery": rng.choice([25, 50]), "attempts": rng.randint(100, 500)}
    if kind == "min":
        return {"kind": kind, **_sides(rng, 4, 500, 1_100_000, 5), "steps": rng.randint(5, 12)}
    if kind == "dmd":
        fp32 = rng.random() < 0.5
        return {"kind": kind, **_sides(rng, 4, 500, 262_144 if fp32 else 65_536, 5), "nquad": rng.choice([3, 5]),
                "fp32": fp32}
    if kind == "newton":
        return {"kind": kind, **_sides(rng, 4, 500, 100_000, 5), "nquad": rng.choice([3, 5])}
    if kind == "gcmc":
        return {"kind": kind, "cells": round(math.exp(rng.uniform(math.log(64), math.log(4096)))),
                "attempts": rng.randint(16, 96)}
    return {"kind": kind, "cells": round(math.exp(rng.uniform(math.log(64), math.log(1024)))),
            "steps": rng.randint(8, 20)}


# ---------------- inputs ----------------

@functools.lru_cache(maxsize=None)
def _knots(name, nr):
    """the tables are files that a user's program reads: the same for every seed"""
    if name == "cu":
        return pot.johnson_cu(nr=nr, nrho=nr)
    if name == "feni":
        return pot.johnson_feni_fs(nr=nr, nrho=nr)
    return pot.johnson_cuh(nr=nr, nrho=nr, rc=5.5)


@functools.lru_cache(maxsize=None)
def _nih_cells(n):
    """boxes and lattice sites of a batch (108 to 4000 atoms a cell)"""
    return pot.gcmc_nih_cells(n, seed=6, jitter=0.0)


def _crystal(case, rng, sigma):
    """positions with a thermal jitter, box, elements and table of a crystal"""
    if case.get("alloy") == "feni":
        a, (x, H), p = A_FE, pot.bcc(A_FE, (case["n0"], case["n1"], case["n2"])), _knots("feni", 5000)
        elem = (rng.random(len(x)) < 0.2).astype(np.uint8)
    else:
        a, (x, H), p = A_CU, pot.fcc(A_CU, (case["n0"], case["n1"], case["n2"])), _knots("cu", case.get("nr", 10000))
        elem = np.zeros(len(x), np.uint8)
    x += 0.25 * a
    x += rng.normal(0.0, sigma, x.shape)
    return x, H, elem, p


def _velocities(elem, masses, T, rng):
    m = np.asarray(masses)[elem][:, None]
    v = rng.standard_normal((len(elem), 3))
    v *= np.sqrt(KB * T / m)
    v -= (m * v).sum(axis=0) / m.sum()
    return v


def _inputs(case, seed):
    """every array of a case, from the seed alone"""
    rng = np.random.default_rng(seed)
    kind = case["kind"]
    if kind in ("force", "nvt", "nst"):
        x, H, elem, p = _crystal(case, rng, 0.05)
        d = {"x": x, "H": H, "elem": elem, "p": p}
        if kind != "force":
            d["v"] = _velocities(elem, p.masses, case["T"], rng)
        return d
    if kind == "min":
        x, H, elem, p = _crystal(case, rng, 0.1)
        keep = np.ones(len(x), bool)
        keep[rng.choice(len(x), max(1, len(x) // 1000), replace=False)] = False
        return {"x": np.ascontiguousarray(x[keep]), "H": H, "elem": elem[keep], "p": p}
    if kind == "muvt":
        k = case["n0"]
        x, H = pot.fcc(A_NI, (k, k, k))
        cells = np.stack(np.meshgrid(*[np.arange(k)] * 3, indexing="ij"), -1).reshape(-1, 3) * A_NI
        h = cells[rng.choice(len(cells), min(case["gas"], len(cells)), replace=False)] + np.array([A_NI / 2, 0.0, 0.0])
        x = np.concatenate([x + rng.normal(0.0, 0.05, x.shape), h]) + 0.25 * A_NI
        elem = np.zeros(len(x), np.uint8)
        elem[len(x) - len(h):] = 2
        return {"x": x, "H": H, "elem": elem, "masses": _nih_masses(), "v": _velocities(elem, _nih_masses(), 300.0, rng)}
    if kind in ("dmd", "newton"):
        x, H, elem, alpha, c = pot.dmd_cuh_sites((case["n0"], case["n1"], case["n2"]), seed=seed)
        x = x + 0.25 * A_CU + rng.normal(0.0, 0.05, x.shape)
        return {"x": x, "H": H, "elem": elem, "alpha": alpha, "c": c, "p": _knots("cuh", 5000)}
    sigma = 0.03 if kind == "gcmc" else 0.1
    return {"cells": [(x + rng.normal(0.0, sigma, x.shape), H, e) for x, H, e in _nih_cells(case["cells"])]}


def _nih_masses():
    return [pot.MASS["Ni"], pot.MASS["Al"], pot.MASS["H"]]


def prepare(case, seed):
    d = _inputs(case, seed)
    s = {"case": dict(case)}
    kind = case["kind"]
    if kind in ("force", "nvt", "nst", "min"):
        s["md"] = M.AtomsMD(M.ForceFieldEAM.from_knots(d["p"]), d["H"], d["x"], d["elem"], skin=0.5)
        s["masses"] = d["p"].masses
        if kind in ("force", "min"):
            s["x"] = d["x"]
        else:
            s["md"].x_d = d["v"]
        if kind == "nvt":
            s["run"] = M.NVT(case["T"], pot.FS)
        elif kind == "nst":
            s["run"] = M.NST(np.zeros((3, 3)), case["T"], pot.FS)
        elif kind == "min":
            s["run"] = M.MinLBFGS(m=2, e_tol=0.0)
    elif kind == "muvt":
        s["md"] = M.AtomsMD(M.ForceFieldEAM.setfl(pot.NIALH_JEA), d["H"], d["x"], d["elem"], skin=0.5)
        s["md"].x_d = d["v"]
        s["masses"] = d["masses"]
        s["rows"] = len(d["x"]) + case["steps"] // case["nevery"] * case["attempts"]
        s["run"] = M.MuVT(-2.3, 300.0, pot.FS, 2, 1 + seed % 1_000_000, nevery=case["nevery"],
                          nattempts=case["attempts"])
    elif kind in ("dmd", "newton"):
        s["dmd"] = M.AtomsDMD(M.ForceFieldEAM.from_knots(d["p"], dmd=True), d["H"], d["x"], d["elem"], d["alpha"],
                              d["c"], nquad=case["nquad"], masses=d["p"].masses)
        if kind == "newton":
            s["state"] = (d["x"], d["alpha"], d["c"])
        elif case["fp32"]:
            s["dmd"].set_fp32(True)
    elif kind == "gcmc":
        s["batch"] = M.GCMCBatch(M.ForceFieldEAM.setfl(pot.NIALH_JEA), d["cells"], 2, -2.3, 300.0, _nih_masses(),
                                 1 + (seed % 1_000_000) + np.arange(case["cells"], dtype=np.int32))
        s["batch"].set_waves([4, 4, 4, 4, 4])
        s["batch"].use_graph(True)
    else:
        s["ff"] = M.ForceFieldEAM.setfl(pot.NIALH_JEA)
        s["cells"] = [(H, x, e) for x, H, e in d["cells"]]
    return s


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "force":
        md = s["md"]
        md.x = s["x"]
        md.update()
        f, e, FH = md.force_calc()
        return {"f": f, "e": e, "virial": FH}
    if kind in ("nvt", "nst", "muvt"):
        md, r = s["md"], s["run"]
        out = r.run(md, case["steps"], s["masses"])
        got = {"e": float(out[0]), "virial": out[1:], "T": r.T_part, "x": md.x, "v": md.x_d}
        if kind == "nst":
            got.update(H=md.H, hist=r.hist[:, :8])
        if kind == "muvt":
            # rows for every atom that the exchanges could have added, zero past the last
            rows = max(md.natms, s["rows"])
            for k in ("x", "v"):
                got[k] = np.concatenate([got[k], np.zeros((rows - md.natms, 3))])
            elem = np.concatenate([md.elem, np.zeros(rows - md.natms, np.uint8)])
            got.update(natms=md.natms, elem=elem, counts=r.counts, gas=r.hist[:, 1])
        return got
    if kind == "min":
        md = s["md"]
        md.x = s["x"]
        rep = s["run"].run(md, case["steps"])
        return {"e0": rep["e0"], "e": rep["e"], "steps": rep["steps"], "energies": s["run"].tally[:, 1], "x": md.x}
    if kind == "dmd":
        f, fa, mu, fe, FH, S = s["dmd"].derivative()
        return {"f": f, "f_alpha": fa, "mu": mu, "fe": float(fe), "virial": FH, "entropy": float(S)}
    if kind == "newton":
        d, (x, alpha, c) = s["dmd"], s["state"]
        d.set_state(x, alpha, c)
        ok, it = d.newton([3.5, 3.5], [1.7, 1.7], 30.0, -c / 30.0, a_tol=1e-8)
        return {"ok": int(ok), "iters": int(it), "c": d.state()[2]}
    if kind == "gcmc":
        dec, du = s["batch"].attempts(case["attempts"])
        n, gas = s["batch"].counts()
        return {"decisions": dec, "du": du, "natms": n, "gas": gas}
    rb = M.ReplicaBatch(s["ff"], s["cells"], skin=0.5)
    r = rb.min_cg(case["steps"], e_tol=0.0)
    return {"steps": r["steps"], "status": r["status"], "e0": r["e0"], "e": r["e"],
            "x": np.concatenate([rb.x(k) for k in range(len(rb))])}


# ---------------- work and tolerances ----------------

# A pair of a density or a force sum: separation, square, root, spline interval
# and offset, the cubics (one for the density; density slope, pair value and
# slope for the force) and the sums. Pairs are those within r_c.
FLOP_RHO, FLOP_FORCE = 25, 50


def _nih_atoms(cells):
    # sizes are log-uniform in [108, 4000] atoms
    return cells * (4000 - 108) / math.log(4000 / 108)


def work(case):
    kind = case["kind"]
    if kind in ("gcmc", "replica"):
        n = _nih_atoms(case["cells"])
        pairs = 58.0  # neighbours within r_c of an atom of the Ni-H table (5.0 to 5.4 A)
        if kind == "gcmc":
            # a trial sums the density and the pair energy over the neighbours of
            # the trial point, and the new embedding energies of those
            t = case["cells"] * case["attempts"]
            return {"bytes": n * 40 + t * 9, "flops": t * pairs * 2 * FLOP_RHO}
        # a step's force call and energies of about two trial points
        return {"bytes": n * 56, "flops": case["steps"] * n * pairs * (FLOP_RHO + FLOP_FORCE + 2 * 2 * FLOP_RHO)}
    per = 2 if case.get("alloy") == "feni" else 4
    n = per * case["n0"] * case.get("n1", case["n0"]) * case.get("n2", case["n0"])
    if kind in ("dmd", "newton"):
        # per pair of components and quadrature point: the spline interval, three
        # cubics and nine moments; both passes
        pairs = n * 78.0 / 2 * 4
        one = pairs * case["nquad"] * 60.0
        if kind == "dmd":
            return {"bytes": n * (24 + 16 + 16 + 24 + 16 + 16), "flops": one}
        # three Newton iterations: the rates, and about four products of the Jacobian
        return {"bytes": n * (24 + 16 * 4), "flops": 3 * (one + 4 * pairs * 12.0)}
    pairs = {"cu": 43.0, "feni": 53.0}["feni" if per == 2 else "cu"]
    if kind == "muvt":
        pairs = 58.0
    call = n * pairs * (FLOP_RHO + FLOP_FORCE)
    if kind == "force":
        return {"bytes": n * (24 + 24), "flops": call}
    if kind == "min":
        return {"bytes": case["steps"] * n * 48, "flops": case["steps"] * call}
    # a step reads and writes positions and velocities once
    return {"bytes": case["steps"] * n * 96, "flops": case["steps"] * (call + n * 40.0)}


def tolerance(case):
    kind = case["kind"]
    if kind in ("gcmc", "replica"):
        # FP64 throughout: sums in another order
        return {"rel": 1e-9, "max": 1e-6}
    if kind == "newton":
        return {"rel": 1e-8, "max": 1e-6}
    if kind == "dmd":
        # FP32 splines with FP64 sums, or FP64
        return {"rel": 1e-5, "max": 1e-3} if case["fp32"] else {"rel": 1e-10, "max": 1e-8}
    # forces are FP32 sums; runs carry them over the steps
    return {"rel": 1e-5, "max": 1e-3}


# ---------------- the same in 64 bits ----------------

def _spline(y, quartic=False):
    """coefficients of the knots' cubics: Hermite with five-point slopes (and the
    term of fourth order that the DMD embedding function adds)"""
    y = np.asarray(y, dtype=np.float64)
    n = len(y)
    s = np.zeros(n)
    s[0], s[1], s[n - 2], s[n - 1] = y[1] - y[0], 0.5 * (y[2] - y[0]), 0.5 * (y[-1] - y[-3]), y[-1] - y[-2]
    s[2:n - 2] = ((y[:-4] - y[4:]) + 8.0 * (y[3:-1] - y[1:-3])) / 12.0
    dy = np.append(y[1:] - y[:-1], 0.0)
    s1 = np.append(s[1:], 0.0)
    c = np.stack([y, s, 3.0 * dy - 2.0 * s - s1, s + s1 - 2.0 * dy], axis=1)
    c[n - 1, 2:] = 0.0
    if quartic:
        q = np.zeros(n)
        q[:-1] = (c[1:, 2] - c[:-1, 2]) / 6.0 - 0.5 * c[:-1, 3]
        c = np.concatenate([c, q[:, None]], axis=1)
    return torch.from_numpy(c)


def _dev():
    return "cuda" if torch.cuda.is_available() else "cpu"


def _cut(p, a, b):
    nz = (p.r_phi[a, b] != 0) | (p.rho[a, b] != 0) | (p.rho[b, a] != 0)
    return int(np.nonzero(nz)[0].max()) * p.dr


def _pairs(x, L, rc):
    """(i, j, image) of every ordered pair within rc in an orthogonal box"""
    dev, n = x.device, len(x)
    nc = torch.clamp((L / rc).floor().long(), min=1)
    ci = torch.minimum((x / L * nc).floor().long() % nc, nc - 1)
    wrap = (x / L).floor()
    cid = ci[:, 0] + nc[0] * (ci[:, 1] + nc[1] * ci[:, 2])
    order = torch.argsort(cid)
    cs = torch.searchsorted(cid[order], torch.arange(int(nc.prod()) + 1, device=dev))
    cap = int((cs[1:] - cs[:-1]).max())
    out = []
    ar = torch.arange(cap, device=dev)
    step = max(1, 60_000_000 // (27 * cap))
    offs = torch.tensor([(a, b, c) for a in (-1, 0, 1) for b in (-1, 0, 1) for c in (-1, 0, 1)], device=dev)
    for i0 in range(0, n, step):
        i = torch.arange(i0, min(n, i0 + step), device=dev)
        c = ci[i][:, None, :] + offs[None]
        img = torch.div(c, nc, rounding_mode="floor")
        c = c - img * nc
        c = c[..., 0] + nc[0] * (c[..., 1] + nc[1] * c[..., 2])
        k = cs[c][..., None] + ar
        ok = k < cs[c + 1][..., None]
        a, o, _ = ok.nonzero(as_tuple=True)
        j = order[k[ok]]
        g = img[a, o].double() - wrap[j] + wrap[i[a]]
        a = i[a]
        d = x[a] - x[j] - g * L
        near = (d * d).sum(1) < rc * rc
        near &= ~((a == j) & (g == 0).all(1))
        out.append((a[near].int(), j[near].int(), g[near].to(torch.int8)))
    return [torch.cat([o[k] for o in out]) for k in range(3)]


def _at(v, inv, n):
    pm = v * inv
    m = torch.clamp(pm.long(), 0, n - 2)
    return m, torch.clamp(pm - m, max=1.0)


def _val(c, p):
    return ((c[..., 3] * p + c[..., 2]) * p + c[..., 1]) * p + c[..., 0]


def _der(c, p):
    return (3.0 * c[..., 3] * p + 2.0 * c[..., 2]) * p + c[..., 1]


class _Eam:
    """energy, forces and virial of the tables in 64 bits"""

    def __init__(self, p, elem, L):
        ne, dev = p.ne, _dev()
        self.p, self.L = p, torch.tensor(L, device=dev)
        self.e = torch.from_numpy(elem.astype(np.int64)).to(dev)
        self.rho = torch.stack([_spline(p.rho[a, b if p.fs else 0]) for a in range(ne) for b in range(ne)]).to(dev)
        self.phi = torch.stack([_spline(p.r_phi[max(a, b), min(a, b)]) for a in range(ne) for b in range(ne)]).to(dev)
        self.F = torch.stack([_spline(p.F[a]) for a in range(ne)]).to(dev)
        self.rc2 = torch.tensor([[_cut(p, a, b) ** 2 for b in range(ne)] for a in range(ne)], device=dev)
        self.list = None

    def __call__(self, x):
        p, n, dev = self.p, len(x), x.device
        if self.list is None or float((x - self.x0).square().sum(1).max()) > 0.2 ** 2:
            self.x0 = x.clone()
            self.list = _pairs(x, self.L, float(self.rc2.max()) ** 0.5 + 0.4)
        li, lj, lg = self.list
        dens = torch.zeros(n, dtype=torch.float64, device=dev)
        f = torch.zeros(n, 3, dtype=torch.float64, device=dev)
        e, vir = 0.0, torch.zeros(3, 3, dtype=torch.float64, device=dev)
        dF = None
        for second in (False, True):
            for k in range(0, len(li), 8_000_000):
                i, j = li[k:k + 8_000_000].long(), lj[k:k + 8_000_000].long()
                d = x[i] - x[j] - lg[k:k + 8_000_000].double() * self.L
                r2 = (d * d).sum(1)
                ei, ej = self.e[i], self.e[j]
                near = r2 < self.rc2[ei, ej]
                i, j, d, r2, ei, ej = i[near], j[near], d[near], r2[near], ei[near], ej[near]
                r = r2.sqrt()
                m, q = _at(r, 1.0 / p.dr, p.nr)
                ct = self.rho[ej * p.ne + ei, m]
                if not second:
                    dens.index_add_(0, i, _val(ct, q))
                    continue
                cz = self.phi[ei * p.ne + ej, m]
                phi = _val(cz, q) / r
                dphi = (_der(cz, q) / p.dr - phi) / r
                co = self.rho[ei * p.ne + ej, m]
                u = -(dphi + (dF[i] * _der(ct, q) + dF[j] * _der(co, q)) / p.dr) / r
                f.index_add_(0, i, u[:, None] * d)
                e = e + 0.5 * phi.sum()
                vir += 0.5 * (u[:, None] * d).T @ d
            if not second:
                m, q = _at(dens, 1.0 / p.drho, p.nrho)
                c = self.F[self.e, m]
                dF = _der(c, q) / p.drho
                e = (_val(c, q) + torch.clamp(dens - p.nrho * p.drho, min=0.0) * dF).sum()
        return f, e, torch.stack([vir[0, 0], vir[0, 1], vir[0, 2], vir[1, 1], vir[1, 2], vir[2, 2]])


def _chain(eta, T_r, ddt, freq2, ndof):
    """a half step of the three-link Nose-Hoover chain; returns the velocity scale"""
    def phi(x):
        return 1.0 + x / 2.0 + x * x / 6.0 + x ** 3 / 24.0 if abs(x) < 0.015625 else math.expm1(x) / x

    h = 0.5 * ddt
    eta[2] += h * (eta[1] ** 2 - freq2)
    eta[1] += h * phi(-eta[2] * h) * (-eta[2] * eta[1] + eta[0] ** 2 - freq2)
    eta[0] += h * phi(-eta[1] * h) * (-eta[1] * eta[0] + freq2 * (T_r - 1.0))
    s = math.exp(-ddt * eta[0])
    T_r *= s * s
    eta[0] += h * phi(-eta[1] * h) * (-eta[1] * eta[0] + (T_r - 1.0) * freq2)
    eta[1] += h * phi(-eta[2] * h) * (-eta[2] * eta[1] + ndof * eta[0] ** 2 - freq2)
    eta[2] += h * (eta[1] ** 2 - freq2)
    return s


def _exact_nvt(case, d):
    dev, dt, n = _dev(), pot.FS, len(d["x"])
    x, v = torch.from_numpy(d["x"]).to(dev), torch.from_numpy(d["v"]).to(dev)
    ff = _Eam(d["p"], d["elem"], np.diag(d["H"]).copy())
    m = torch.from_numpy(np.asarray(d["p"].masses)).to(dev)[ff.e][:, None]
    f, e, vir = ff(x)
    eta, fac, freq2 = [0.0, 0.0, 0.0], 1.0, 1.0 / (100.0 * dt) ** 2
    T = float((m * v * v).sum()) / (3 * n * KB)
    for _ in range(case["steps"]):
        s = _chain(eta, T / case["T"], 0.5 * dt, freq2, 3 * n)
        v = v * (fac * s) + f * (0.5 * dt) / m
        x = x + v * dt
        x = x - (v * dt).mean(0)
        f, e, vir = ff(x)
        v = v + f * (0.5 * dt) / m
        T = float((m * v * v).sum()) / (3 * n * KB)
        fac = _chain(eta, T / case["T"], 0.5 * dt, freq2, 3 * n)
        T *= fac * fac
    return {"e": float(e), "virial": vir, "T": T, "x": x, "v": v * fac}


def _exact_dmd(case, d):
    """free energy and gradient of the smeared pair functions (d/dr and d/dalpha
    of the smeared integral, by the moments of the rule)"""
    p, dev, n = d["p"], _dev(), len(d["x"])
    xi, wi = np.polynomial.hermite.hermgauss(case["nquad"])
    L = torch.tensor(np.diag(d["H"]).copy(), device=dev)
    x, al, c = (torch.from_numpy(d[k]).to(dev) for k in ("x", "alpha", "c"))
    kT = KB * 300.0
    r = np.arange(p.nr) * p.dr
    rho = [_spline(r * p.rho[a, 0]).to(dev) for a in range(2)]
    phi = [[_spline(p.r_phi[max(a, b), min(a, b)]).to(dev) for b in range(2)] for a in range(2)]
    F = [_spline(p.F[a], quartic=True).to(dev) for a in range(2)]
    lam = [pot.HP / math.sqrt(2.0 * math.pi * kT * m) for m in p.masses]
    mu0 = torch.tensor([kT * 1.5 * (2.0 * math.log(v) - 1.0 - math.log(math.pi)) for v in lam], device=dev)
    li, lj, lg = _pairs(x, L, max(_cut(p, 0, 0), _cut(p, 0, 1), _cut(p, 1, 1)) + xi[-1] * math.sqrt(2.0) * 0.3)
    dens = torch.zeros(n, 2, dtype=torch.float64, device=dev)
    f = torch.zeros(n, 3, dtype=torch.float64, device=dev)
    fa, mu = torch.zeros_like(dens), torch.zeros_like(dens)
    vir = torch.zeros(3, 3, dtype=torch.float64, device=dev)
    pi2 = 1.0 / math.sqrt(math.pi)
    fe, dE = 0.0, None
    for second in (False, True):
        for k in range(0, len(li), 4_000_000):
            si, sj = li[k:k + 4_000_000].long(), lj[k:k + 4_000_000].long()
            sd = x[si] - x[sj] - lg[k:k + 4_000_000].double() * L
            sr = sd.square().sum(1).sqrt()
            for a in range(2):
                for b in range(2):
                    q = (al[si, a] ** 2 + al[sj, b] ** 2).sqrt()
                    near = sr - q * xi[-1] < _cut(p, a, b)
                    i, j, dx, rr, w = si[near], sj[near], sd[near], sr[near], q[near]
                    mom = torch.zeros(3, 3, len(i), dtype=torch.float64, device=dev)
                    for xl, wl in zip(xi, wi):
                        u = rr - xl * w
                        m, o = _at(u.abs(), 1.0 / p.dr, p.nr)
                        for t, tab in enumerate((phi[a][b], rho[a], rho[b])):
                            y = _val(tab[m], o) * torch.sign(u) * wl
                            mom[t, 0] += y
                            mom[t, 1] += y * xl
                            mom[t, 2] += y * xl * xl
                    g = pi2 * mom[:, 0] / rr
                    if not second:
                        dens[:, a].index_add_(0, i, c[j, b] * g[2])
                        fe = fe + 0.5 * (c[i, a] * c[j, b] * g[0]).sum()
                        continue
                    gr = -(g + 2.0 * pi2 * mom[:, 1] / w) / rr ** 2
                    ga = -(g - 2.0 * pi2 * mom[:, 2] / rr) / w ** 2
                    cc = c[i, a] * c[j, b]
                    fp = -(gr[2] * dE[i, a] + gr[1] * dE[j, b] + gr[0]) * cc
                    ap = -(ga[2] * dE[i, a] + ga[1] * dE[j, b] + ga[0]) * cc
                    f.index_add_(0, i, fp[:, None] * dx)
                    vir += 0.5 * (fp[:, None] * dx).T @ dx
                    fa[:, a].index_add_(0, i, al[i, a] * ap)
                    mu[:, a].index_add_(0, i, c[j, b] * (g[0] + g[1] * dE[j, b]))
        if not second:
            dE = torch.zeros_like(dens)
            for a in range(2):
                m, o = _at(dens[:, a], 1.0 / p.drho, p.nrho)
                t = F[a][m]
                dE[:, a] = (((4.0 * t[:, 4] * o + 3.0 * t[:, 3]) * o + 2.0 * t[:, 2]) * o + t[:, 1]) / p.drho
                E = (((t[:, 4] * o + t[:, 3]) * o + t[:, 2]) * o + t[:, 1]) * o + t[:, 0]
                E = E + torch.clamp(dens[:, a] - p.nrho * p.drho, min=0.0) * dE[:, a]
                mu[:, a] += E
                fe = fe + (c[:, a] * (E + mu0[a] - 3.0 * kT * al[:, a].log())).sum()
    fa += 3.0 * kT * c / al
    cv = 1.0 - c.sum(1)
    S = float((torch.xlogy(c, c)).sum() + torch.xlogy(cv, cv).sum())
    vir = torch.stack([vir[0, 0], vir[0, 1], vir[0, 2], vir[1, 1], vir[1, 2], vir[2, 2]])
    return {"f": f, "f_alpha": fa, "mu": mu, "fe": float(fe) + kT * S, "virial": vir, "entropy": S}


def exact(case, seed):
    """forces, runs at constant temperature up to a million atoms or so, and the
    DMD gradient; the other kinds return where a chain of decisions (exchanges,
    line searches, iterations) has led, which has no closed value"""
    kind = case["kind"]
    if kind == "force":
        d = _inputs(case, seed)
        f, e, vir = _Eam(d["p"], d["elem"], np.diag(d["H"]).copy())(torch.from_numpy(d["x"]).to(_dev()))
        return {"f": f, "e": float(e), "virial": vir}
    if kind == "nvt":
        d_atoms = case["n0"] * case["n1"] * case["n2"] * (2 if case["alloy"] == "feni" else 4)
        if d_atoms * case["steps"] > 120_000_000:
            return None
        return _exact_nvt(case, _inputs(case, seed))
    if kind == "dmd":
        return _exact_dmd(case, _inputs(case, seed))
    return None
