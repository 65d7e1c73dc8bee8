"""The EAM passes that hold splines in LDS, of one element (k_eam_*_lds) and of
several (k_eam_*_alloy), against the oracle and against the passes over the
global tables, which read the same splines: single calls for every table layout
and mix of elements, and runs, whose passes sum no energies, carry the second
half of the kick and are launched ahead of the skin check. Bars as in
test_gpu_eam.py.
"""
import numpy as np
import pytest

import oracle_lib as O
from mapp4py_amd import potentials as pot
from test_gpu_eam import E_ATOM, F_TOL, M, both, jitter, say, triples  # noqa: F401

pytestmark = pytest.mark.gpu

NIH = [pot.MASS["Ni"], pot.MASS["Al"], pot.MASS["H"]]


def four(fs, nr=5000):
    """four elements, each pair with functions of its own"""
    a = pot.johnson_feni_fs(nr=nr, nrho=nr)
    rho, F, z = np.zeros((4, 4, nr)), np.zeros((4, nr)), np.zeros((4, 4, nr))
    for i in range(4):
        F[i] = a.F[i % 2]
        for j in range(4):
            rho[i, j] = a.rho[i % 2, j % 2 if fs else 0] * (1 + 0.03 * i + (0.02 * j if fs else 0))
        for j in range(i + 1):
            z[i, j] = z[j, i] = a.r_phi[max(i % 2, j % 2), min(i % 2, j % 2)] * (1 + 0.01 * (i + j))
    return pot.EamKnots(["A", "B", "C", "D"], [50.0, 52.0, 55.0, 58.0], nr, a.dr, nr, a.drho, F, rho, z, fs)


def system(kind, cells, shares, tilt=(0.0, 0.0, 0.0)):
    """force fields, box, positions and elements; shares: of each element, a
    negative one a number of atoms"""
    if kind == "nih":
        ff, of, (x, H) = None, O.OEam.read(pot.NIALH_JEA), pot.fcc(3.52, cells)
    else:
        p = {"feni": pot.johnson_feni_fs, "feni_fine": lambda: pot.johnson_feni_fs(nr=10000, nrho=5000),
             "four_fs": lambda: four(True), "four_alloy": lambda: four(False)}[kind]()
        ff, of, (x, H) = p, O.OEam.from_knots(p), pot.bcc(2.86, cells)
    rng = np.random.default_rng(len(x))
    H = H.copy()
    H[1, 0], H[2, 0], H[2, 1] = tilt
    x = jitter(x, 0.05, 7)
    n = len(x)
    frac = np.array([max(s, 0.0) for s in shares])
    elem = rng.choice(len(shares), n, p=frac / frac.sum()).astype(np.uint8)
    for e, s in enumerate(shares):
        if s < 0:
            elem[rng.choice(n, int(-s), replace=False)] = e
    import mapp4py_amd

    gff = mapp4py_amd.ForceFieldEAM.setfl(pot.NIALH_JEA) if ff is None else mapp4py_amd.ForceFieldEAM.from_knots(ff)
    masses = NIH if ff is None else ff.masses
    return gff, of, H, x, elem, masses


@pytest.mark.parametrize("kind,cells,shares,tilt,below", [
    ("feni", (9, 10, 8), (0.8, 0.2), (0.4, -0.3, 0.5), False),
    ("nih", (6, 7, 6), (0.7, 0.2, 0.1), (0.0, 0.0, 0.0), False),     # three elements, one density each
    ("nih", (6, 6, 8), (1.0, -1, 0.0), (0.5, 0.2, -0.4), False),     # one atom of an element, none of another
    ("nih", (6, 7, 6), (0.0, 0.0, 1.0), (0.0, 0.0, 0.0), False),     # atoms of the last element only
    # the first shell (2.48 A) below both windows, read from the global rows
    ("feni_fine", (9, 9, 9), (0.5, 0.5), (0.0, 0.0, 0.0), True),
    ("four_fs", (9, 8, 9), (0.4, 0.3, 0.2, 0.1), (0.0, 0.3, 0.0), True),
    ("four_alloy", (9, 8, 9), (0.4, 0.0, 0.5, -3), (0.0, 0.0, 0.0), True),
    ("nih", (24, 24, 24), (0.75, 0.22, 0.03), (0.0, 0.0, 0.0), False),  # 55,296 atoms: LDS by their number
])
def test_passes_of_several_elements_give_the_oracle_forces(M, kind, cells, shares, tilt, below):
    ff, of, H, x, elem, _ = system(kind, cells, shares, tilt)
    g = M.AtomsMD(ff, H, x, elem, skin=0.5)
    o = O.OMD(of, H, x, elem, skin=0.5)
    fo, eo, FHo, rho_o = o.force()
    n, out = len(x), {}
    pairs = triples(*o.pairs()) if n < 10000 else None
    lo = np.array(g.lds_window()) * of.dr
    say(f"{kind} {n} atoms, elements {np.bincount(elem)}: windows from r = {lo[0]:.2f} and {lo[1]:.2f} A")
    assert below == bool((lo > 2.48).all()) and (lo >= 0).all()
    for lds in ((None, False) if n >= 49152 else (True, False, True)):
        if lds is not None:
            assert g.set_lds(lds) == lds
        f, e, FH = g.force_calc()
        df = np.abs(f - fo).max()
        say(f"  lds={lds}: max|df|={df:.2e} eV/A  |dE|/N={abs(e - eo) / n:.2e} eV  "
            f"max|dF_H|/N={np.abs(FH - FHo).max() / n:.2e} eV")
        assert df < F_TOL
        assert abs(e - eo) < E_ATOM * n + 1e-6
        assert np.abs(FH - FHo).max() < 2e-7 * n + 5e-6
        np.testing.assert_allclose(g.rho(), rho_o, rtol=2e-7)
        assert abs(g.value() - e) < 1e-12 * abs(e)
        if pairs is not None:
            assert triples(*g.half_pairs()) == pairs
        out[bool(lds) or lds is None] = f
    assert np.abs(out[True] - out[False]).max() < F_TOL


def test_alloy_forces_are_no_further_off_than_from_the_global_rows(M):
    # FP32 knots against FP32 rows of the same splines, over 10,000 forces:
    # the knots' derivative errors are 0.91 of the rows'
    ff, of, H, x, elem, _ = system("feni", (12, 12, 13), (0.8, 0.2))
    g = M.AtomsMD(ff, H, x, elem, skin=0.5)
    fo = O.OMD(of, H, x, elem, skin=0.5).force()[0]
    rms = {}
    for lds in (True, False):
        g.set_lds(lds)
        rms[lds] = np.sqrt(np.mean((g.force_calc()[0] - fo) ** 2))
    say(f"rms force error: knots {rms[True]:.3e}, rows {rms[False]:.3e} eV/A")
    assert rms[True] < rms[False]


@pytest.mark.parametrize("kind", ["cu", "feni", "nih"])
@pytest.mark.parametrize("lds", [True, False])
def test_run_matches_the_oracle_with_and_without_lds(M, kind, lds):
    # 40 steps at 900 K: the list is rebuilt within groups of steps that were
    # launched ahead
    if kind == "cu":
        p = pot.johnson_cu(nr=5000, nrho=5000)
        x, H = pot.fcc(3.615, (6, 6, 7))
        ff, of, x, elem, masses = (M.ForceFieldEAM.from_knots(p), O.OEam.from_knots(p), jitter(x, 0.05, 3),
                                   np.zeros(4 * 252, np.uint8), p.masses)
    else:
        ff, of, H, x, elem, masses = system(kind, (8, 9, 8) if kind == "feni" else (6, 6, 7),
                                            (0.8, 0.2) if kind == "feni" else (0.8, 0.2, 0.0))
    v = O.o_create_T(elem, masses, pot.KB_EV, 900.0, 3)
    g = M.AtomsMD(ff, H, x, elem, skin=0.3)
    o = O.OMD(of, H, x, elem, skin=0.3)
    assert g.set_lds(lds) == lds
    g.x_d = v
    nvt = M.NVT(900.0, 1.0 * pot.FS)
    out = nvt.run(g, 40, masses)
    vo, outo, Tpo, nreb_o = o.nvt_run(v, masses, pot.KB_EV, 900.0, 1.0 * pot.FS, 40)
    dx, dv = np.abs(g.x - o.x).max(), np.abs(g.x_d - vo).max()
    say(f"{kind} lds={lds}: max|dx|={dx:.2e} A max|dv|={dv:.2e} T {nvt.T_part:.6f} vs {Tpo:.6f} "
        f"rebuilds {nvt.rebuilds} vs {nreb_o}")
    assert nvt.rebuilds == nreb_o and nreb_o >= 1
    assert dx < 1e-6 and dv < 1e-6
    assert abs(nvt.T_part - Tpo) < 1e-6 * Tpo
    assert abs(out[0] - outo[0]) < E_ATOM * len(x) + 1e-6


@pytest.mark.parametrize("kind,cells", [("cu", (15, 15, 16)), ("cu", (27, 28, 29)), ("cu", (52, 51, 50)),
                                        ("feni", (29, 30, 31)), ("feni", (52, 51, 50)), ("nih", (24, 23, 25))])
def test_run_with_lds_is_the_run_without(M, kind, cells):
    # the sizes at which the passes split an atom over 16 to 1 lanes and an
    # element's atoms over its workgroups, against the global tables
    if kind == "cu":
        p = pot.johnson_cu(nr=5000, nrho=5000)
        x, H = pot.fcc(3.615, cells)
        ff, x, elem, masses = M.ForceFieldEAM.from_knots(p), jitter(x, 0.05, 3), np.zeros(len(x), np.uint8), p.masses
    else:
        ff, _, H, x, elem, masses = system(kind, cells, (0.8, 0.2) if kind == "feni" else (0.79, 0.2, -5))
    rng = np.random.default_rng(1)
    m = np.asarray(masses)[elem][:, None]
    v = rng.standard_normal(x.shape) * np.sqrt(pot.KB_EV * 700.0 / m)
    got = []
    for lds in (None, False):
        g = M.AtomsMD(ff, H, x, elem, skin=0.3)
        if lds is not None:
            assert not g.set_lds(lds)
        g.x_d = v
        nvt = M.NVT(700.0, 1.0 * pot.FS)
        out = nvt.run(g, 30, masses)
        got.append((g.x, g.x_d, nvt.T_part, nvt.rebuilds, out))
    (xa, va, Ta, ra, oa), (xb, vb, Tb, rb, ob) = got
    say(f"{kind} {len(x)} atoms: max|dx|={np.abs(xa - xb).max():.2e} max|dv|={np.abs(va - vb).max():.2e} rebuilds {ra}")
    assert ra == rb and ra >= 1
    assert np.abs(xa - xb).max() < 1e-6 and np.abs(va - vb).max() < 1e-6
    assert abs(Ta - Tb) < 1e-7 * Tb and abs(oa[0] - ob[0]) < E_ATOM * len(x)


def test_exchanges_follow_the_element_counts(M):
    # the alloy passes on a system whose gas atoms come and go: the same chain,
    # and the forces of a system made of the final atoms
    x, H = pot.fcc(3.52, (6, 6, 6))
    h = x[::9] + np.array([1.76, 0.0, 0.0])
    x = np.concatenate([jitter(x, 0.03, 2), h])
    elem = np.zeros(len(x), np.uint8)
    elem[len(x) - len(h):] = 2
    v = O.o_create_T(elem, NIH, pot.KB_EV, 300.0, 5)
    got = []
    for lds in (True, False):
        g = M.AtomsMD(M.ForceFieldEAM.setfl(pot.NIALH_JEA), H, x, elem, skin=0.5)
        assert g.set_lds(lds) == lds
        g.x_d = v
        run = M.MuVT(-2.2, 300.0, 0.5 * pot.FS, 2, 77, nevery=5, nattempts=60)
        run.run(g, 20, NIH)
        assert g.set_lds(lds) == lds
        f = g.force_calc()[0]
        fresh = M.AtomsMD(M.ForceFieldEAM.setfl(pot.NIALH_JEA), H, g.x, g.elem, skin=0.5)
        assert np.abs(f - fresh.force_calc()[0]).max() < F_TOL
        got.append((g.elem, run.counts, g.x))
    (ea, ca, xa), (eb, cb, xb) = got
    say(f"exchange counts {ca}, {len(ea)} atoms of {len(x)}")
    assert np.array_equal(ea, eb) and np.array_equal(ca, cb) and len(ea) != len(x)
    assert np.abs(xa - xb).max() < 1e-6


def test_barostat_and_minimiser_on_the_alloy_passes(M):
    ff, _, H, x, elem, masses = system("feni", (8, 9, 8), (0.8, 0.2))
    v = O.o_create_T(elem, masses, pot.KB_EV, 600.0, 3)
    S = np.zeros((3, 3))
    got = []
    for lds in (True, False):
        g = M.AtomsMD(ff, H, x, elem, skin=0.3)
        assert g.set_lds(lds) == lds
        g.x_d = v
        nst = M.NST(S, 600.0, 1.0 * pot.FS, tau=np.full((3, 3), 60.0 * pot.FS))
        nst.run(g, 30, masses)
        m = M.AtomsMD(ff, H, x, elem, skin=0.3)
        assert m.set_lds(lds) == lds
        r = M.MinLBFGS(m=2, e_tol=0.0).run(m, 6)
        got.append((g.x, g.H, nst.rebuilds, m.x, r["e"], r["steps"]))
    (xa, Ha, ra, ma, ea, sa), (xb, Hb, rb, mb, eb, sb) = got
    say(f"NST: max|dx| {np.abs(xa - xb).max():.1e}, max|dH| {np.abs(Ha - Hb).max():.1e}, rebuilds {ra}; "
        f"L-BFGS: {sa} steps, max|dx| {np.abs(ma - mb).max():.1e}, dE {abs(ea - eb):.1e}")
    assert ra == rb and np.abs(xa - xb).max() < 1e-6 and np.abs(Ha - Hb).max() < 1e-6
    assert sa == sb and np.abs(ma - mb).max() < 1e-5 and abs(ea - eb) < E_ATOM * len(x) + 1e-6


@pytest.mark.parametrize("kind", ["cu", "feni"])
def test_profiled_runs_time_every_pass_once(M, kind):
    # with the kernels timed a run counts one pass a step and the first, none
    # for the steps that find the list due, and takes the steps of one untimed
    if kind == "cu":
        p = pot.johnson_cu(nr=5000, nrho=5000)
        x, H = pot.fcc(3.615, (6, 6, 7))
        ff, x, elem, masses = M.ForceFieldEAM.from_knots(p), jitter(x, 0.05, 3), np.zeros(len(x), np.uint8), p.masses
    else:
        ff, _, H, x, elem, masses = system("feni", (8, 9, 8), (0.8, 0.2))
    v = O.o_create_T(elem, masses, pot.KB_EV, 900.0, 3)
    for run in (M.NVT(900.0, pot.FS), M.NST(np.zeros((3, 3)), 900.0, pot.FS)):
        got = []
        for timed in (True, False):
            g = M.AtomsMD(ff, H, x, elem, skin=0.3)
            g.set_lds(True)
            g.x_d = v
            g.profile(timed)
            run.run(g, 40, masses)
            if timed:
                counts = {k: g.profile_read(k)[1] for k in ("eam_rho", "eam_force", "build_list")}
            got.append((g.x, g.x_d, run.T_part, run.rebuilds))
        (xa, va, Ta, ra), (xb, vb, Tb, rb) = got
        say(f"{kind} {type(run).__name__}: launches {counts}, {ra} rebuilds")
        assert ra == rb and ra >= 1
        assert counts["eam_rho"] == counts["eam_force"] == 41 and counts["build_list"] == ra
        assert np.array_equal(xa, xb) and np.array_equal(va, vb) and Ta == Tb
