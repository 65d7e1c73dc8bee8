"""NST on the GPU (mapp_md_nst_run) against the oracle's restatement of
MDNST::run (src/md_nst.cpp:376-460): the same box, stress, temperature and
energy history step by step, the same rebuild count, and box, positions and
velocities within the FP32-force bar of the NVT parity tests (1e-6) after
200 steps in which every box component moves."""
import sys

import numpy as np
import pytest

import oracle_lib as O
from mapp4py_amd import potentials as pot

pytestmark = pytest.mark.gpu


def say(msg):
    print(msg, flush=True)
    sys.stdout.flush()


@pytest.fixture(scope="module")
def M():
    import mapp4py_amd

    return mapp4py_amd


def setup(M, cells, seed, T):
    p = pot.johnson_cu(nr=5000, nrho=5000)
    x, H = pot.fcc(3.615, (cells,) * 3)
    x = x + np.random.default_rng(seed).normal(0, 0.03, x.shape)
    elem = np.zeros(len(x), np.uint8)
    masses = [pot.MASS["Cu"]]
    v = O.o_create_T(elem, masses, pot.KB_EV, T, seed + 1)
    g = M.AtomsMD(M.ForceFieldEAM.from_knots(p), H, x, elem)
    g.x_d = v
    o = O.OMD(O.OEam.from_knots(p), H, x, elem)
    return p, H, g, o, v, masses


@pytest.mark.parametrize("full", [False, True])
def test_nst_matches_the_oracle(M, full):
    T, dt, nsteps = 600.0, 2.0 * pot.FS, 200
    p, H, g, o, v, masses = setup(M, 6, 7, T)
    S = np.full((3, 3), np.nan)
    np.fill_diagonal(S, [0.01, -0.005, 0.0])
    if full:
        S[1, 0], S[2, 0], S[2, 1] = 0.004, -0.003, 0.002
    tau = np.full((3, 3), 60.0 * pot.FS)
    say(f"NST {'all six components' if full else 'diagonal'}: {len(v)} Cu atoms, {nsteps} steps at {T} K")
    nst = M.NST(S, T, dt, kB=pot.KB_EV, tau=tau)
    out = nst.run(g, nsteps, masses)
    vo, Ho, Tpo, outo, histo, nro = o.nst_run(v, masses, pot.KB_EV, T, dt, S, nsteps, tau=tau)
    hg = nst.hist
    dH = np.abs(g.H - Ho).max()
    dx = np.abs(g.x - o.x).max()
    dv = np.abs(g.x_d - vo).max()
    strain = np.abs(Ho - H).max()
    say(f"  box moved {strain:.3f} A; max|dH| {dH:.2e} A, max|dx| {dx:.2e} A, max|dv| {dv:.2e}, "
        f"T {nst.T_part:.6f} vs {Tpo:.6f}, rebuilds {nst.rebuilds} vs {nro}")
    assert nro >= 1 and nst.rebuilds == nro
    assert strain > 0.05
    if full:
        assert min(abs(Ho[1, 0]), abs(Ho[2, 0]), abs(Ho[2, 1])) > 1e-3
    # the bar of the NVT parity tests (1e-6 A, 1e-6 A/time) for positions,
    # velocities and the box edges alike
    assert dH < 1e-6 and dx < 1e-6 and dv < 1e-6
    assert abs(nst.T_part - Tpo) < 1e-6 * Tpo
    n = len(v)
    np.testing.assert_allclose(hg[:, 2:8], histo[:, 2:8], rtol=0, atol=1e-6)
    np.testing.assert_allclose(hg[:, 0], histo[:, 0], rtol=1e-6)
    np.testing.assert_allclose(hg[:, 1], histo[:, 1], rtol=0, atol=5e-8 * n + 1e-6)
    # stress from FP32 pair forces summed in FP64: the single-call virial bar
    # per atom / volume after the first step; over the run the trajectories'
    # separation (dx above) adds to it, held to 1e-6 of the largest stress
    vol = histo[:, 2] * histo[:, 4] * histo[:, 7]
    assert np.abs(hg[0, 8:] - histo[0, 8:]).max() < (2e-7 * n + 5e-6) / vol[0]
    assert np.abs(hg[:, 8:] - histo[:, 8:]).max() < 1e-6 * np.abs(histo[:, 8:]).max()


def test_immobile_box_gives_the_gpu_nvt_trajectory(M):
    T, dt, nsteps = 300.0, 1.0 * pot.FS, 80
    p, H, g, o, v, masses = setup(M, 5, 3, T)
    S = np.full((3, 3), np.nan)
    np.fill_diagonal(S, 0.0)
    nst = M.NST(S, T, dt, kB=pot.KB_EV, tau=np.full((3, 3), 1e12))
    nst.run(g, nsteps, masses)
    g2 = M.AtomsMD(M.ForceFieldEAM.from_knots(p), H, o.x, np.zeros(len(v), np.uint8))
    g2.x_d = v
    nvt = M.NVT(T, dt, kB=pot.KB_EV)
    nvt.run(g2, nsteps, masses)
    say(f"NST with an immobile box vs NVT, {nsteps} steps: max|dx| {np.abs(g.x - g2.x).max():.2e} A")
    np.testing.assert_allclose(g.H, H, rtol=0, atol=1e-12)
    assert np.abs(g.x - g2.x).max() < 1e-9 and np.abs(g.x_d - g2.x_d).max() < 1e-9
    assert abs(nst.T_part - nvt.T_part) < 1e-9 * nvt.T_part


@pytest.mark.parametrize("cells,nreset", [(2, 3), (14, 0), (15, 4)])
def test_step_ends_for_every_way_to_sum_the_rows(M, cells, nreset):
    # 32 atoms; 10,976 (global tables, more rows of energies than the step's
    # end adds up itself); 13,500 (splines in LDS). The virial bar of a single
    # call, 2e-7 eV an atom from FP32 pair forces, moves a box edge of H by up
    # to H (N dt / tau)^2 / 2 times 2e-7 / (3 kB T): 7e-6 A at H = 54 A over 10
    # steps; held to the 1e-6 A of the longer runs
    T, dt, nsteps = 300.0, 2.0 * pot.FS, 10
    p, H, g, o, v, masses = setup(M, cells, 5, T)
    S = np.full((3, 3), np.nan)
    np.fill_diagonal(S, [0.02, 0.0, -0.01])
    S[2, 1] = 0.01
    tau = np.full((3, 3), 60.0 * pot.FS)
    nst = M.NST(S, T, dt, kB=pot.KB_EV, tau=tau, nreset=nreset)
    nst.run(g, nsteps, masses)
    vo, Ho, Tpo, outo, histo, nro = o.nst_run(v, masses, pot.KB_EV, T, dt, S, nsteps, tau=tau, nreset=nreset)
    say(f"{len(v)} atoms: max|dH| {np.abs(g.H - Ho).max():.2e} A, max|dx| {np.abs(g.x - o.x).max():.2e} A")
    assert np.abs(g.H - Ho).max() < 1e-6 and np.abs(g.x - o.x).max() < 1e-6
    assert np.abs(g.x_d - vo).max() < 1e-6
    np.testing.assert_allclose(nst.hist[:, 1], histo[:, 1], rtol=0, atol=5e-8 * len(v) + 1e-6)
    np.testing.assert_allclose(nst.hist[:, 0], histo[:, 0], rtol=1e-6)


def test_a_box_that_leaves_its_bounds_stops_the_run(M):
    p, H, g, o, v, masses = setup(M, 5, 3, 300.0)
    S = np.full((3, 3), np.nan)
    np.fill_diagonal(S, 0.2)
    nst = M.NST(S, 300.0, 2.0 * pot.FS, kB=pot.KB_EV, tau=np.full((3, 3), 60.0 * pot.FS))
    with pytest.raises(M.MappError, match="the box left"):
        nst.run(g, 100, masses)


def test_rejects_a_target_with_no_component(M):
    p, H, g, o, v, masses = setup(M, 4, 1, 300.0)
    nst = M.NST(np.full((3, 3), np.nan), 300.0, pot.FS, kB=pot.KB_EV)
    with pytest.raises(M.MappError, match="at least one stress component"):
        nst.run(g, 10, masses)
