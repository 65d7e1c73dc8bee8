"""GPU parity of the DMD (Gaussian-smeared EAM) path against the oracle.

Bars: per-component neighbor sets bit-exact; the DMD kernels run FP64, so
forces on x and alpha, the chemical-potential sums, free energy, virial and
entropy agree with the FP64 oracle to 1e-9 relative (summation order only).
"""
import sys

import numpy as np
import pytest

import oracle_lib as O
from mapp4py_amd import potentials as pot

pytestmark = pytest.mark.gpu

RTOL = 1e-9


def say(msg):
    print(msg, flush=True)
    sys.stdout.flush()


@pytest.fixture(scope="module")
def M():
    import mapp4py_amd

    return mapp4py_amd


@pytest.fixture(scope="module")
def cuh():
    return pot.johnson_cuh(nr=5000, nrho=5000, rc=5.5)


def sites(cells, seed, tilt=(0, 0, 0)):
    x, H, elem, alpha, c = pot.dmd_cuh_sites(cells, seed=seed)
    H = H.copy()
    H[1, 0], H[2, 0], H[2, 1] = tilt
    x = x + np.random.default_rng(seed + 100).normal(0, 0.05, x.shape)
    return x, H, elem, alpha, c


def both(M, p, x, H, elem, alpha, c, nquad=3):
    g = M.AtomsDMD(M.ForceFieldEAM.from_knots(p, dmd=True), H, x, elem, alpha, c, nquad=nquad, masses=p.masses)
    o = O.ODMD(O.OEam.from_knots(p, dmd=True), H, x, elem, alpha, c, nquad=nquad, masses=p.masses)
    return g, o


def triples(i, j, img):
    return {(int(a), int(b), *map(int, m)) for a, b, m in zip(i, j, img)}


def close(a, b, tag):
    a, b = np.asarray(a), np.asarray(b)
    err = np.abs(a - b).max() / max(1e-300, np.abs(b).max())
    assert err < RTOL, (tag, err)
    return err


def test_box_change_and_static_force_calc_match_oracle(M, cuh):
    # a strained box through mapp_dmd_set_box gives the oracle's derivative
    # in that box; force_calc_static then re-sums the free energy, virial and
    # entropy of the state c_d left (src/ff_dmd.cpp:429-445), and refuses a
    # changed state
    x, H, elem, alpha, c = sites((3, 3, 3), 7)
    g, _ = both(M, cuh, x, H, elem, alpha, c)
    strain = np.eye(3) + np.array([[0.015, 0, 0], [0.04, -0.01, 0], [-0.03, 0.02, 0.012]])
    H1, x1 = H @ strain, x @ strain
    g.set_box(H1, x1)
    o = O.ODMD(O.OEam.from_knots(cuh, dmd=True), H1, x1, elem, alpha, c, nquad=3, masses=cuh.masses)
    assert triples(*g.half_pairs()) == triples(*o.pairs())
    fo, fao, muo, feo, FHo, So = o.force()
    f, fa, mu, fe, FH, S = g.derivative()
    errs = [close(f, fo, "f_x"), close(fa, fao, "f_alpha"), close([fe], [feo], "fe"), close(FH, FHo, "F_H")]
    say(f"DMD strained box: rel errors f {errs[0]:.1e} f_a {errs[1]:.1e} fe {errs[2]:.1e} F_H {errs[3]:.1e}")
    g.c_d([3.5, 3.5], [1.7, 1.7])
    fe_s, FH_s, S_s = g.force_calc_static()
    close([fe_s], [feo], "static fe")
    close(FH_s, FHo, "static F_H")
    close([S_s], [So], "static S")
    assert abs(fe_s - fe) < 1e-12 * abs(fe) and np.abs(FH_s - FH).max() < 1e-12 * np.abs(FH).max()
    g.set_state(*g.state())
    with pytest.raises(M.MappError):
        g.force_calc_static()
    with pytest.raises(M.MappError):
        g.set_box(np.diag([2.0, 30.0, 30.0]))
    f2 = g.derivative()[0]
    close(f2, fo, "f_x after a rejected box")


@pytest.mark.parametrize("face", [False, True])
def test_coincident_sites_have_no_finite_gradient(M, cuh, face):
    # a site given twice, or on both faces of the box: r = 0 stays a pair, and
    # its 1 / r makes the totals and the two sites' gradient non-finite, in
    # every table mode; what the oracle has finite stays so
    x, H, elem, alpha, c = pot.dmd_cuh_sites((3, 3, 3), seed=3)
    x = x - x[0]
    x = np.concatenate([x, [H[0] if face else x[0]]])
    elem, alpha, c = (np.concatenate([v, v[:1]]) for v in (elem, alpha, c))
    g, o = both(M, cuh, x, H, elem, alpha, c)
    fo, fao, muo, feo, FHo, So = o.force()
    assert not np.isfinite(feo) and 0 < np.isfinite(fo).all(1).sum() < len(x)
    for mode in ("FP64", "batch 2", "single pairs", "FP32 knots", "FP32 rows"):
        g.set_batch({"batch 2": 2, "single pairs": 1}.get(mode, 4))
        g.set_fp32(mode.startswith("FP32"), rows=mode == "FP32 rows")
        f, fa, mu, fe, FH, S = g.derivative()
        say(f"DMD coincident sites, {mode}: fe {fe}, {np.isfinite(f).all(1).sum()} of {len(x)} sites with finite f")
        assert not np.isfinite(fe) and not np.isfinite(FH).any() and not np.isfinite(g.value())
        for a, b in ((f, fo), (fa, fao), (mu, muo)):
            assert not np.isfinite(a[[0, -1]]).all(1).any()
            assert np.isfinite(a[np.isfinite(b)]).all()
        assert abs(S - So) < 1e-12 * abs(So)


@pytest.mark.parametrize("nr,rows", [(5000, True), (5000, False), (20000, False)])
def test_fp32_tables_stay_within_the_stated_bars(M, nr, rows):
    # FP32 pair splines, FP64 moments and sums: the free energy and gradient
    # against the FP64 oracle, from FP32 copies of the coefficient rows
    # (rows) or from FP32 knot values and slopes with the top knots in LDS.
    # At nr = 20000 the LDS window starts near 4.4 A, so most Hermite points
    # read the knots below it from device memory. Bars: forces on x and
    # alpha 1e-4 eV/A (the DMD force bar), mu 1e-4 eV, free energy 1e-8
    # relative, virial 1e-6 of its largest component. The rate path does not
    # read the FP32 tables.
    p = pot.johnson_cuh(nr=nr, nrho=5000, rc=5.5)
    x, H, elem, alpha, c = sites((4, 4, 4), 5, (0.3, -0.2, 0.4))
    g, o = both(M, p, x, H, elem, alpha, c)
    fo, fao, muo, feo, FHo, So = o.force()
    r_crd, zeta = [3.5, 3.5], [1.7, 1.7]
    cd64 = g.c_d(r_crd, zeta)[0]
    g.set_fp32(True, rows=rows)
    first = g.knot_window()
    say(f"DMD FP32 {'rows' if rows else 'knots'}, nr {nr}: LDS window from knot {first} "
        f"(r = {first * p.dr:.2f} A)")
    assert first >= 0
    if nr == 20000:
        assert first * p.dr > 3.0
    for batch in (2, 4):
        g.set_batch(batch)
        f, fa, mu, fe, FH, S = g.derivative()
        df, dfa, dmu = np.abs(f - fo).max(), np.abs(fa - fao).max(), np.abs(mu - muo).max()
        dfe = abs(fe - feo) / abs(feo)
        dFH = np.abs(FH - FHo).max() / np.abs(FHo).max()
        say(f"  batch {batch}: max|df| {df:.1e} eV/A, max|df_a| {dfa:.1e}, max|dmu| {dmu:.1e} eV, "
            f"fe rel {dfe:.1e}, F_H rel {dFH:.1e}, S rel {abs(S - So) / abs(So):.1e}")
        assert df < 1e-4 and dfa < 1e-4 and dmu < 1e-4
        assert dfe < 1e-8 and dFH < 1e-6
        assert abs(S - So) < 1e-12 * abs(So)
        assert abs(g.value() - o.energy()) < 1e-8 * abs(feo)
    cd32 = g.c_d(r_crd, zeta)[0]
    np.testing.assert_array_equal(cd32, cd64)
    g.set_fp32(False)
    f64 = g.derivative()[0]
    close(f64, fo, "f_x back on the FP64 rows")


@pytest.mark.parametrize("lbfgs", [False, True])
def test_minimisers_run_on_the_fp32_knots(M, cuh, lbfgs):
    # the DMD minimisers with the FP32 knots in LDS (alternating energy and
    # gradient passes over the packed records each pass 1 writes) descend as
    # they do on the FP64 rows: the same start, and a descent within 1e-4 of
    # the FP64 one after 25 iterations (seen 1e-6 to 2e-6)
    x, H, elem, alpha, c = sites((3, 3, 3), 9, (0.2, 0.0, -0.1))
    res = {}
    for fp32 in (False, True):
        g = M.AtomsDMD(M.ForceFieldEAM.from_knots(cuh, dmd=True), H, x, elem, alpha, c, nquad=3,
                       masses=cuh.masses)
        g.set_fp32(fp32)
        res[fp32] = g.min_lbfgs(max_iter=25, e_tol=0.0) if lbfgs else g.min_cg(max_iter=25, e_tol=0.0)
    r32, r64 = res[True], res[False]
    d32, d64 = r32["fe0"] - r32["fe"], r64["fe0"] - r64["fe"]
    say(f"DMD {'L-BFGS' if lbfgs else 'CG'} 25 iterations: descent FP32 knots {d32:.6e}, FP64 rows {d64:.6e} eV")
    assert abs(r32["fe0"] - r64["fe0"]) < 1e-8 * abs(r64["fe0"])
    assert d64 > 0.0 and abs(d32 - d64) < 1e-4 * d64


@pytest.mark.parametrize("cells,tilt,seed", [((3, 3, 3), (0, 0, 0), 1), ((3, 4, 3), (0.6, -0.4, 0.5), 2),
                                             ((2, 2, 2), (0, 0, 0), 3)])
def test_dmd_lists_and_derivative_match_oracle(M, cuh, cells, tilt, seed):
    x, H, elem, alpha, c = sites(cells, seed, tilt)
    g, o = both(M, cuh, x, H, elem, alpha, c)
    assert triples(*g.half_pairs()) == triples(*o.pairs())
    fo, fao, muo, feo, FHo, So = o.force()
    for batch in (1, 2, 4):  # per-pair loop, batched passes
        g.set_batch(batch)
        f, fa, mu, fe, FH, S = g.derivative()
        errs = [close(f, fo, "f_x"), close(fa, fao, "f_alpha"), close(mu, muo, "mu"), close([fe], [feo], "fe"),
                close(FH, FHo, "F_H"), close([S], [So], "S")]
        say(f"DMD {cells} tilt {tilt} batch {batch}: rel errors f {errs[0]:.1e} f_a {errs[1]:.1e} "
            f"mu {errs[2]:.1e} fe {errs[3]:.1e} F_H {errs[4]:.1e} S {errs[5]:.1e}")
        close([g.value()], [o.energy()], "value")
        fe_r, FH_r, S_r = g.evaluate()
        assert fe_r == fe and np.array_equal(FH_r, FH) and S_r == S


def test_chemical_potential_transform(M, cuh):
    x, H, elem, alpha, c = sites((3, 3, 3), 5)
    g, _ = both(M, cuh, x, H, elem, alpha, c)
    ext = np.array([-3.2, -2.3])
    _, _, raw, fe0, _, _ = g.derivative(False)
    _, _, chem, fe1, _, _ = g.derivative(True, ext)
    kT = pot.KB_EV * 300.0
    lam = pot.HP / np.sqrt(2 * np.pi * kT * np.asarray(cuh.masses))
    mu0 = kT * 1.5 * (2 * np.log(lam) - 1 - np.log(np.pi))
    cv = 1.0 - c.sum(1, keepdims=True)
    want = -raw - kT * (np.log(c) - np.log(cv) - 3 * np.log(alpha)) - mu0[elem] + ext[elem]
    np.testing.assert_allclose(chem, want, rtol=1e-12, atol=1e-12)
    assert abs((fe0 - fe1) - (c * ext[elem]).sum()) < 1e-9 * abs(fe0)
    assert abs(g.value(True, ext) - fe1) < 1e-9 * abs(fe1)


def test_smear_matches_oracle_pair_eval(M, cuh):
    x, H, elem, alpha, c = sites((2, 2, 2), 7)
    g, o = both(M, cuh, x, H, elem, alpha, c)
    rng = np.random.default_rng(3)
    r = rng.uniform(1.5, 6.0, 64)
    a = rng.uniform(0.07, 0.42, 64)
    for ei in range(2):
        for ej in range(2):
            out = g.smear(ei, ej, r, a)
            ref = np.array([o.pair_eval(ei, ej, rr, aa) for rr, aa in zip(r, a)])
            np.testing.assert_allclose(out, ref, rtol=1e-12, atol=1e-13)


def test_dmd_update_and_rebuild(M, cuh):
    x, H, elem, alpha, c = sites((3, 3, 3), 9)
    g, _ = both(M, cuh, x, H, elem, alpha, c)
    xw, aw, cw = g.state()
    g.set_state(xw + 0.05, aw, cw)
    assert g.update() is False
    a2 = aw.copy()
    a2[3, 1] += 0.3  # alpha growth times x_max beyond skin/2
    g.set_state(xw + 0.05, a2, cw)
    assert g.update() is True
    xs, as_, cs = g.state()
    o = O.ODMD(O.OEam.from_knots(cuh, dmd=True), H, xs, elem, as_, cs, nquad=3, masses=cuh.masses)
    assert triples(*g.half_pairs()) == triples(*o.pairs())
    f, fa, mu, fe, FH, S = g.derivative()
    fo, fao, muo, feo, FHo, So = o.force()
    close(f, fo, "f after rebuild")
    close(fa, fao, "f_alpha after rebuild")


def test_cg_lowers_free_energy_and_gradient(M, cuh):
    x, H, elem, alpha, c = sites((3, 3, 3), 11)
    g, _ = both(M, cuh, x, H, elem, alpha, c)
    r = g.min_cg(max_iter=60, e_tol=1e-12, grad_tol=1e-6)
    f, fa, mu, fe, FH, S = g.derivative()
    say(f"CG: {r['iters']} iterations status {r['status']} fe {r['fe0']:.6f} -> {r['fe']:.6f} "
        f"max|grad| {r['grad_max']:.2e}")
    assert r["fe"] < r["fe0"]
    assert abs(fe - r["fe"]) < 1e-9 * abs(fe)
    assert max(np.abs(f).max(), np.abs(fa).max()) == pytest.approx(r["grad_max"], rel=1e-12)
    # the result is a stationary point of the oracle's free energy too
    xs, as_, cs = g.state()
    o = O.ODMD(O.OEam.from_knots(cuh, dmd=True), H, xs, elem, as_, cs, nquad=3, masses=cuh.masses)
    fo, fao, _, feo, _, _ = o.force()
    assert abs(feo - r["fe"]) < 1e-9 * abs(feo)
    assert max(np.abs(fo).max(), np.abs(fao).max()) < 10 * r["grad_max"] + 1e-9


@pytest.mark.parametrize("cells,tilt,seed", [((3, 3, 3), (0, 0, 0), 11), ((3, 4, 3), (0.6, -0.4, 0.5), 12)])
def test_concentration_rates_match_oracle(M, cuh, cells, tilt, seed):
    # ForceFieldDMD::c_d_calc over the second list (same element, r < r_crd)
    x, H, elem, alpha, c = sites(cells, seed, tilt)
    g, o = both(M, cuh, x, H, elem, alpha, c)
    r_crd, zeta = [3.5, 3.5], [1.7, 1.7]
    cd, norm = g.c_d(r_crd, zeta)
    cdo, normo = o.c_d(r_crd, zeta, cuh.masses)
    err = np.abs(cd - cdo).max() / normo
    say(f"c_d {cells} tilt {tilt}: max|c_d| {norm:.6e} vs {normo:.6e}, rel error {err:.1e}")
    assert normo > 0.0 and err < RTOL
    assert abs(norm - normo) < RTOL * normo
    for e in (0, 1):  # exchange conserves each element
        assert abs(cd[elem == e].sum()) < 1e-11 * np.abs(cd[elem == e]).sum()
    _, norm2 = g.c_d(r_crd, zeta, fetch=False)
    assert norm2 == norm


@pytest.mark.parametrize("cells,tilt,seed", [((3, 3, 3), (0, 0, 0), 11), ((3, 4, 3), (0.6, -0.4, 0.5), 12)])
def test_jacobian_product_matches_oracle(M, cuh, cells, tilt, seed):
    # ForceFieldEAMDMD::__J at the state of the last c_d call
    x, H, elem, alpha, c = sites(cells, seed, tilt)
    g, o = both(M, cuh, x, H, elem, alpha, c)
    r_crd, zeta = [3.5, 3.5], [1.7, 1.7]
    with pytest.raises(RuntimeError):
        g.J(np.zeros_like(c))  # no c_d at this state yet
    g.c_d(r_crd, zeta, fetch=False)
    rng = np.random.default_rng(seed)
    v, w = rng.normal(0.0, 1.0, c.shape), rng.normal(0.0, 1.0, c.shape)
    Jv = g.J(v)
    Jvo = o.J(r_crd, zeta, cuh.masses, v)
    scale = np.abs(Jvo).max()
    err = np.abs(Jv - Jvo).max() / scale
    say(f"J {cells} tilt {tilt}: max|Jx| {scale:.6e}, rel error vs oracle {err:.1e}")
    assert scale > 0.0 and err < RTOL
    # a second product at the same state reuses the slot values; linear in x
    Jw = g.J(w)
    Jvw = g.J(2.0 * v - 3.0 * w)
    assert np.abs(Jvw - (2.0 * Jv - 3.0 * Jw)).max() < 1e-12 * np.abs(Jvw).max()
    for e in (0, 1):  # exchange conserves each element, also to first order
        assert abs(Jv[elem == e].sum()) < 1e-11 * np.abs(Jv[elem == e]).sum()
    live, exch = g.J_entries()  # every pair from both sides
    assert 0 < exch <= live <= 2 * len(g.half_pairs()[0]) and exch % 2 == 0
    # a new state needs a new c_d (here the same values written again)
    xs, as_, cs = g.state()
    g.set_state(xs, as_, cs)
    with pytest.raises(RuntimeError):
        g.J(v)
    g.c_d(r_crd, zeta, fetch=False)
    np.testing.assert_allclose(g.J(v), Jv, rtol=0, atol=1e-13 * scale)


@pytest.mark.parametrize("dt", [30.0, 300.0])
def test_implicit_step_matches_oracle(M, cuh, dt):
    # DAEImplicit::newton for one backward-Euler step c - c_n = dt c_d(c)
    x, H, elem, alpha, c = sites((3, 3, 3), 11)
    g, o = both(M, cuh, x, H, elem, alpha, c)
    r_crd, zeta = [3.5, 3.5], [1.7, 1.7]
    ok, it = g.newton(r_crd, zeta, dt, -c / dt, a_tol=1e-8)
    oko, ito, co = o.newton(r_crd, zeta, cuh.masses, dt, -c / dt, a_tol=1e-8)
    cg = g.state()[2]
    err = np.abs(cg - co).max() / np.abs(co - c).max()
    say(f"implicit step dt {dt}: converged {ok}/{oko}, iterations {it}/{ito}, max|dc| {np.abs(co - c).max():.3e}, "
        f"rel diff vs oracle {err:.1e}")
    assert ok and oko and it == ito
    assert err < 1e-6
    for e in (0, 1):
        assert abs((cg - c)[elem == e].sum()) < 1e-12
    # the solution is a root of F: the rates there agree with the oracle's
    g.c_d(r_crd, zeta, fetch=False)
    cdg = g.c_d(r_crd, zeta)[0]
    F = cg / dt - c / dt - cdg
    assert np.linalg.norm(F) < 0.01 * 1e-8 * np.sqrt(c.size)


def test_implicit_step_that_does_not_converge_restores_c(M, cuh):
    x, H, elem, alpha, c = sites((3, 3, 3), 11)
    g, o = both(M, cuh, x, H, elem, alpha, c)
    ok, _ = g.newton([3.5, 3.5], [1.7, 1.7], 3000.0, -c / 3000.0, a_tol=1e-8)
    oko, _, _ = o.newton([3.5, 3.5], [1.7, 1.7], cuh.masses, 3000.0, -c / 3000.0, a_tol=1e-8)
    assert not ok and not oko
    np.testing.assert_array_equal(g.state()[2], c)
    with pytest.raises(RuntimeError):
        g.newton([3.5, 3.5], [1.7, 1.7], 30.0, -c / 30.0, max_ngmres_iters=9)


def test_unit_gradient_matches_oracle(M, cuh):
    # calc_mu's f and f_alpha (per unit c, fcoef-weighted) after c_d
    x, H, elem, alpha, c = sites((3, 3, 3), 11)
    c = c.copy()
    c[0] = 0.0  # an empty site: fcoef 1 on its zero components
    g, o = both(M, cuh, x, H, elem, alpha, c)
    g.c_d([3.5, 3.5], [1.7, 1.7], fetch=False)
    gu, gau = g.unit_gradient()
    ou, oau = o.unit_grad()
    err = max(np.abs(gu - ou).max() / np.abs(ou).max(), np.abs(gau - oau).max() / np.abs(oau).max())
    say(f"unit gradient: max|g| {np.abs(ou).max():.3e}, max|g_alpha| {np.abs(oau).max():.3e}, rel error {err:.1e}")
    assert err < RTOL
    g.set_state(*g.state())
    with pytest.raises(RuntimeError):
        g.unit_gradient()


def test_absent_components_match_oracle(M, cuh):
    # a quarter of the sites without their H component (c = -1): no list rows
    # or entries for it, zero rates, Jacobian rows and gradients there, and the
    # implicit step leaves it at -1
    x, H, elem, alpha, c = sites((3, 3, 3), 21)
    c, alpha = c.copy(), alpha.copy()
    gone = np.random.default_rng(22).uniform(size=len(c)) < 0.25
    c[gone, 1] = -1.0
    alpha[gone, 1] = 0.0
    g, o = both(M, cuh, x, H, elem, alpha, c)
    assert triples(*g.half_pairs()) == triples(*o.pairs())
    f, fa, mu, fe, FH, S = g.derivative()
    fo, fao, muo, feo, FHo, So = o.force()
    # absent components: the reference adds 3 kT c / alpha to their f_alpha
    # (-inf for the importer's alpha = 0); the GPU leaves 0 there
    assert np.all(fa[gone, 1] == 0.0) and np.all(np.isinf(fao[gone, 1]))
    fao = np.where(np.isinf(fao), 0.0, fao)
    errs = [close(f, fo, "f"), close(fa, fao, "f_alpha"), close(mu, muo, "mu"), close([fe], [feo], "fe")]
    r_crd, zeta = [3.5, 3.5], [1.7, 1.7]
    cd, _ = g.c_d(r_crd, zeta)
    cdo, normo = o.c_d(r_crd, zeta, cuh.masses)
    assert np.abs(cd - cdo).max() < RTOL * normo and np.all(cd[gone, 1] == 0.0)
    gu, gau = g.unit_gradient()
    ou, oau = o.unit_grad()
    assert np.abs(gu - ou).max() < RTOL * np.abs(ou).max() and np.abs(gau - oau).max() < RTOL * np.abs(oau).max()
    v = np.random.default_rng(23).normal(0.0, 1.0, c.shape)
    Jv, Jvo = g.J(v), o.J(r_crd, zeta, cuh.masses, v)
    assert np.abs(Jv - Jvo).max() < RTOL * np.abs(Jvo).max() and np.all(Jv[gone, 1] == 0.0)
    ok, it = g.newton(r_crd, zeta, 30.0, -c / 30.0, a_tol=1e-8)
    oko, ito, co = o.newton(r_crd, zeta, cuh.masses, 30.0, -c / 30.0, a_tol=1e-8)
    cg = g.state()[2]
    say(f"absent components: f/f_a/mu/fe {max(errs):.1e}, c_d, unit gradient and J within {RTOL}; implicit step "
        f"{ok}/{oko} in {it}/{ito}, max|dc| vs oracle {np.abs(cg - co).max():.1e}")
    assert ok and oko and it == ito
    assert np.abs(cg - co).max() < 1e-6 * np.abs(co - c).max() and np.all(cg[gone, 1] == -1.0)


def test_cg_through_list_rebuilds(M, cuh):
    # with a tiny skin the CG's trial points trigger many rebuilds, which
    # reorder the sites; the minimisation must follow them and land where a run
    # with few rebuilds (large skin; alpha growth still triggers some) lands
    x, H, elem, alpha, c = sites((3, 3, 3), 31)
    x = x + np.random.default_rng(32).normal(0, 0.12, x.shape)
    out = []
    for skin in (0.02, 1.0):
        g = M.AtomsDMD(M.ForceFieldEAM.from_knots(cuh, dmd=True), H, x, elem, alpha, c, nquad=3, skin=skin,
                       masses=cuh.masses)
        g.profile(True)
        r = g.min_cg(max_iter=40, e_tol=0.0, max_dx=0.1, grad_tol=0.0)
        rebuilds = g.profile_read("cell_sort")[1]
        g.profile(False)
        out.append((r, rebuilds, g.state()))
    (ra, na, sa), (rb, nb, sb) = out
    say(f"CG 40 iterations: skin 0.02 {na} rebuilds fe {ra['fe']:.10f}; skin 1.0 {nb} rebuilds fe {rb['fe']:.10f}")
    assert na > 3 * max(nb, 1)
    assert ra["iters"] == rb["iters"] and abs(ra["fe"] - rb["fe"]) < 1e-8 * abs(rb["fe"])
    assert ra["fe"] < ra["fe0"] - 1.0
    ds = (sa[0] - sb[0]) @ np.linalg.inv(H)
    ds -= np.round(ds)
    assert np.abs(ds @ H).max() < 1e-6 and np.abs(sa[1] - sb[1]).max() < 1e-7


def test_lbfgs_lowers_free_energy_below_the_cg(M, cuh):
    # MinLBFGSDMD over x and alpha: its free energy and gradient are the
    # oracle's at the state it stops in, and it gets lower than the CG does
    # from the same start (both stop on the energy tolerance while widths
    # approach zero, the limit that caps their steps)
    x, H, elem, alpha, c = sites((3, 3, 3), 11)
    g, _ = both(M, cuh, x, H, elem, alpha, c)
    r = g.min_lbfgs(m=5, max_iter=300, e_tol=1e-14, grad_tol=1e-6)
    f, fa, mu, fe, FH, S = g.derivative()
    say(f"DMD L-BFGS: {r['iters']} iterations status {r['status']} fe {r['fe0']:.6f} -> {r['fe']:.10f} "
        f"max|grad| {r['grad_max']:.2e}")
    assert r["fe"] < r["fe0"]
    assert abs(fe - r["fe"]) < 1e-9 * abs(fe)
    xs, as_, cs = g.state()
    o = O.ODMD(O.OEam.from_knots(cuh, dmd=True), H, xs, elem, as_, cs, nquad=3, masses=cuh.masses)
    fo, fao, _, feo, _, _ = o.force()
    assert abs(feo - r["fe"]) < 1e-9 * abs(feo)
    assert max(np.abs(fo).max(), np.abs(fao).max()) == pytest.approx(r["grad_max"], rel=1e-6)
    g2, _ = both(M, cuh, x, H, elem, alpha, c)
    rc = g2.min_cg(max_iter=3000, e_tol=1e-14, grad_tol=1e-6)
    say(f"  CG from the same start: {rc['iters']} iterations fe {rc['fe']:.10f} max|grad| {rc['grad_max']:.2e}")
    assert r["fe"] < rc["fe"]


def test_lbfgs_through_list_rebuilds(M, cuh):
    # the stored pairs follow their sites through the rebuilds of a tiny skin
    x, H, elem, alpha, c = sites((3, 3, 3), 31)
    x = x + np.random.default_rng(32).normal(0, 0.12, x.shape)
    out = []
    for skin in (0.02, 1.0):
        g = M.AtomsDMD(M.ForceFieldEAM.from_knots(cuh, dmd=True), H, x, elem, alpha, c, nquad=3, skin=skin,
                       masses=cuh.masses)
        g.profile(True)
        r = g.min_lbfgs(m=3, max_iter=25, e_tol=0.0, max_dx=0.1, grad_tol=0.0)
        rebuilds = g.profile_read("cell_sort")[1]
        g.profile(False)
        out.append((r, rebuilds, g.state()))
    (ra, na, sa), (rb, nb, sb) = out
    say(f"DMD L-BFGS 25 iterations: skin 0.02 {na} rebuilds fe {ra['fe']:.10f}; skin 1.0 {nb} rebuilds "
        f"fe {rb['fe']:.10f}")
    assert na > 3 * max(nb, 1)
    assert ra["iters"] == rb["iters"] and abs(ra["fe"] - rb["fe"]) < 1e-8 * abs(rb["fe"])
    assert ra["fe"] < ra["fe0"] - 1.0
    ds = (sa[0] - sb[0]) @ np.linalg.inv(H)
    ds -= np.round(ds)
    assert np.abs(ds @ H).max() < 1e-6 and np.abs(sa[1] - sb[1]).max() < 1e-7


@pytest.mark.parametrize("which,ls", [("cg", "golden"), ("cg", "brent"), ("lbfgs", "golden"), ("lbfgs", "brent")])
def test_dmd_minimisers_with_golden_and_brent(M, cuh, which, ls):
    # dmd.min_cg / dmd.min_lbfgs with ls_golden or ls_brent: the free energy
    # falls, and at the state they stop in it and its gradient are the oracle's
    x, H, elem, alpha, c = sites((3, 3, 3), 41)
    g, _ = both(M, cuh, x, H, elem, alpha, c)
    search = M.LineSearchGoldenSection() if ls == "golden" else M.LineSearchBrent()
    if which == "cg":
        r = g.min_cg(max_iter=30, e_tol=0.0, ls=search)
    else:
        r = g.min_lbfgs(m=3, max_iter=30, e_tol=0.0, ls=search)
    say(f"DMD {which} with {ls}: {r['iters']} iterations status {r['status']} fe {r['fe0']:.6f} -> {r['fe']:.8f}")
    assert r["fe"] < r["fe0"] - 1.0
    f, fa, mu, fe, FH, S = g.derivative()
    xs, as_, cs = g.state()
    o = O.ODMD(O.OEam.from_knots(cuh, dmd=True), H, xs, elem, as_, cs, nquad=3, masses=cuh.masses)
    fo, fao, _, feo, _, _ = o.force()
    assert abs(feo - fe) < 1e-9 * abs(feo)
    assert max(np.abs(fo - f).max(), np.abs(fao - fa).max()) < 1e-8 * max(np.abs(fo).max(), 1.0)
