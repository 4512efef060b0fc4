"""The benchmark configurations on the HIP path, at their own sizes, through
the C ABI, each against the oracle, the reference's golden outputs or the
mathematics that fixes the result:

  C1  8^3x4 trajectory of the reference's update() (golden_c1), leapfrog
  C2  16^4 Dslash + 15-shift multi-shift (FP64 and FP32+FP64 refinement)
  C3  24^4 fermion force: tests/test_force_adjoint.py (parametrised)
  C4  32^3x8, 8 pseudofermions x 16 shifts: every shifted FP64 true
      residual, Delta H of the mixed trajectory against its FP64
      recomputation; the six uneven lattices in lockstep = one by one
  C5  48^3x12 mixed trajectory, Delta H against the FP64 recomputation

plus the spectral bounds against dense eigenvalues, the free-field spectrum
of the device operator, the device Gaussian draws against their host
restatement, reversibility of the MD, and the solver's failure statuses.
Tolerances are written in each test."""
import os
import sys

import numpy as np
import pytest

import rng
from oracle import Oracle
from rhmc_amd import Gpu, RhmcError, fields, multi_trajectory
from rhmc_amd.lib import RHMC_EINVAL, RHMC_EMAXCG, RHMC_ENONFINITE
from rhmc_amd.remez import rhmc_approximations

pytestmark = pytest.mark.gpu

GOLD = os.path.join(os.path.dirname(__file__), "golden")


def rel(a, b):
    return np.linalg.norm((a - b).ravel()) / max(np.linalg.norm(b.ravel()), 1e-300)


def say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


def coeffs(app):
    return app.a0, np.array(app.a), np.array(app.b)


def measured_bounds(g, mass, tol=1e-6):
    mx = g.find_max(tol, seed=11)
    mn = max(g.find_min(mx, tol, seed=12), mass * mass)
    return mn, mx


# ------------------------------------------------------------------ C1
def test_c1_golden_on_device():
    """C1 (8^3x4, am=0.05, beta=5.5, 1 pseudofermion, 8 MD / 12 action
    poles, 10 Omelyan steps, residuals 1e-10) against the reference's own
    CPU outputs: Dslash 1e-14, multi-shift solutions 1e-10, the trajectory's
    Delta H 1e-9 absolute, links/momenta/chi 1e-10, phi_new 1e-9,
    measurements 1e-11-1e-13.  The inputs are regenerated from their seeds
    and pinned by the fixture's checksum."""
    gd = dict(np.load(os.path.join(GOLD, "golden_c1.npz")))
    dims = tuple(int(x) for x in gd["dims"])
    lat = fields.Lattice(*dims)
    U = fields.random_links(lat, int(gd["link_seed"]), None)
    P = fields.gauss_momenta(lat, 202)
    phi = fields.gauss_spinor(lat, 303, 1)
    chk = np.array([np.abs(U).sum(), np.abs(P).sum(), np.abs(phi).sum()])
    np.testing.assert_allclose(chk, gd["input_checksum"], rtol=1e-13)
    mass, beta = float(gd["mass"]), float(gd["beta"])
    say("C1", dims)
    g = Gpu(dims, mass=mass, beta=beta, n_pf=1, max_order=12)
    g.init0(U)
    assert rel(g.dslash(1, gd["dslash_in"][0], 0)[0], gd["doe"]) < 1e-14
    assert rel(g.dslash(0, gd["dslash_in"][1], 0)[0], gd["deo"]) < 1e-14
    assert rel(g.dslash(1, gd["dslash_in"][0], 1)[0], gd["doe"]) < 2e-6
    # the reference's multi-shift golden solves for the chi draw (seed 606)
    g.init1(phi=fields.gauss_spinor(lat, 606, 1))
    g.multishift(gd["ms_shifts"], float(gd["ms_res"]), relative=False, precision=0)
    x = g.get_fermions("smf").reshape(gd["ms_x"].shape)
    assert rel(x, gd["ms_x"]) < 1e-10
    np.testing.assert_allclose(g.gauge_meas(), gd["meas_gauge"], rtol=1e-13, atol=1e-15)
    v, _ = g.chiral_meas(float(gd["n_flavours"]), float(gd["res_metro"]), gd["meas_rnd_e"], gd["meas_rnd_o"])
    np.testing.assert_allclose(v, gd["meas_chiral"], rtol=1e-11, atol=1e-12)
    g.init1(momenta=P)
    g.put_fermions("phi", phi)
    r = g.trajectory(precision=0, n_flavours=int(gd["n_flavours"]), no_md=int(gd["no_md"]),
                     integrator="omelyan", gauge_scale=int(gd["gauge_scale"]), res_md=float(gd["res_md"]),
                     res_metro=float(gd["res_metro"]),
                     first=(float(gd["first_a0"]), gd["first_a"], gd["first_b"]),
                     md=(float(gd["md_a0"]), gd["md_a"], gd["md_b"]),
                     last=(float(gd["last_a0"]), gd["last_a"], gd["last_b"]),
                     bounds=(float(gd["eig_min"]), float(gd["eig_max"])))
    U1, _, P1 = g.end(links=True, ipdot=False, momenta=True)
    sel = gd["traj_sel"]
    say("C1 dH", r.delta_h, "reference", float(gd["traj_dh"]), "iterations", r.cg_iterations)
    assert abs(r.delta_h - float(gd["traj_dh"])) < 1e-9
    assert rel(g.get_fermions("chi"), gd["traj_chi"]) < 1e-10
    assert rel(g.get_fermions("phinew"), gd["traj_phinew"]) < 1e-9
    assert rel(U1[sel], gd["traj_links_sel"]) < 1e-10
    assert rel(P1[sel], gd["traj_mom_sel"]) < 1e-10
    g.close()


@pytest.mark.parametrize("precision", [0, 1])
def test_leapfrog_trajectory_against_oracle(precision):
    """The leapfrog integrator (leapfrog.cc:18-62, with the live momentum
    sign) on the device against the oracle's leapfrog trajectory, C1's
    scheme with 10 steps on the 4^4 t4o inputs: Delta H 1e-9 absolute, links
    and momenta 1e-10 (FP64 solves, or FP32 iterations with FP64 defect
    correction for every solve)."""
    gd = dict(np.load(os.path.join(GOLD, "golden_t4o.npz")))
    dims = tuple(int(x) for x in gd["dims"])
    kw = dict(n_flavours=int(gd["n_flavours"]), no_md=10, integrator="leapfrog", res_md=1e-12, res_metro=1e-12,
              first=(float(gd["first_a0"]), gd["first_a"], gd["first_b"]),
              md=(float(gd["md_a0"]), gd["md_a"], gd["md_b"]),
              last=(float(gd["last_a0"]), gd["last_a"], gd["last_b"]))
    bounds = (float(gd["eig_min"]), float(gd["eig_max"]))
    g = Gpu(dims, mass=float(gd["mass"]), beta=float(gd["beta"]), n_pf=int(gd["no_ps"]), max_order=12)
    g.init0(gd["links"])
    g.init1(momenta=gd["mom"])
    g.put_fermions("phi", gd["phi"])
    r = g.trajectory(precision=precision, metro_precision=1, bounds=bounds, **kw)
    U1, _, P1 = g.end(links=True, ipdot=False, momenta=True)
    g.close()
    o = Oracle(dims)
    dh, Uo, Po, _, _ = o.trajectory(gd["links"], gd["mom"], gd["phi"], beta=float(gd["beta"]), mass=float(gd["mass"]),
                                    eig_min=bounds[0], eig_max=bounds[1], **kw)
    say("leapfrog dH", r.delta_h, "oracle", dh)
    assert abs(r.delta_h - dh) < 1e-9
    assert rel(U1, Uo) < 1e-10
    assert rel(P1, Po) < 1e-10


# ------------------------------------------------------------------ C2
@pytest.mark.parametrize("precision", [0, 1])
def test_c2_dslash_and_multishift_16c4(precision):
    """C2: 16^4, links exp(i 0.3 H), am=0.02, even-site Gaussian source, the
    15 poles of the Remez approximation rescaled to the measured bounds,
    relative residual 1e-10.  Dslash: FP64 1e-14, FP32 12-real 2e-6 against
    the oracle.  Multi-shift: every shifted FP64 true residual <= 1e-10 |b|,
    solutions within 1e-9 of the oracle's FP64 solve to 1e-12."""
    dims, mass = (16, 16, 16, 16), 0.02
    lat = fields.Lattice(*dims)
    U = fields.random_links(lat, 2024, 0.3)
    src = fields.gauss_spinor(lat, 7, 1)
    _, md, _ = rhmc_approximations(2, 1, 15, 15, 15)
    say("C2", dims, "precision", precision)
    g = Gpu(dims, mass=mass, beta=5.5, n_pf=1, max_order=15)
    g.init0(U)
    o = Oracle(dims)
    if precision == 0:
        v = fields.gauss_spinor(lat, 5, 2)
        assert rel(g.dslash(1, v, 0), np.stack([o.doe(U, v[k]) for k in range(2)])) < 1e-14
        assert rel(g.dslash(0, v, 0), np.stack([o.deo(U, v[k]) for k in range(2)])) < 1e-14
        assert rel(g.dslash(1, v, 1), np.stack([o.doe(U, v[k]) for k in range(2)])) < 2e-6
    mn, mx = measured_bounds(g, mass)
    _, _, b, _ = md.rescaled(mn, mx, -0.5)
    b = np.array(b)
    g.init1(phi=src)
    it = g.multishift(b, 1e-10, relative=True, precision=precision)
    bn = np.linalg.norm(src)
    res = g.shifted_residuals(b)[0] / bn
    say("C2 iterations", it, g.solve_stats(), "worst true residual", res.max())
    assert np.all(res <= 1e-10), res
    x = g.get_fermions("smf")
    xo, _ = o.multishift(U, mass, src[0], b, 1e-12 * bn)
    for k in range(len(b)):
        assert rel(x[k], xo[k]) < 1e-9, (k, rel(x[k], xo[k]))
    g.close()


def test_c2_fp64_basis_solve_to_1e_12():
    """The FP64 stored-basis solve stops on its recursive residual, which in
    the single-reduction form can drift from the true one; with the FP64
    true-residual check and defect correction after it, every shifted true
    residual meets a 1e-12 relative target at C2's conditioning (16^4,
    am=0.02, 15 Remez shifts on the measured bounds), for 2 right-hand
    sides, and the solutions agree with the oracle's solve to 1e-13 to
    within 1e-10."""
    dims, mass = (16, 16, 16, 16), 0.02
    lat = fields.Lattice(*dims)
    U = fields.random_links(lat, 2025, 0.3)
    src = fields.gauss_spinor(lat, 8, 2)
    _, md, _ = rhmc_approximations(2, 1, 15, 15, 15)
    g = Gpu(dims, mass=mass, beta=5.5, n_pf=2, max_order=15)
    g.init0(U)
    mn, mx = measured_bounds(g, mass)
    _, _, b, _ = md.rescaled(mn, mx, -0.5)
    b = np.array(b)
    g.init1(phi=src)
    it = g.multishift(b, 1e-12, relative=True, precision=0)
    bn = np.linalg.norm(src.reshape(2, -1), axis=1)
    res = g.shifted_residuals(b) / bn[:, None]
    say("C2 1e-12 iterations", it, g.solve_stats(), "worst true residual", res.max())
    assert np.all(res <= 1e-12), res.max()
    x = g.get_fermions("smf").reshape(2, 15, lat.Vh, 3)
    g.close()
    o = Oracle(dims)
    xo, _ = o.multishift(U, mass, src[1], b, 1e-13 * bn[1])
    for k in (0, 7, 14):
        assert rel(x[1, k], xo[k]) < 1e-10, (k, rel(x[1, k], xo[k]))


# ------------------------------------------------------------------ C4
def test_c4_32c8_residuals_and_delta_h():
    """C4 at full size: 32^3x8, am=0.01, beta=5.6, exp(i 0.3 H) links, 8
    pseudofermions x 16 poles.  FP64 and mixed multi-shift solves at relative
    residual 1e-10: all 128 shifted FP64 true residuals <= 1e-10 |b|, and
    the two solves agree to 1e-7.  One mixed trajectory as benchmarked (MD
    in FP32 on 12-real links, heatbath and Metropolis in FP64): its Delta H
    within 1e-9 of the FP64 recomputation of the same endpoints at 1e-13."""
    dims, mass, beta, n_pf, order = (32, 32, 32, 8), 0.01, 5.6, 8, 16
    lat = fields.Lattice(*dims)
    U = fields.random_links(lat, 3208, 0.3)
    first, md, last = rhmc_approximations(2, n_pf, order, order, order)
    say("C4", dims)
    g = Gpu(dims, mass=mass, beta=beta, n_pf=n_pf, max_order=order)
    g.init0(U)
    mn, mx = measured_bounds(g, mass)
    _, _, b, _ = last.rescaled(mn, mx, -2.0 / 4 / n_pf)
    b = np.array(b)
    phi = fields.gauss_spinor(lat, 9, n_pf)
    bn = np.linalg.norm(phi.reshape(n_pf, -1), axis=1)
    sols = []
    for precision in (0, 1):
        g.init1(phi=phi)
        it = g.multishift(b, 1e-10, relative=True, precision=precision)
        res = g.shifted_residuals(b) / bn[:, None]
        say("C4 precision", precision, "iterations", it, g.solve_stats(), g.solver_counters(),
            "worst true residual", res.max())
        assert np.all(res <= 1e-10), res.max()
        sols.append(g.get_fermions("smf"))
    assert rel(sols[1], sols[0]) < 1e-7
    co = dict(first=(first.a0, first.a, first.b), md=(md.a0, md.a, md.b), last=(last.a0, last.a, last.b))
    r = g.trajectory(precision=1, fp32_threshold=1e-7, n_flavours=2, no_md=10, integrator="omelyan",
                     res_md=1e-6, res_metro=1e-10, relative=True, bounds=(mn, mx), draw_fields=True, seed=77,
                     verify_fp64=True, verify_res=1e-13, **co)
    err = abs(r.delta_h - r.delta_h_fp64)
    say("C4 trajectory", r.seconds_total, "s dH", r.delta_h, "dH(FP64 1e-13)", r.delta_h_fp64, "error", err)
    assert err <= 1e-9
    g.close()


def test_c4_refined_metropolis_is_variational():
    """C4 trajectory with the Metropolis solve as FP32 iterations + FP64
    defect correction (metro_precision=2, heatbath FP64).  The refined
    solutions are not Galerkin, so each pole term is taken as
    Re<chi, x> + Re<x, r> (r the FP64 true residual), whose error is
    quadratic in the solution's: Delta H within 1e-9 of the FP64
    recomputation at 1e-13.  The correction itself is nonzero, and zero
    with the FP64 Metropolis solve (metro_precision=0)."""
    dims, mass, beta, n_pf, order = (32, 32, 32, 8), 0.01, 5.6, 8, 16
    lat = fields.Lattice(*dims)
    U = fields.random_links(lat, 3208, 0.3)
    first, md, last = rhmc_approximations(2, n_pf, order, order, order)
    g = Gpu(dims, mass=mass, beta=beta, n_pf=n_pf, max_order=order)
    g.init0(U)
    mn, mx = measured_bounds(g, mass)
    co = dict(first=(first.a0, first.a, first.b), md=(md.a0, md.a, md.b), last=(last.a0, last.a, last.b))
    kw = dict(precision=1, fp32_threshold=1e-7, n_flavours=2, no_md=10, integrator="omelyan", res_md=1e-6,
              res_metro=1e-10, relative=True, bounds=(mn, mx), draw_fields=True, seed=78, verify_fp64=True,
              verify_res=1e-13, **co)
    out = {}
    for mp in (0, 2):
        g.init0(U)
        r = g.trajectory(metro_precision=mp, **kw)
        err = abs(r.delta_h - r.delta_h_fp64)
        lin = abs(r.delta_h - r.metro_correction - r.delta_h_fp64)
        say("C4 metro_precision", mp, "dH", r.delta_h, "error", err, "without the correction", lin,
            "correction", r.metro_correction, "iterations", r.cg_iterations, "s", r.seconds_total)
        out[mp] = (r, err)
    assert out[0][0].metro_correction == 0.0
    assert out[2][0].metro_correction != 0.0
    assert out[2][1] <= 1e-9
    # same fields, same MD: the two Delta H agree to the Metropolis accuracy
    assert abs(out[2][0].delta_h - out[0][0].delta_h) <= 2e-9
    g.close()


@pytest.mark.parametrize("precision", [0, 1])
def test_c4b_six_uneven_lattices_in_lockstep(precision):
    """C4's six independent lattices (8^4, 12^4 x2, 16^4 x2, 8^3x16), Omelyan
    10 steps, 12/8/12 poles, each its own seed and bounds, advanced in
    lockstep by gpu_multi_trajectory (one launch per solver step over every
    lattice's tiles, solver chunks replayed as HIP graphs).  Each lattice's
    trajectory matches the one it runs alone from the same start: with FP64
    solves Delta H to 1e-9 and links to 1e-10; with the mixed dispatch (FP32
    MD solves, whose rounding depends on the launch shape) Delta H to
    1e-4 max(1, |Delta H|) and links to 1e-5.  Two lockstep runs from the
    same start are identical bit for bit."""
    lats = [(8, 8, 8, 8), (12, 12, 12, 12), (12, 12, 12, 12), (16, 16, 16, 16), (16, 16, 16, 16), (8, 8, 8, 16)]
    mass, beta = 0.01, 5.6
    first, md, last = rhmc_approximations(2, 1, 12, 8, 12)
    co = dict(first=(first.a0, first.a, first.b), md=(md.a0, md.a, md.b), last=(last.a0, last.a, last.b))
    gpus, starts, kws = [], [], []
    for i, d in enumerate(lats):
        lat = fields.Lattice(*d)
        U = fields.random_links(lat, 900 + i, 0.3)
        g = Gpu(d, mass=mass, beta=beta, n_pf=1, max_order=12)
        g.init0(U)
        mn, mx = measured_bounds(g, mass)
        gpus.append(g)
        starts.append(U)
        kws.append(dict(n_flavours=2, no_md=10, integrator="omelyan", res_md=1e-6 if precision else 1e-10,
                        res_metro=1e-10, relative=True, bounds=(mn, mx), draw_fields=True, precision=precision,
                        fp32_threshold=1e-7, seed=40 + i, **co))
    alone = []
    for g, U, kw in zip(gpus, starts, kws):
        g.init0(U)
        r = g.trajectory(**kw)
        Ua, _, _ = g.end(links=True, ipdot=False, momenta=False)
        alone.append((r.delta_h, Ua))
    runs = []
    for rep in range(2):
        for g, U in zip(gpus, starts):
            g.init0(U)
        say("C4b lockstep", precision, rep)
        res, st = multi_trajectory(gpus, kws)
        assert st == [0] * len(lats)
        runs.append([(r.delta_h, g.end(links=True, ipdot=False, momenta=False)[0], r.seconds_total)
                     for g, r in zip(gpus, res)])
    for (dh, Uc, sec), (dh2, Uc2, _), (dha, Ua), d in zip(runs[0], runs[1], alone, lats):
        say("C4b", d, "dH", dh, "alone", dh2, dha, "s", sec)
        assert dh == dh2 and np.array_equal(Uc, Uc2)
        if precision == 0:
            assert abs(dh - dha) < 1e-9
            assert rel(Uc, Ua) < 1e-10
        else:
            assert abs(dh - dha) < 1e-4 * max(1.0, abs(dha))
            assert rel(Uc, Ua) < 1e-5
    for g in gpus:
        g.close()


def test_lockstep_first_on_fresh_handles():
    """Handles whose first solve ever is a lockstep one (the launch shapes of
    the group are timed before any lattice has iterated alone) give each
    lattice the trajectory it runs alone on another handle: Delta H to 1e-9,
    links to 1e-10 (FP64 solves)."""
    lats = [(8, 8, 8, 4), (6, 4, 4, 6), (16, 8, 8, 8)]
    first, md, last = rhmc_approximations(2, 1, 12, 8, 12)
    co = dict(first=(first.a0, first.a, first.b), md=(md.a0, md.a, md.b), last=(last.a0, last.a, last.b))

    def handles():
        out = []
        for i, d in enumerate(lats):
            g = Gpu(d, mass=0.05, beta=5.6, n_pf=1, max_order=12)
            g.init0(fields.random_links(fields.Lattice(*d), 70 + i, 0.3))
            out.append(g)
        return out

    kws = [dict(n_flavours=2, no_md=2, integrator="omelyan", res_md=1e-10, res_metro=1e-10, relative=True,
                bounds=(0.02, 5.6), draw_fields=True, seed=50 + i, **co) for i in range(len(lats))]
    together, single = handles(), handles()
    say("lockstep on fresh handles", lats)
    res, st = multi_trajectory(together, kws)
    assert st == [0] * len(lats)
    for g, s, r, kw in zip(together, single, res, kws):
        ra = s.trajectory(**kw)
        assert abs(r.delta_h - ra.delta_h) < 1e-9
        assert rel(g.end(ipdot=False, momenta=False)[0], s.end(ipdot=False, momenta=False)[0]) < 1e-10
        g.close()
        s.close()


@pytest.mark.parametrize("lats", [[((8, 8, 8, 4), 8)] * 12, [((16, 16, 16, 16), 1)] + [((8, 8, 8, 4), 8)] * 3],
                         ids=["twelve_of_8", "one_and_three_of_8"])
def test_lockstep_of_more_systems_than_one_launch_lists(lats):
    """Groups with more right-hand sides (96; 25) than the argument table of a
    one-launch solve has members, which the CUs would have room for: each
    lattice gets the trajectory it runs alone, Delta H to 1e-9 max(1, |Delta
    H|) (one MD step: |Delta H| of 8 10^4), links to 1e-10 (FP64 solves)."""
    kws, gpus, starts = [], [], []
    for i, (d, n_pf) in enumerate(lats):
        order = (16, 16, 16) if n_pf == 8 else (12, 8, 12)
        first, md, last = rhmc_approximations(2, n_pf, *order)
        g = Gpu(d, mass=0.05, beta=5.6, n_pf=n_pf, max_order=16)
        starts.append(fields.random_links(fields.Lattice(*d), 170 + i, 0.3))
        gpus.append(g)
        kws.append(dict(n_flavours=2, no_md=1, integrator="omelyan", res_md=1e-10, res_metro=1e-10, relative=True,
                        bounds=(0.02, 5.6), draw_fields=True, seed=90 + i, first=(first.a0, first.a, first.b),
                        md=(md.a0, md.a, md.b), last=(last.a0, last.a, last.b)))
    say("lockstep of many systems", len(lats), sum(n for _, n in lats))
    alone = []
    for g, U, kw in zip(gpus, starts, kws):
        g.init0(U)
        r = g.trajectory(**kw)
        alone.append((r.delta_h, g.end(ipdot=False, momenta=False)[0]))
        g.init0(U)
    say("alone done")
    res, st = multi_trajectory(gpus, kws)
    assert st == [0] * len(lats)
    for g, r, (dh, U) in zip(gpus, res, alone):
        assert abs(r.delta_h - dh) < 1e-9 * max(1.0, abs(dh))
        assert rel(g.end(ipdot=False, momenta=False)[0], U) < 1e-10
        g.close()


# ------------------------------------------------------------------ C5
def test_c5_48c12_trajectory_delta_h():
    """C5: 48^3x12, Nf=2, am=0.01, beta=5.6, 2 pseudofermions, Omelyan 20
    steps, 16 MD / 20 heatbath and Metropolis poles, exp(i 0.3 H) links, one
    mixed trajectory (MD FP32, heatbath/Metropolis FP64 at 1e-12): Delta H
    within 1e-9 of the FP64 recomputation of the same endpoints at 1e-13."""
    dims, mass, beta, n_pf = (48, 48, 48, 12), 0.01, 5.6, 2
    lat = fields.Lattice(*dims)
    U = fields.random_links(lat, 4812, 0.3)
    first, md, last = rhmc_approximations(2, n_pf, 20, 16, 20)
    co = dict(first=(first.a0, first.a, first.b), md=(md.a0, md.a, md.b), last=(last.a0, last.a, last.b))
    say("C5", dims)
    g = Gpu(dims, mass=mass, beta=beta, n_pf=n_pf, max_order=20)
    g.init0(U)
    mn, mx = measured_bounds(g, mass)
    r = g.trajectory(precision=1, fp32_threshold=1e-7, n_flavours=2, no_md=20, integrator="omelyan", res_md=1e-6,
                     res_metro=1e-12, relative=True, bounds=(mn, mx), draw_fields=True, seed=4000,
                     verify_fp64=True, verify_res=1e-13, **co)
    err = abs(r.delta_h - r.delta_h_fp64)
    say("C5 trajectory", r.seconds_total, "s dH", r.delta_h, "error", err, "iterations", r.cg_iterations)
    assert err <= 1e-9
    assert np.isfinite(r.delta_h)
    g.close()


# ------------------------------------------------- spectral bounds
def _dense_gpu_mdagm(g, lat, mass):
    """M^dag M = m^2 - D_eo D_oe assembled column by column from the device
    Dslash (FP64 18-real links)."""
    n = 3 * lat.Vh
    E = np.eye(n, dtype=np.complex128).reshape(n, lat.Vh, 3)
    h = g.dslash(1, E, 0)
    s = g.dslash(0, h, 0)
    M = mass * mass * np.eye(n) - s.reshape(n, n).T
    return M


def test_power_method_against_dense_spectrum():
    """gpu_find_max / gpu_find_min (findminmax.cc:12-183) on 4^4 exp(i 0.3 H)
    links at a tight tolerance reach the extreme eigenvalues of the dense
    device operator within 1e-9 of the largest (a lattice whose lowest
    eigenvalues are separated enough for the shifted power method to
    converge in ~4000 steps); on 8^3x4 they agree with the oracle's power
    method from the same start vector (the device draw, restated on the
    host) to 10x the tolerance."""
    dims, mass = (4, 4, 4, 4), 0.1
    lat = fields.Lattice(*dims)
    U = fields.random_links(lat, 5, 0.3)
    g = Gpu(dims, mass=mass)
    g.init0(U)
    M = _dense_gpu_mdagm(g, lat, mass)
    assert np.abs(M - M.conj().T).max() < 1e-13
    ev = np.linalg.eigvalsh(M)
    mx = g.find_max(1e-14, seed=3)
    mn = g.find_min(mx, 1e-14, seed=4)
    say("dense", ev[0], ev[-1], "power", mn, mx)
    assert abs(mx - ev[-1]) < 1e-9 * ev[-1]
    assert abs(mn - ev[0]) < 1e-9 * ev[-1]
    g.close()

    dims = (8, 8, 8, 4)
    lat = fields.Lattice(*dims)
    U = fields.random_links(lat, 31, 0.3)
    g = Gpu(dims, mass=0.05)
    g.init0(U)
    o = Oracle(dims)
    tol = 1e-8
    mx = g.find_max(tol, seed=5)
    mn = g.find_min(mx, tol, seed=6)
    # gpu_find_max / gpu_find_min draw their start on the device: stream 7 / 8
    mxo, _ = o.findmaxeig(U, 0.05, rng.spinors(lat.Vh, 1, 5, 7)[0], tol)
    mno, _ = o.findmineig(U, 0.05, rng.spinors(lat.Vh, 1, 6, 8)[0], mx, tol)
    say("power 8^3x4", mn, mx, "oracle", mno, mxo)
    assert abs(mx - mxo) < 10 * tol * mxo
    assert abs(mn - mno) < 10 * tol * mx
    g.close()


def test_free_field_dense_spectrum():
    """U = eta 1 on 4^4: the dense device M^dag M has the eigenvalues
    m^2 + sum_mu sin^2 p_mu (periodic x, y, z; antiperiodic t), each with
    half of its full-lattice multiplicity on the even sites (the closed form
    the oracle is pinned to)."""
    dims, mass = (4, 4, 4, 4), 0.1
    lat = fields.Lattice(*dims)
    U = np.ascontiguousarray(np.eye(3)[None] * lat.eta()[:, None, None]).astype(np.complex128)
    g = Gpu(dims, mass=mass)
    g.init0(U)
    ev = np.linalg.eigvalsh(_dense_gpu_mdagm(g, lat, mass))
    g.close()
    px = 2 * np.pi * np.arange(4) / 4
    pt = (2 * np.arange(4) + 1) * np.pi / 4
    lam = mass ** 2 + (np.sin(px)[:, None, None, None] ** 2 + np.sin(px)[None, :, None, None] ** 2
                       + np.sin(px)[None, None, :, None] ** 2 + np.sin(pt)[None, None, None, :] ** 2)
    vals, counts = np.unique(np.round(ev, 10), return_counts=True)
    evals, ecounts = np.unique(np.round(np.repeat(lam.ravel(), 3), 10), return_counts=True)
    assert np.allclose(vals, evals, atol=1e-10)
    assert np.all(counts * 2 == ecounts)
    assert ev.min() > mass ** 2 + 0.4


# ------------------------------------------------------ device Gaussians
def test_device_gaussians_against_host_restatement():
    """gpu_gauss_momenta / gpu_gauss_phi (Philox4x32-10, Box-Muller, the
    su(3) layout of gauss.cc:63-86) equal the host restatement oracle/rng.py
    (pinned to Random123's known answers) to 1e-14, for several seeds and
    streams; at 16^4 the device draws have the reference's normalisation:
    Re and Im N(0, 1/2), P hermitian and traceless, <1/2 tr P^2> = 4."""
    dims = (8, 8, 8, 4)
    lat = fields.Lattice(*dims)
    g = Gpu(dims, mass=0.1, n_pf=3)
    for seed, stream in ((1, 0), (12345678901, 5)):
        g.gauss_momenta(seed, stream)
        _, _, P = g.end(links=False, ipdot=False, momenta=True)
        assert np.abs(P - rng.momenta(lat.Vh, seed, stream)).max() < 1e-14
        g.gauss_phi(seed, stream + 1)
        phi = g.get_fermions("phi")
        assert np.abs(phi - rng.spinors(lat.Vh, 3, seed, stream + 1)).max() < 1e-14
    g.close()
    dims = (16, 16, 16, 16)
    lat = fields.Lattice(*dims)
    g = Gpu(dims, mass=0.1, n_pf=2)
    g.gauss_momenta(99, 0)
    _, _, P = g.end(links=False, ipdot=False, momenta=True)
    g.gauss_phi(99, 1)
    phi = g.get_fermions("phi")
    g.close()
    assert np.abs(P - np.conj(np.swapaxes(P, 1, 2))).max() < 1e-15
    assert np.abs(np.trace(P, axis1=1, axis2=2)).max() < 1e-14
    half_tr = 0.5 * np.einsum("nij,nji->n", P, P).real
    n = len(half_tr)
    assert abs(half_tr.mean() - 4.0) < 5 * np.sqrt(4.0 / n)
    z = phi.ravel()
    for x in (z.real, z.imag):
        assert abs(x.mean()) < 5 * np.sqrt(0.5 / len(x))
        assert abs(x.var() - 0.5) < 5 * 0.5 * np.sqrt(2.0 / len(x))


# ------------------------------------------------------ reversibility
@pytest.mark.parametrize("mode", ["fp32_md", "fp64"])
def test_reversibility(mode):
    """rev_update (revupdate.cc:19-97) on 8^3x4, Omelyan 10 steps: forward,
    momenta reversed, back.  With FP64 solves at 1e-12 the return is exact
    to 1e-9 per degree of freedom; the benchmarked FP32 MD solves (relative
    residual 1e-6, FP32 12-real links, FP32 force input) depart by at most
    1e-4."""
    gd = dict(np.load(os.path.join(GOLD, "golden_c1.npz")))
    dims = tuple(int(x) for x in gd["dims"])
    lat = fields.Lattice(*dims)
    U = fields.random_links(lat, 31, 0.3)
    g = Gpu(dims, mass=0.05, beta=5.5, n_pf=1, max_order=12)
    g.init0(U)
    mn, mx = measured_bounds(g, 0.05)
    co = dict(first=(float(gd["first_a0"]), gd["first_a"], gd["first_b"]),
              md=(float(gd["md_a0"]), gd["md_a"], gd["md_b"]),
              last=(float(gd["last_a0"]), gd["last_a"], gd["last_b"]))
    if mode == "fp64":
        kw = dict(precision=0, res_md=1e-12, res_metro=1e-12)
        bound = 1e-9
    else:
        kw = dict(precision=1, fp32_threshold=1e-7, res_md=1e-6, res_metro=1e-10)
        bound = 1e-4
    dc, dm, r = g.rev_update(n_flavours=2, no_md=10, integrator="omelyan", relative=True, bounds=(mn, mx),
                             draw_fields=True, seed=21, **kw, **co)
    say("reversibility", mode, "dconf/dof", dc, "dmom/dof", dm, "iterations", r.cg_iterations)
    assert 0.0 <= dc < bound and 0.0 <= dm < bound
    g.close()


# ---------------------------------------------------- failure statuses
def _solve_status(g, b, precision, max_cg=100000):
    try:
        g.multishift(b, 1e-5 if precision == 2 else 1e-10, relative=True, precision=precision, max_cg=max_cg)
        return 0
    except RhmcError as e:
        return e.rc


@pytest.mark.parametrize("precision", [0, 1, 2])
def test_nonfinite_links_and_max_cg(precision, monkeypatch):
    """A NaN in one link stops every solver form with RHMC_ENONFINITE (the
    reference would iterate on NaN to max_cg); max_cg below the iterations
    needed returns RHMC_EMAXCG (cu_inverter.cc:62-69 exits instead).  Both
    for the stored-basis and the explicit-shift solvers; a trajectory on
    NaN links returns RHMC_ENONFINITE."""
    dims, mass = (8, 8, 8, 4), 0.05
    lat = fields.Lattice(*dims)
    U = fields.random_links(lat, 5, 0.3)
    phi = fields.gauss_spinor(lat, 6, 2)
    b = np.geomspace(1e-4, 1.0, 6)
    for explicit in (False, True):
        if explicit:
            monkeypatch.setenv("RHMC_MS_EXPLICIT", "1")
        g = Gpu(dims, mass=mass, n_pf=2, max_order=6)
        g.init0(U)
        g.init1(phi=phi)
        assert _solve_status(g, b, precision=precision) == 0
        assert _solve_status(g, b, precision=precision, max_cg=24) == RHMC_EMAXCG
        Ubad = U.copy()
        Ubad[123, 1, 2] = np.nan
        g.init0(Ubad)
        g.init1(phi=phi)
        assert _solve_status(g, b, precision=precision) == RHMC_ENONFINITE
        g.close()
        monkeypatch.delenv("RHMC_MS_EXPLICIT", raising=False)
    g = Gpu(dims, mass=mass, n_pf=1, max_order=12)
    g.init0(Ubad)
    gd = dict(np.load(os.path.join(GOLD, "golden_c1.npz")))
    co = dict(first=(float(gd["first_a0"]), gd["first_a"], gd["first_b"]),
              md=(float(gd["md_a0"]), gd["md_a"], gd["md_b"]),
              last=(float(gd["last_a0"]), gd["last_a"], gd["last_b"]))
    with pytest.raises(RhmcError) as e:
        g.trajectory(precision=precision if precision < 2 else 1, n_flavours=2, no_md=2, res_md=1e-6,
                     res_metro=1e-10, relative=True, bounds=(0.01, 5.0), draw_fields=True, **co)
    assert e.value.rc == RHMC_ENONFINITE
    g.close()


def test_trajectory_rejects_bad_metro_precision():
    """metro_precision outside 0-2 is RHMC_EINVAL with a message, before any
    work is done."""
    dims = (4, 4, 4, 4)
    lat = fields.Lattice(*dims)
    g = Gpu(dims, mass=0.1, n_pf=1, max_order=12)
    g.init0(fields.random_links(lat, 5, 0.3))
    gd = dict(np.load(os.path.join(GOLD, "golden_c1.npz")))
    co = dict(first=(float(gd["first_a0"]), gd["first_a"], gd["first_b"]),
              md=(float(gd["md_a0"]), gd["md_a"], gd["md_b"]),
              last=(float(gd["last_a0"]), gd["last_a"], gd["last_b"]))
    with pytest.raises(RhmcError) as e:
        g.trajectory(precision=1, metro_precision=3, n_flavours=2, no_md=2, res_md=1e-6, res_metro=1e-10,
                     relative=True, bounds=(0.01, 5.0), draw_fields=True, **co)
    assert e.value.rc == RHMC_EINVAL and "metro_precision" in str(e.value)
    g.close()


def test_links_must_be_unitary():
    """The 12-real link copies rebuild row 2 as eta (row 0 x row 1)^*, which
    reproduces only unitary links, so gpu_init0 refuses links that differ
    from that by more than 1e-10: RHMC_EINVAL naming the deviation, and the
    device keeps its previous links.  A rounding-level deviation passes."""
    dims = (8, 8, 8, 4)
    lat = fields.Lattice(*dims)
    U = fields.random_links(lat, 5, 0.3)
    g = Gpu(dims, mass=0.1)
    g.init0(U)
    bad = U.copy()
    bad[77, 2, 1] += 3e-7
    with pytest.raises(RhmcError) as e:
        g.init0(bad)
    say("refused:", str(e.value))
    assert e.value.rc == RHMC_EINVAL and "not unitary" in str(e.value) and "3e-07" in str(e.value)
    U1, _, _ = g.end(links=True, ipdot=False, momenta=False)
    assert np.array_equal(U1, U)
    ok = U.copy()
    ok[77, 2, 1] += 1e-13
    g.init0(ok)
    U2, _, _ = g.end(links=True, ipdot=False, momenta=False)
    assert np.array_equal(U2, ok)
    g.close()


# --------------------------------------------------- basis continuation
@pytest.mark.parametrize("precision", [0, 1, 2])
def test_basis_continuation_with_small_capacity(precision, monkeypatch):
    """A stored basis of 24 slots for solves needing ~100 iterations: each
    solve continues from its last residual (collinear shifted residuals)
    several times instead of restarting from zero; FP64 and mixed reach
    every shifted true residual <= 1e-10 |b| and the oracle's solutions to
    1e-9, the FP32 solver its own FP32 level (2e-5) and 5e-4."""
    dims, mass = (8, 8, 8, 4), 0.05
    lat = fields.Lattice(*dims)
    U = fields.random_links(lat, 21, None)
    phi = fields.gauss_spinor(lat, 22, 2)
    b = np.geomspace(1e-5, 1.5, 12) * (4.0 + mass * mass)
    monkeypatch.setenv("RHMC_BASIS_CAP", "24")
    g = Gpu(dims, mass=mass, n_pf=2, max_order=12)
    g.init0(U)
    g.init1(phi=phi)
    res_target = 1e-6 if precision == 2 else 1e-10
    it = g.multishift(b, res_target, relative=True, precision=precision)
    restarts, captures, worst = g.solver_counters()
    res = g.shifted_residuals(b)
    x = g.get_fermions("smf").reshape(2, 12, lat.Vh, 3)
    g.close()
    bn = np.linalg.norm(phi.reshape(2, -1), axis=1)
    say("continuation", precision, "iterations", it, "continuations", restarts, "worst", (res / bn[:, None]).max())
    assert restarts >= 2
    assert np.all(res / bn[:, None] <= (2e-5 if precision == 2 else 1e-10))
    o = Oracle(dims)
    for ps in range(2):
        xo, _ = o.multishift(U, mass, phi[ps], b, 1e-12 * bn[ps])
        for k in range(12):
            assert rel(x[ps, k], xo[k]) < (5e-4 if precision == 2 else 1e-9), (ps, k)


def test_graph_capture_once_per_solve_shape():
    """Solver chunks replayed as HIP graphs: repeated solves with the same
    arguments reuse the captured graph.  The second solve may capture once
    more, because the basis capacity adapts to the iterations the first one
    needed (a launch argument); from then on no solve recaptures, and every
    solve returns the same solutions bit for bit."""
    dims, mass = (8, 8, 8, 4), 0.05
    lat = fields.Lattice(*dims)
    U = fields.random_links(lat, 8, 0.3)
    phi = fields.gauss_spinor(lat, 9, 2)
    b = np.geomspace(1e-4, 1.0, 8)
    g = Gpu(dims, mass=mass, n_pf=2, max_order=8)
    g.init0(U)
    counts, sols = [], []
    for _ in range(5):
        g.init1(phi=phi)
        g.multishift(b, 1e-10, relative=True, precision=0)
        counts.append(g.solver_counters()[1])
        sols.append(g.get_fermions("smf"))
    g.close()
    say("graph captures after each solve", counts)
    assert counts[0] <= 1 and counts[1] <= counts[0] + 1
    assert counts[4] == counts[1]
    for x in sols[1:]:
        assert np.array_equal(x, sols[0])


# ----------------------------------------- small lattices: one-launch solves
@pytest.mark.parametrize("dims,n_pf", [((4, 4, 4, 4), 1), ((6, 4, 4, 6), 3), ((6, 6, 6, 6), 1), ((6, 6, 6, 6), 2),
                                       ((8, 8, 8, 4), 8), ((20, 14, 12, 6), 2), ((20, 14, 12, 6), 4),
                                       ((16, 16, 16, 16), 1), ((16, 16, 16, 16), 3), ((18, 16, 16, 16), 1),
                                       ((24, 24, 24, 8), 1)])
def test_one_launch_solves(dims, n_pf, monkeypatch):
    """Multi-shift solves whose iterations run as one launch, over the forms
    that launch takes: one workgroup and a partly filled one, systems split
    over members and together (1, 2, 4 per member), odd V/16 (slots that are no
    whole cache lines in FP32 for an odd number of systems), 256 and 512
    lanes, two sites per lane.  FP64 solutions agree with the launches per
    iteration (RHMC_DSLASH_NR set) to 1e-9, the true residuals meet 1e-10 |b|;
    FP32 ones to 2e-4 and 2e-5 (both stop at 1e-6, on recurrences that round
    differently); iteration counts are the same in FP64, a repeated solve is
    the same bit for bit."""
    mass = 0.05
    lat = fields.Lattice(*dims)
    U = fields.random_links(lat, 31, 0.3)
    phi = fields.gauss_spinor(lat, 32, n_pf)
    b = np.geomspace(1e-4, 2.0, 7)
    bn = np.linalg.norm(phi.reshape(n_pf, -1), axis=1)
    say("one-launch solve", dims, n_pf)
    out = {}
    for mode in ("one", "many"):
        if mode == "many":
            monkeypatch.setenv("RHMC_DSLASH_NR", "1")
        g = Gpu(dims, mass=mass, n_pf=n_pf, max_order=7)
        g.init0(U)
        g.init1(phi=phi)
        for prec, res in ((0, 1e-10), (2, 1e-6)):
            # the first solve may fill the initial basis, after which its
            # capacity follows the iterations needed
            g.multishift(b, res, relative=True, precision=prec)
            it = g.multishift(b, res, relative=True, precision=prec)
            x = g.get_fermions("smf")
            rn = g.shifted_residuals(b) / bn[:, None]
            assert rn.max() <= (1e-10 if prec == 0 else 2e-5)
            g.multishift(b, res, relative=True, precision=prec)
            assert np.array_equal(g.get_fermions("smf"), x)
            out[mode, prec] = (it, x)
        g.close()
    assert out["one", 0][0] == out["many", 0][0]
    for prec, tol in ((0, 1e-9), (2, 2e-4)):
        for x, y in zip(out["one", prec][1], out["many", prec][1]):
            assert rel(x, y) < tol


@pytest.mark.parametrize("dims,n_pf,n_shift", [((4, 4, 4, 4), 1, 1), ((8, 8, 8, 4), 3, 7), ((6, 10, 14, 6), 2, 5),
                                               ((16, 16, 16, 16), 4, 24), ((24, 24, 24, 8), 1, 9)])
def test_defect_correction_on_the_stored_basis(dims, n_pf, n_shift, monkeypatch):
    """Mixed-precision solves, whose systems are corrected as right-hand sides
    with an operator each: in one launch (few workgroups), in two launches per
    iteration, with a last chunk that is not full, and in two batches (96
    systems of 16^4).  Every true residual meets 1e-10 |b|; the solutions are
    the FP64 solver's to 1e-9, as are those of the correction without a basis
    (explicit shifts).  A second solve is the third bit for bit (the capacity
    follows the first)."""
    mass = 0.05
    lat = fields.Lattice(*dims)
    U = fields.random_links(lat, 41, 0.3)
    phi = fields.gauss_spinor(lat, 42, n_pf)
    b = np.geomspace(1e-4, 2.0, n_shift) if n_shift > 1 else np.array([1e-3])
    bn = np.linalg.norm(phi.reshape(n_pf, -1), axis=1)
    say("defect correction", dims, n_pf, n_shift)
    g = Gpu(dims, mass=mass, n_pf=n_pf, max_order=n_shift)
    g.init0(U)
    g.init1(phi=phi)
    g.multishift(b, 1e-11, relative=True, precision=0)
    exact = g.get_fermions("smf")
    for explicit in (True, False):
        if explicit:
            monkeypatch.setenv("RHMC_MS_EXPLICIT", "1")
        else:
            monkeypatch.delenv("RHMC_MS_EXPLICIT")
        g.multishift(b, 1e-10, relative=True, precision=1)
        assert (g.shifted_residuals(b) / bn[:, None]).max() <= 1e-10
        x = g.get_fermions("smf")
        for p, q in zip(x, exact):
            assert rel(p, q) < 1e-9, explicit
    g.multishift(b, 1e-10, relative=True, precision=1)
    y = g.get_fermions("smf")
    g.multishift(b, 1e-10, relative=True, precision=1)
    assert np.array_equal(g.get_fermions("smf"), y)
    g.close()


@pytest.mark.parametrize("precision", [0, 2])
def test_one_launch_solve_that_gives_up(precision, monkeypatch):
    """A one-launch solve whose waits are bounded at 0 ticks leaves (every
    workgroup exits) and the solve is repeated with the launches per
    iteration: the same status and solutions as without it."""
    dims, mass = (16, 16, 16, 16), 0.05
    lat = fields.Lattice(*dims)
    U = fields.random_links(lat, 33, 0.3)
    phi = fields.gauss_spinor(lat, 34, 1)
    b = np.geomspace(1e-4, 2.0, 7)
    say("one-launch solve, no wait", precision)
    xs = []
    for wait in ("0", None):
        if wait is None:
            monkeypatch.delenv("RHMC_RESIDENT_WAIT")
        else:
            monkeypatch.setenv("RHMC_RESIDENT_WAIT", wait)
        g = Gpu(dims, mass=mass, n_pf=1, max_order=7)
        g.init0(U)
        g.init1(phi=phi)
        for _ in range(2):
            g.multishift(b, 1e-10 if precision == 0 else 1e-6, relative=True, precision=precision)
        xs.append(g.get_fermions("smf"))
        g.close()
    assert rel(xs[0], xs[1]) < (1e-9 if precision == 0 else 2e-4)


# members, right-hand sides per member, lanes and sites per lane in FP64 and FP32 (None: launches per iteration)
@pytest.mark.parametrize("dims,n_pf,forms", [
    ((4, 4, 4, 4), 1, [(1, 1, 256, 1)] * 2), ((6, 4, 4, 6), 3, [(3, 1, 256, 1)] * 2),
    ((6, 6, 6, 6), 1, [(1, 1, 256, 1), None]), ((6, 6, 6, 6), 2, [(2, 1, 256, 1), (1, 2, 256, 1)]),
    ((8, 8, 8, 4), 8, [(8, 1, 256, 1)] * 2), ((20, 14, 12, 6), 2, [(2, 1, 512, 1)] * 2),
    ((20, 14, 12, 6), 4, [(2, 2, 512, 1)] * 2), ((16, 16, 16, 16), 1, [(1, 1, 512, 1)] * 2),
    ((16, 16, 16, 16), 2, [(1, 2, 512, 1)] * 2), ((16, 16, 16, 16), 3, [(1, 4, 512, 1)] * 2),
    ((16, 16, 16, 16), 8, [None] * 2), ((18, 16, 16, 16), 1, [(1, 1, 512, 2)] * 2),
    ((24, 24, 24, 8), 1, [(1, 1, 512, 2)] * 2), ((24, 24, 24, 12), 1, [None] * 2)])
def test_one_launch_solves_take_their_form(dims, n_pf, forms, monkeypatch):
    """Which solves run their iterations as one launch on a device of 256
    compute units, and over how many members; none do with a forced launch
    shape.  (Whether their solutions are right: test_one_launch_solves.)"""
    lat = fields.Lattice(*dims)
    U = fields.random_links(lat, 35, 0.3)
    phi = fields.gauss_spinor(lat, 36, n_pf)
    say("form", dims, n_pf)
    for forced in (False, True):
        if forced:
            monkeypatch.setenv("RHMC_DSLASH_NR", "1")
        g = Gpu(dims, mass=0.1, n_pf=n_pf, max_order=2)
        g.init0(U)
        g.init1(phi=phi)
        for prec, form in zip((0, 2), forms):
            before = g.path_counters()["one_launch"]
            g.multishift([1e-2, 1.0], 1e-5, relative=True, precision=prec)
            c = g.path_counters()
            assert (c["one_launch"] > before) == (form is not None and not forced)
            if form and not forced:
                assert (c["members"], c["member_rhs"], c["lanes"], c["lane_sites"]) == form
        assert c["gave_up"] == 0
        g.close()


@pytest.mark.parametrize("precision", [0, 2])
def test_one_launch_work_that_does_not_wait_is_repeated(precision, monkeypatch):
    """A bound of 0 ticks: some workgroup finds an empty slot and gives up, the
    others follow and every one exits.  The solve, a lockstep solve of two
    lattices and the bounds are then repeated with the launches per iteration,
    each counted, with the results of an unbounded run (solutions 1e-9 in FP64,
    2e-4 in FP32; trajectories' links 1e-9; bounds 1e-11 of the largest)."""
    dims, mass = (16, 16, 16, 16), 0.1
    lat = fields.Lattice(*dims)
    U = fields.random_links(lat, 37, 0.3)
    phi = fields.gauss_spinor(lat, 38, 1)
    b = np.geomspace(1e-3, 2.0, 5)
    first, md, last = rhmc_approximations(2, 1, 6, 5, 6)
    kw = dict(n_flavours=2, no_md=1, integrator="omelyan", res_md=1e-10, res_metro=1e-10, relative=True,
              bounds=(0.02, 5.6), draw_fields=True, first=(first.a0, first.a, first.b), md=(md.a0, md.a, md.b),
              last=(last.a0, last.a, last.b))
    out = []
    for wait in ("0", None):
        if wait is None:
            monkeypatch.delenv("RHMC_RESIDENT_WAIT")
        else:
            monkeypatch.setenv("RHMC_RESIDENT_WAIT", wait)
        say("wait", wait, precision)
        g = Gpu(dims, mass=mass, max_order=6)
        g.init0(U)
        g.init1(phi=phi)
        g.multishift(b, 1e-10 if precision == 0 else 1e-6, relative=True, precision=precision)
        x = g.get_fermions("smf")
        c = g.path_counters()
        assert c["one_launch"] >= 1 and c["gave_up"] == (0 if wait is None else 1)
        g.close()
        say("solve done")
        g = Gpu(dims, mass=mass, max_order=6)
        g.init0(U)
        mx = g.find_max(1e-4, seed=3)
        c = g.path_counters()
        assert c["power"] == 1 and c["gave_up"] == (0 if wait is None else 1)
        say("bounds done")
        g.close()
        gs = [Gpu(d, mass=mass, max_order=6) for d in (dims, (8, 8, 8, 4))]
        links = []
        for i, h in enumerate(gs):
            h.init0(fields.random_links(fields.Lattice(*h.dims), 39 + i, 0.3))
        res, st = multi_trajectory(gs, [dict(seed=5 + i, **kw) for i in range(2)])
        assert st == [0, 0]
        c = gs[0].path_counters()
        assert c["one_launch"] >= 1 and c["gave_up"] == (0 if wait is None else 1)
        for h in gs:
            links.append(h.end(ipdot=False, momenta=False)[0])
            h.close()
        say("lockstep done")
        out.append((x, mx, links))
    (x0, m0, l0), (x1, m1, l1) = out
    assert rel(x0, x1) < (1e-9 if precision == 0 else 2e-4)
    assert abs(m0 - m1) < 1e-11 * m1
    assert all(rel(p, q) < 1e-9 for p, q in zip(l0, l1))


@pytest.mark.parametrize("dims", [(4, 4, 4, 4), (6, 4, 4, 6), (6, 6, 6, 6), (20, 14, 12, 6), (16, 16, 16, 16),
                                  (18, 16, 16, 16), (24, 24, 24, 12)])
def test_power_iterations_in_one_launch(dims, monkeypatch):
    """The power iterations of small lattices (64 per launch, one or two sites
    per lane; several launches each) stop at the same iteration as the two
    launches per iteration (RHMC_DSLASH_NR set; 24^3x12 always runs those):
    both bounds equal to 1e-11 of the largest eigenvalue, the rounding of
    a few hundred normalised applications (1e-16 each)."""
    lat = fields.Lattice(*dims)
    g = Gpu(dims, mass=0.05)
    g.init0(fields.random_links(lat, 41, 0.3))
    say("power iterations", dims)
    got = []
    for many in (False, True):
        if many:
            monkeypatch.setenv("RHMC_DSLASH_NR", "1")
        mx = g.find_max(1e-5, seed=5)
        got.append((mx, g.find_min(mx, 1e-5, seed=6)))
    say(got)
    assert abs(got[0][0] - got[1][0]) < 1e-11 * got[1][0]
    assert abs(got[0][1] - got[1][1]) < 1e-11 * got[1][0]
    g.close()


def test_one_launch_solves_of_several_threads():
    """Four handles, each in a thread of its own: two of 16^4, whose one-launch
    solves fill the device's workgroups one handle at a time, and two small
    ones, whose solves run beside each other.  Solutions and bounds are those
    of the handle working alone, bit for bit (every sum has a fixed order), and
    no solve gives up."""
    import threading
    mass, b = 0.05, np.geomspace(1e-4, 2.0, 7)
    handles = []
    for i, dims in enumerate([(16, 16, 16, 16), (8, 8, 8, 4), (16, 16, 16, 16), (6, 4, 4, 6)]):
        lat = fields.Lattice(*dims)
        g = Gpu(dims, mass=mass, n_pf=2, max_order=7)
        g.init0(fields.random_links(lat, 47 + i, 0.3))
        g.init1(phi=fields.gauss_spinor(lat, 57 + i, 2))
        handles.append(g)

    def work(g):
        g.multishift(b, 1e-10, relative=True, precision=0)
        x = g.get_fermions("smf")
        return x, g.find_max(1e-4, seed=9)

    say("threads")
    # the slots follow the iterations: settled after a few solves
    alone = [[work(g) for _ in range(4)][-1] for g in handles]
    ran = [g.path_counters()["one_launch"] for g in handles]
    err = []

    def thread(g, want):
        try:
            for _ in range(10):
                x, mx = work(g)
                assert np.array_equal(x, want[0]) and mx == want[1]
        except BaseException as e:  # reported by the main thread
            err.append(e)

    th = [threading.Thread(target=thread, args=a) for a in zip(handles, alone)]
    for t in th:
        t.start()
    for t in th:
        t.join()
    assert not err, err
    for g, n in zip(handles, ran):
        c = g.path_counters()
        assert c["one_launch"] >= n + 10 and c["power"] == 14 and c["gave_up"] == 0
        g.close()


def test_one_launch_solves_are_tried_again(monkeypatch):
    """After a solve that gave up, 256 solves use the launches per iteration;
    then one launch is tried again, and used from there on when it is let."""
    dims = (8, 8, 8, 4)
    lat = fields.Lattice(*dims)
    g = Gpu(dims, mass=0.5, max_order=1)
    g.init0(fields.random_links(lat, 45, 0.3))
    g.init1(phi=fields.gauss_spinor(lat, 46, 1))

    def solves(n):
        for _ in range(n):
            g.multishift([1.0], 1e-1, relative=True, precision=0)
        c = g.path_counters()
        return c["one_launch"], c["gave_up"]

    monkeypatch.setenv("RHMC_RESIDENT_WAIT", "0")
    say("gives up, rests")
    assert solves(1) == (1, 1)
    assert solves(256) == (1, 1)
    assert solves(1) == (2, 2)
    monkeypatch.delenv("RHMC_RESIDENT_WAIT")
    say("rests, then runs")
    assert solves(256) == (2, 2)
    assert solves(3) == (5, 2)
    g.close()


def test_one_launch_solve_takes_the_memory_its_iterations_need(monkeypatch):
    """The second set of slots of a one-launch solve: after a correction of 24
    systems has grown the handle's basis to 2.4 GB, solves of one system of
    16^4 take slots for at most twice their iterations (128 at least; 64 MB for
    the rest), and where those would be more than half of the free memory the
    launches per iteration.  Solutions agree with those of a fresh handle
    to 1e-9 (true residuals of 1e-10 |b|)."""
    import torch
    dims, mass = (16, 16, 16, 16), 0.05
    lat = fields.Lattice(*dims)
    U = fields.random_links(lat, 43, 0.3)
    phi = fields.gauss_spinor(lat, 44, 1)
    many, one = np.geomspace(1e-4, 2.0, 24), np.array([1e-3])
    vector = 48 * lat.Vh
    fresh = Gpu(dims, mass=mass, max_order=24)
    fresh.init0(U)
    fresh.init1(phi=phi)
    fresh.multishift(one, 1e-10, relative=True, precision=0)
    want = fresh.get_fermions("smf")
    fresh.close()
    g = Gpu(dims, mass=mass, max_order=24)
    g.init0(U)
    g.init1(phi=phi)
    g.multishift(many, 1e-10, relative=True, precision=1)
    say("basis grown")
    free = torch.cuda.mem_get_info()[0]
    monkeypatch.setenv("RHMC_FREE_BYTES", "1000000")
    before = g.path_counters()["one_launch"]
    g.multishift(one, 1e-10, relative=True, precision=0)
    assert g.path_counters()["one_launch"] == before
    assert rel(g.get_fermions("smf"), want) < 1e-9
    monkeypatch.delenv("RHMC_FREE_BYTES")
    for _ in range(4):
        it = g.multishift(one, 1e-10, relative=True, precision=0)
    assert g.path_counters()["one_launch"] > before
    assert rel(g.get_fermions("smf"), want) < 1e-9
    took = free - torch.cuda.mem_get_info()[0]
    say("iterations", it, "memory", took)
    assert took < max(128, 2 * it) * vector + (64 << 20)
    g.close()


@pytest.mark.parametrize("dims", [(4, 4, 4, 4), (16, 16, 16, 16), (24, 24, 24, 8)])
def test_power_iterations_without_room_for_their_slots(dims, monkeypatch):
    """Where the 129 vectors of the many-per-launch form would take more than
    half of the free device memory, the bounds run two launches per iteration
    on three vectors: the same bounds to 1e-11 of the largest, no error."""
    lat = fields.Lattice(*dims)
    U = fields.random_links(lat, 42, 0.3)
    vectors = 129 * 48 * lat.Vh
    say("power iterations, room", dims)
    got = []
    for room, taken in ((vectors, 0), (2 * vectors, 2)):
        monkeypatch.setenv("RHMC_FREE_BYTES", str(room))
        g = Gpu(dims, mass=0.05)
        g.init0(U)
        mx = g.find_max(1e-4, seed=5)
        got.append((mx, g.find_min(mx, 1e-4, seed=6)))
        assert g.path_counters()["power"] == taken
        g.close()
    for a, b in zip(*got):
        assert abs(a - b) < 1e-11 * got[0][0]


@pytest.mark.parametrize("dims,n_pf,n_shift", [((4, 4, 4, 4), 1, 1), ((6, 6, 4, 4), 3, 5), ((8, 8, 8, 4), 1, 17),
                                               ((8, 8, 8, 4), 2, 32), ((12, 10, 8, 6), 9, 4)])
def test_assembly_of_few_workgroups(dims, n_pf, n_shift):
    """Shifted solutions of lattices whose assembly has fewer workgroups than
    there are CUs (4 shifts per thread, a ragged last group), against the
    oracle to 1e-9 (residuals of 1e-11 |b|, the smallest eigenvalue 0.01)."""
    lat = fields.Lattice(*dims)
    U = fields.random_links(lat, 61, 0.3)
    phi = fields.gauss_spinor(lat, 62, n_pf)
    b = np.geomspace(1e-3, 2.0, n_shift) if n_shift > 1 else np.array([1e-2])
    say("assembly", dims, n_pf, n_shift)
    g = Gpu(dims, mass=0.1, n_pf=n_pf, max_order=n_shift)
    g.init0(U)
    g.init1(phi=phi)
    g.multishift(b, 1e-11, relative=True, precision=0)
    x = g.get_fermions("smf").reshape(n_pf, n_shift, lat.Vh, 3)
    g.close()
    o = Oracle(dims)
    for ps in range(n_pf):
        xo, _ = o.multishift(U, 0.1, phi[ps], b, 1e-12 * np.linalg.norm(phi[ps]))
        for k in range(n_shift):
            assert rel(x[ps, k], xo[k]) < 1e-9, (ps, k)


@pytest.mark.parametrize("dims,n_pf", [((40, 40, 40, 12), 2), ((48, 48, 48, 12), 1), ((64, 64, 64, 12), 2)])
def test_streamed_links(dims, n_pf, monkeypatch):
    """Lattices whose links exceed the Infinity Cache, where the launches of one
    or two systems stream the links of some directions (FP64 of 40^3x12 and
    48^3x12: three; FP32 of 48^3x12: two; 64^3x12: all).  Against the
    lane-split kernels, which stream none: FP64 solutions to 4e-8 (both have
    true residuals of 1e-10 |b|, eigenvalues in 0.09 .. 16.1), FP32 true
    residuals to 1e-4 |b|, the largest eigenvalue to 1e-11."""
    lat = fields.Lattice(*dims)
    say("streamed links", dims, n_pf)
    rng = np.random.default_rng(51)
    U = fields.haar_su3(rng, 4096)[rng.integers(0, 4096, 4 * lat.V)]
    U *= lat.eta()[:, None, None]
    phi = fields.gauss_spinor(lat, 52, n_pf)
    bn = np.linalg.norm(phi.reshape(n_pf, -1), axis=1)
    b = np.array([1e-3, 1.0])
    out = []
    for shape in (f"{n_pf}x4", f"{n_pf}"):
        monkeypatch.setenv("RHMC_DSLASH_NR", shape)
        g = Gpu(dims, mass=0.3, n_pf=n_pf, max_order=2)
        g.init0(U)
        g.init1(phi=phi)
        g.multishift(b, 1e-5, relative=True, precision=2)
        assert (g.shifted_residuals(b) / bn[:, None]).max() <= 1e-4
        g.multishift(b, 1e-10, relative=True, precision=0)
        assert (g.shifted_residuals(b) / bn[:, None]).max() <= 1e-10
        out.append((g.get_fermions("smf"), g.find_max(1e-3, seed=7)))
        g.close()
        say("done", shape)
    for x, y in zip(out[0][0], out[1][0]):
        assert rel(x, y) < 4e-8
    assert abs(out[0][1] - out[1][1]) < 1e-11 * out[0][1]


# ------------------------------------------------- large host transfers
@pytest.mark.parametrize("dims", [(8, 8, 8, 4), (16, 14, 12, 6), (18, 16, 14, 10), (32, 32, 16, 8)])
def test_host_transfers_round_trip(dims):
    """Links, momenta, force and pseudofermions go to the device and come back
    bit for bit, below and above the size that is moved in chunks (8 MB; the
    last chunk partly filled), also with two handles transferring from two
    threads at once."""
    import threading
    lat = fields.Lattice(*dims)
    say("transfers", dims)
    err = []

    def work(seed):
        try:
            U = fields.random_links(lat, seed, 0.3)
            P = fields.gauss_momenta(lat, seed + 1)
            F = 1j * fields.gauss_momenta(lat, seed + 2)
            phi = fields.gauss_spinor(lat, seed + 3, 2)
            g = Gpu(dims, mass=0.1, n_pf=2, max_order=2)
            for _ in range(2):
                g.init0(U)
                g.init1(phi=phi, ipdot=F, momenta=P)
                U1, F1, P1 = g.end()
                assert np.array_equal(U1, U)
                # packed as 8 reals: the third diagonal entry is rebuilt
                for a, b in ((P1, P), (F1, F)):
                    assert np.array_equal(a[:, 0, 1:], b[:, 0, 1:]) and np.array_equal(a[:, 1, 2], b[:, 1, 2])
                    assert np.abs(a - b).max() < 1e-14
                assert np.array_equal(g.get_fermions("mf"), phi)
            g.close()
        except Exception as e:  # reported by the main thread
            err.append(e)

    th = [threading.Thread(target=work, args=(60 + 10 * k,)) for k in range(2)]
    for t in th:
        t.start()
    for t in th:
        t.join()
    assert not err, err


def test_host_transfers_of_pinned_arrays():
    """Links of 75 MB from and to ordinary arrays go through the pinned chunks,
    from and to arrays that are pinned already directly; both come back bit
    for bit."""
    import ctypes as C

    import torch
    dims = (32, 32, 16, 8)
    lat = fields.Lattice(*dims)
    U = fields.random_links(lat, 75, 0.3)
    say("pinned transfers", dims)
    pin = torch.empty(U.size * 2, dtype=torch.float64, pin_memory=True).numpy()
    pin[:] = U.view(np.float64).ravel()
    g = Gpu(dims, mass=0.1)
    g.init0(U)
    staged = g.path_counters()["staged"]
    assert staged >= 1
    assert g.L.gpu_init0(g.h, pin.ctypes.data_as(C.c_void_p)) == 0
    pin[:] = 0.0
    assert g.L.gpu_end(g.h, pin.ctypes.data_as(C.c_void_p), None, None) == 0
    assert g.path_counters()["staged"] == staged
    assert np.array_equal(pin, U.view(np.float64).ravel())
    assert np.array_equal(g.end(ipdot=False, momenta=False)[0], U)
    assert g.path_counters()["staged"] == staged + 1
    g.close()


# ------------------------------------------------------------- gauge force
@pytest.mark.parametrize("dims,antiperiodic", [((2, 2, 2, 2), True), ((2, 4, 6, 8), True), ((8, 2, 4, 2), False),
                                               ((6, 6, 6, 6), True), ((16, 16, 16, 8), True), ((10, 8, 6, 4), False)])
def test_gauge_force_against_oracle(dims, antiperiodic):
    """The gauge force on extents of 2 (forward and backward neighbours
    coincide), partly filled and permuted tiles and both temporal boundary
    conditions, alone and added to a force: against the oracle's to 1e-13 (a
    staple is three rounded products of unitary matrices, 1e-15)."""
    lat = fields.Lattice(*dims, antiperiodic_t=antiperiodic)
    U = fields.random_links(lat, 71, None)
    F = 1j * fields.gauss_momenta(lat, 72)
    say("gauge force", dims, antiperiodic)
    g = Gpu(dims, mass=0.1, beta=5.7, antiperiodic_t=antiperiodic)
    g.init0(U)
    g.init1(ipdot=F)
    ref = Oracle(dims, antiperiodic).ipdot_total(U, 5.7)
    g.gauge_deriv(accumulate=True)
    added = g.end(links=False, momenta=False)[1] - F
    g.gauge_deriv()
    alone = g.end(links=False, momenta=False)[1]
    g.close()
    assert rel(alone, ref) < 1e-13
    assert rel(added, ref) < 1e-13


# ------------------------------------------------- loops and pairwise sums
@pytest.mark.parametrize("dims", [(2, 2, 2, 2), (4, 4, 4, 4), (6, 10, 4, 14), (14, 14, 14, 10), (18, 18, 18, 18),
                                  (32, 16, 16, 16)])
def test_loops_and_action_sums(dims):
    """Plaquettes, Polyakov loop and the action over site counts that the
    pairwise sums take by 5, 3 and 1 levels at a time, with an odd count above
    the last launch's size (18^4) and below it: against the oracle's loops to
    1e-13 and its action to 1e-12 of the sum of absolute values (each term is
    rounded at 1e-15, the sums are in the same order)."""
    lat = fields.Lattice(*dims)
    U = fields.random_links(lat, 81, 0.3)
    P = fields.gauss_momenta(lat, 82)
    say("loops", dims)
    o = Oracle(dims)
    g = Gpu(dims, mass=0.1, beta=5.7)
    g.init0(U)
    g.init1(momenta=P)
    for a, b in zip(g.gauge_meas(), o.gauge_meas(U)):
        assert abs(a - b) < 1e-13
    g.action(0, with_fermions=False)
    v = o.action(U, P, 5.7, None, None, with_fermions=False)
    assert abs(g.action_sum() - o.global_sum(v.copy())) < 1e-12 * np.abs(v).sum()
    g.close()
