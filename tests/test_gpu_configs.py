"""The five benchmark configurations on the GPU, each at its own workload or at
the largest slice of it the CPU oracle can follow, plus size-independent
properties where the oracle cannot:

  C1  64^3, c + 4 eta, small-noise start (c = 0.5 +- 0.01, |eta| <= 1e-3), dt = 0.01,
      kappa = 0.5: the FP64 forms against the oracle step by step until the state
      goes non-finite, then PF_ENONFINITE at the same step;
  C2  256^3, c + 16 eta, FP64 drop-in (fp64_faithful): 256-point lines on every
      axis against the oracle, and the full-size run's mass and energy;
  C3  FP32-mixed against the FP64 drop-in over 1000 steps at 256^3 x 17, per-field
      max and RMS differences every 100 steps, bound 1e-5;
  C4  a parameter-sweep ensemble over 64/96/128/160/192^3 with c + 8 eta: the 64^3
      member against the oracle, the others conserve mass and lower the energy;
  C5  512^3, c + 36 eta, FP32-mixed: 512-point y and z lines against the oracle,
      and the full size built on the device (pf_put_voronoi) over a few steps.

Tolerances are written per test; each print line records what was measured.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

VOR = dict(t_step=0.005, grad_coeff_phi=1.0, grad_coeff_c=1.0)


def _rel(a, b):
    return np.abs(a - b).max() / max(np.abs(b).max(), 1e-300)


def _escale(o, k):
    """The magnitude a summary energy's error is relative to (its own; for e_tot
    the sum of the three terms' magnitudes, which can nearly cancel)."""
    if k == "e_tot":
        return max(abs(o["f_int"]) + abs(o["f_ch"]) + abs(o["f_eta"]), 1.0)
    return max(abs(o[k]), 1.0)


# ---------------------------------------------------------------------------
# device-built initial condition
# ---------------------------------------------------------------------------
@pytest.mark.parametrize("mode", ["fp64_faithful", "fp64_reduced", "fp32_mixed"])
def test_put_voronoi_equals_host_ic_and_put_state(pf, mode):
    nx, ny, nz, var, seeds, iseed = 24, 16, 32, 5, 7, -3
    phi, con = pf.ic_voronoi(nx, ny, nz, var, seeds, iseed, 0.41, 0.03)
    prm = pf.make_params(**dict(VOR, D_gb=0.2))
    out = []
    for dev in (False, True):
        with pf.Simulation(prm, nx, ny, nz, var, mode) as sim:
            if dev:
                sim.put_voronoi(seeds, iseed, 0.41, 0.03)
            else:
                sim.put_state(phi, con)
            s0 = sim.get_state()
            d = sim.step(4, diag_every=2)
            out.append((s0, sim.get_state(), d))
    (a0, a1, da), (b0, b1, db) = out
    for x, y in zip(a0 + a1, b0 + b1):
        assert np.array_equal(x, y)
    assert da == db


# ---------------------------------------------------------------------------
# C1: small-noise start, dt = 0.01, kappa = 0.5 (diverges in FP64)
# ---------------------------------------------------------------------------
C1 = dict(t_step=0.01, grad_coeff_phi=0.5, grad_coeff_c=0.5)


@pytest.mark.parametrize("dgb", [0.0, 1.0])
def test_c1_faithful_per_step_vs_oracle_until_nonfinite(pf, oracle, dgb):
    """The h-derivative terms of loops 7-9 scale like 1/eta (src/var_diff.f90:
    829-835, no guard on D4 at :743), so this start blows up within a few steps
    in exact FP64 as well (max|phi| 2.6e2, 4.6e5, 4.3e15, 4.4e45, then NaN).  Near
    the blow-up the step amplifies rounding: a 1-ulp perturbation of the start
    moves the oracle's own c by 1e-11 at step 3 and 4e-6 at step 4 (D_gb = 0).
    So each step's bound is the oracle's own sensitivity, measured alongside
    (the oracle from a start perturbed by 1 ulp), times 30, and never tighter
    than 1e-13 for the state (1e-12 for the summed energies).  Once the oracle's state is
    non-finite, the drop-in must report that step as PF_ENONFINITE."""
    n, var = 64, 4
    phi, con = pf.ic_random(n, n, n, var)
    prm = dict(C1, D_gb=dgb)
    op = oracle.make_params(**prm)
    rng = np.random.default_rng(1)
    a_phi, a_con = phi.copy(), con.copy()
    b_phi = phi * (1 + 2.0 ** -52 * rng.choice([-1.0, 1.0], phi.shape))
    b_con = con * (1 + 2.0 ** -52 * rng.choice([-1.0, 1.0], con.shape))
    fin = lambda x, y: np.isfinite(x).all() and np.isfinite(y).all()
    with pf.Simulation(pf.make_params(**prm), n, n, n, var, "fp64_faithful") as sim:
        sim.put_state(phi, con)
        step = 0
        while True:
            step += 1
            print(f"C1 dgb={dgb} step {step}", flush=True)
            if not fin(a_phi, a_con):
                with pytest.raises(pf.PfError) as e:
                    sim.step(1, diag_every=1)
                assert e.value.code == pf.PF_ENONFINITE
                break
            ra = oracle.run(op, a_phi, a_con, 1)[0]
            rb = oracle.run(op, b_phi, b_con, 1)[0]
            gd = sim.step(1, diag_every=1)[0]
            # the energies are sums over all points; the oracle adds them serially
            # and uncompensated (as the reference), the library in a compensated
            # tree, so they differ by the oracle's own summation rounding as well
            # (measured 4.6e-13 in f_eta at step 3, terms up to 1e22): 1e-12 floor
            for k in ("f_int", "f_ch", "f_eta", "e_tot"):
                tol = max(1e-12, 30 * abs(ra[k] - rb[k]) / abs(ra[k]))
                assert abs(gd[k] - ra[k]) <= tol * abs(ra[k]), (step, k, gd[k], ra[k], tol)
            if fin(a_phi, a_con):
                gphi, gcon = sim.get_state()
                ep, ec = _rel(gphi, a_phi), _rel(gcon, a_con)
                sp, sc = _rel(b_phi, a_phi), _rel(b_con, a_con)
                print(f"  rel diff phi {ep:.2e} c {ec:.2e} (oracle's 1-ulp sensitivity {sp:.2e} {sc:.2e}), "
                      f"max|phi| {np.abs(a_phi).max():.2e}")
                assert ep <= max(1e-13, 30 * sp) and ec <= max(1e-13, 30 * sc)
            assert step < 20
    assert step >= 4  # the run did follow the oracle for several steps


@pytest.mark.parametrize("mode", ["fp64_reduced", "fp32_mixed"])
def test_c1_reduced_forms_report_nonfinite(pf, mode):
    """The reduced forms blow up on the same start (FP32 overflows first) and
    report it as PF_ENONFINITE instead of returning garbage rows."""
    n, var = 64, 4
    phi, con = pf.ic_random(n, n, n, var)
    with pf.Simulation(pf.make_params(**C1), n, n, n, var, mode) as sim:
        sim.put_state(phi, con)
        for step in range(1, 8):
            try:
                sim.step(1, diag_every=1)
            except pf.PfError as e:
                assert e.code == pf.PF_ENONFINITE
                print(f"C1 {mode}: PF_ENONFINITE at step {step}")
                break
        else:
            pytest.fail("no PF_ENONFINITE within 7 steps")


# ---------------------------------------------------------------------------
# C2: the FP64 drop-in with 256-point transforms
# ---------------------------------------------------------------------------
@pytest.mark.parametrize("shape", [(256, 8, 8), (8, 256, 8), (8, 8, 256)], ids=lambda s: "x".join(map(str, s)))
def test_c2_faithful_256_point_lines_vs_oracle(pf, oracle, shape):
    """The faithful form's 256-point kernels (k_xline's FAITH form, k_ypass and
    k_zfaithful at 256) with 17 fields, D_gb != 0, against the oracle."""
    nx, ny, nz = shape
    var = 16
    prm = dict(VOR, D_gb=0.3)
    phi, con = pf.ic_voronoi(nx, ny, nz, var, 12)
    with pf.Simulation(pf.make_params(**prm), nx, ny, nz, var, "fp64_faithful") as sim:
        sim.put_state(phi, con)
        dg = sim.step(6, diag_every=2)
        gphi, gcon = sim.get_state()
    ophi, ocon = phi.copy(), con.copy()
    od = oracle.run(oracle.make_params(**prm), ophi, ocon, 6)
    ep, ec = _rel(gphi, ophi), _rel(gcon, ocon)
    worst = max(abs(d[k] - od[d["step"] - 1][k]) / _escale(od[d["step"] - 1], k)
                for d in dg for k in ("f_int", "f_ch", "f_eta", "e_tot"))
    print(f"C2 faithful {shape}: state {ep:.2e} {ec:.2e}, energies {worst:.2e}")
    assert ep < 1e-13 and ec < 1e-13 and worst < 1e-13
    for d in dg:
        o = od[d["step"] - 1]
        for k in ("c_max", "c_min", "phi_min", "phi_3_max"):
            assert abs(d[k] - o[k]) <= 1e-13, (k, d[k], o[k])


# ---------------------------------------------------------------------------
# C2 / C3 at full size: 256^3, c + 16 eta
# ---------------------------------------------------------------------------
def test_full_size_three_forms_agree(pf):
    """40 steps of the benchmark workload in all three forms from one
    device-built start: the FP64 forms conserve the mean of c to 1e-12 and agree
    with each other to 1e-11 per field; FP32-mixed agrees with FP64 to 2e-6 per
    field and 1e-6 in e_tot; every form lowers e_tot at every reported step."""
    n, var = 256, 16
    res = {}
    for mode in ("fp64_faithful", "fp64_reduced", "fp32_mixed"):
        print("full size", mode, flush=True)
        with pf.Simulation(pf.make_params(**VOR), n, n, n, var, mode) as sim:
            sim.put_voronoi(64)
            rows = sim.step(40, diag_every=2)
            res[mode] = (rows, sim.get_state())
    m0 = res["fp64_faithful"][0][0]["c_mean"]
    for mode, (rows, (phi, con)) in res.items():
        assert np.isfinite(phi).all() and np.isfinite(con).all()
        assert len(rows) == 20
        e = [r["e_tot"] for r in rows]
        assert all(b < a for a, b in zip(e, e[1:])), (mode, e)
        if mode != "fp32_mixed":
            assert abs(float(con.mean()) - m0) <= 1e-12 * m0, mode
            for r in rows:
                assert abs(r["c_mean"] - m0) <= 1e-12 * m0, (mode, r["step"])
    (pf_, cf), (pr, cr), (p3, c3) = (res[m][1] for m in ("fp64_faithful", "fp64_reduced", "fp32_mixed"))
    d64 = max(np.abs(cf - cr).max(), max(np.abs(pf_[..., i] - pr[..., i]).max() for i in range(var)))
    d32 = max(np.abs(c3 - cf).max(), max(np.abs(p3[..., i] - pf_[..., i]).max() for i in range(var)))
    e32 = max(abs(a["e_tot"] - b["e_tot"]) / abs(b["e_tot"])
              for a, b in zip(res["fp32_mixed"][0], res["fp64_faithful"][0]))
    print(f"256^3 x 17, 40 steps: |reduced - faithful| {d64:.2e}, |fp32 - faithful| {d32:.2e}, "
          f"e_tot rel {e32:.2e}")
    assert d64 < 1e-11
    assert d32 < 2e-6 and e32 < 1e-6


def test_c3_fp32_error_after_1000_steps_256(pf):
    """The accuracy target of the FP32-mixed form on its own workload: per-field
    max |fp32 - fp64| <= 1e-5 at every 100-step checkpoint up to step 1000,
    against the FP64 drop-in (which follows the oracle to 1e-12 over 500 steps)."""
    n, var = 256, 16
    prm = pf.make_params(**VOR)
    worst = 0.0
    with pf.Simulation(prm, n, n, n, var, "fp32_mixed") as a, \
            pf.Simulation(prm, n, n, n, var, "fp64_faithful") as b:
        a.put_voronoi(64)
        b.put_voronoi(64)
        for ck in range(1, 11):
            a.step(100)
            b.step(100)
            pa, ca = a.get_state()
            pb, cb = b.get_state()
            dmax = [float(np.abs(ca - cb).max())] + [float(np.abs(pa[..., i] - pb[..., i]).max())
                                                     for i in range(var)]
            drms = [float(np.sqrt(np.mean((ca - cb) ** 2)))] + \
                   [float(np.sqrt(np.mean((pa[..., i] - pb[..., i]) ** 2))) for i in range(var)]
            print(f"C3 step {ck * 100}: max c {dmax[0]:.2e} eta {max(dmax[1:]):.2e}; "
                  f"rms c {drms[0]:.2e} eta {max(drms[1:]):.2e}", flush=True)
            worst = max(worst, max(dmax))
            assert max(dmax) <= 1e-5, (ck * 100, dmax)
    assert worst > 0


# ---------------------------------------------------------------------------
# C4: parameter-sweep ensemble, c + 8 eta, one member per grid size
# ---------------------------------------------------------------------------
def test_c4_ensemble_members(pf, oracle):
    import pf_amd.runconfig as rc

    members = rc.ensemble_members(pf, n=5, var=8)
    assert [m["grid"] for m in members] == [64, 96, 128, 160, 192]
    sims = []
    try:
        for m in members:
            g = m["grid"]
            s = pf.Simulation(m["params"], g, g, g, m["var"], "fp32_mixed")
            s.put_voronoi(16, -(m["member"] + 1))
            sims.append(s)
        d0 = [s.diagnose() for s in sims]
        pf.ensemble_step(sims, 6)
        d1 = [s.diagnose() for s in sims]
        pf.ensemble_step(sims, 14)
        d2 = [s.diagnose() for s in sims]
        # the 64^3 member against the oracle after 6 steps
        m = members[0]
        phi, con = pf.ic_voronoi(64, 64, 64, 8, 16, -1, 0.4, 0.02)
        p = m["params"]
        op = oracle.make_params(**{k: getattr(p, k) for k in pf.PARAM_NAMES})
        oracle.run(op, phi, con, 6)
        s64 = pf.Simulation(m["params"], 64, 64, 64, 8, "fp32_mixed")
        try:
            s64.put_voronoi(16, -1)
            s64.step(6)
            gphi, gcon = s64.get_state()
        finally:
            s64.close()
        err = max(np.abs(gphi - phi).max(), np.abs(gcon - con).max())
        print(f"C4 64^3 member (kappa {m['kappa']:.3f}, M {m['M']:.3f}, L {m['L']:.3f}): "
              f"|fp32 - oracle| {err:.2e} after 6 steps")
        assert err < 2e-6
        for mm, a, b, c in zip(members, d0, d1, d2):
            print(f"C4 member {mm['grid']}^3: e_tot {a['e_tot']:.6e} -> {b['e_tot']:.6e} -> {c['e_tot']:.6e}")
            assert abs(c["c_mean"] - a["c_mean"]) <= 1e-12 * abs(a["c_mean"])
            assert c["e_tot"] < b["e_tot"] < a["e_tot"]
    finally:
        for s in sims:
            s.close()


# ---------------------------------------------------------------------------
# C5: 512-point transforms with 37 fields (FP32-mixed)
# ---------------------------------------------------------------------------
@pytest.mark.parametrize("shape", [(8, 512, 8), (8, 8, 512)], ids=lambda s: "x".join(map(str, s)))
def test_c5_512_point_lines_vs_oracle(pf, oracle, shape):
    """k_ypass<float, 512> and k_zline<float, 512> (1024-thread blocks) with 37
    fields against the oracle."""
    nx, ny, nz = shape
    var = 36
    prm = dict(VOR, D_gb=0.0)
    phi, con = pf.ic_voronoi(nx, ny, nz, var, 40)
    with pf.Simulation(pf.make_params(**prm), nx, ny, nz, var, "fp32_mixed") as sim:
        sim.put_state(phi, con)
        dg = sim.step(6, diag_every=2)
        gphi, gcon = sim.get_state()
    ophi, ocon = phi.copy(), con.copy()
    od = oracle.run(oracle.make_params(**prm), ophi, ocon, 6)
    err = max(np.abs(gphi - ophi).max(), np.abs(gcon - ocon).max())
    worst = max(abs(d[k] - od[d["step"] - 1][k]) / _escale(od[d["step"] - 1], k)
                for d in dg for k in ("f_int", "f_ch", "f_eta", "e_tot"))
    print(f"C5 {shape} x 37 fp32: state {err:.2e}, energies {worst:.2e}")
    assert err < 2e-6 and worst < 2e-6


def test_c5_full_size_512(pf):
    """512^3 with c + 36 eta (the C5 workload, ~100 GB on the device) from the
    device-built 512-seed polycrystal: 6 steps, rows every 2 steps from the
    library's own reductions (no 40 GB state download): finite, the FP64 mean of
    c kept, e_tot falling, extrema in range."""
    n, var = 512, 36
    with pf.Simulation(pf.make_params(**VOR), n, n, n, var, "fp32_mixed") as sim:
        print("C5 512^3 x 37: building the start on the device", flush=True)
        sim.put_voronoi(512)
        d0 = sim.diagnose()
        print("C5 512^3 x 37: stepping", flush=True)
        rows = sim.step(6, diag_every=2)
    # rows of steps 1 (pf_diagnose before stepping), 2, 4, 6
    assert [r["step"] for r in rows] == [2, 4, 6] and d0["step"] == 1
    e = [d0["e_tot"]] + [r["e_tot"] for r in rows]
    print("C5 512^3 x 37 e_tot:", ["%.6e" % x for x in e], "c_mean", d0["c_mean"],
          "extrema of the last row", [rows[-1][k] for k in ("c_max", "c_min", "phi_min", "phi_3_max")])
    assert all(np.isfinite(x) for x in e)
    assert all(b < a for a, b in zip(e, e[1:])), e
    # the sharp precipitate boundaries of the Voronoi start drive c quickly
    # (mu_c jumps by ~6 across them), with the overshoot of Cahn-Hilliard at
    # sharp fronts: measured c in [-0.05, 0.75] after 5 steps
    for r in rows:
        assert r["c_mean"] == d0["c_mean"]
        assert -0.5 < r["c_min"] < 0.4 < r["c_max"] < 1.5
        assert 0.0 < r["phi_min"] <= 1.0 and 0.9 <= r["phi_3_max"] <= 1.1
