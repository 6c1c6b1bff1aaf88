"""The step kernels where their choices by size change, on the GPU.

  * Fields beyond what one round of an x-line block's waves takes: the smallest
    such count and the largest accepted one, against the oracle.
  * Spectra below, within and above the sizes that stay in the last-level cache
    (over 24 and up to 256 MiB, counted without their Nyquist planes): one member and a
    batch of equal ones take different sides of that rule and agree bit for bit; every
    form on the cached side, with the mobility chain, against the oracle.

Tolerances: those of the short runs against the oracle (1e-13 for FP64, 2e-6 for
FP32: 30 times the largest differences measured over the parity shapes)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

PRM = dict(t_step=0.005, grad_coeff_phi=1.0, grad_coeff_c=0.8, D_gb=0.0)
TOL = {"fp64_reduced": 1e-13, "fp64_faithful": 1e-13, "fp32_mixed": 2e-6}


def _run(pf, oracle, shape, var, mode, steps, tuning=None, dgb=0.0):
    phi, con = pf.ic_voronoi(*shape, var, var + 3)
    prm = dict(PRM, D_gb=dgb)
    with pf.Simulation(pf.make_params(**prm), *shape, var, mode) as sim:
        if tuning:
            sim.set_tuning(**tuning)
        sim.put_state(phi, con)
        rows = sim.step(steps, diag_every=1)
        gphi, gcon = sim.get_state()
    od = oracle.run(oracle.make_params(**prm), phi, con, steps)  # advances phi, con
    tol = TOL[mode]
    err = max(np.abs(gphi - phi).max(), np.abs(gcon - con).max())
    print(f"{mode} {shape} x {var + 1}: {err:.2e}", flush=True)
    assert err <= tol
    for d, o in zip(rows, od):
        scale = abs(o["f_int"]) + abs(o["f_ch"]) + abs(o["f_eta"]) + 1.0
        for k in ("f_int", "f_ch", "f_eta", "e_tot"):
            assert abs(d[k] - o[k]) <= tol * scale, k


@pytest.mark.parametrize("mode,shape,var", [("fp64_reduced", (160, 8, 8), 48), ("fp64_reduced", (160, 8, 8), 50),
                                            ("fp64_reduced", (192, 8, 8), 40), ("fp64_reduced", (192, 8, 12), 63),
                                            ("fp64_reduced", (64, 8, 8), 128), ("fp64_reduced", (32, 8, 8), 256),
                                            ("fp32_mixed", (160, 8, 8), 96), ("fp32_mixed", (160, 8, 8), 101),
                                            ("fp32_mixed", (48, 8, 8), 256)])
def test_more_fields_than_one_round_of_a_block(pf, oracle, mode, shape, var):
    _run(pf, oracle, shape, var, mode, 3)


@pytest.mark.parametrize("lines", [1, 2])
def test_lines_per_block_beyond_its_threads(pf, oracle, lines):
    """25 FP64 fields of 160 points in 2-line blocks: 50 lines, two more than one
    round of a block's waves."""
    _run(pf, oracle, (160, 8, 8), 24, "fp64_reduced", 3, dict(xline_lines=lines))


@pytest.mark.parametrize("members", [2, 3, 14, 28, 29])
def test_batch_on_the_other_side_of_the_cache_rule(pf, members):
    """A member's spectrum is 9 MiB: alone and in a batch of 2 it is streamed, in one of
    3, 14 and 28 (27, 126 and 252 MiB; from 15 on not together with the carried
    spectrum's) it stays cached, in one of 29 (261 MiB) it does not fit."""
    n, var = 64, 8
    p = pf.make_params(**PRM)
    phi, con = pf.ic_voronoi(n, n, n, var, 12)
    with pf.Simulation(p, n, n, n, var, "fp32_mixed") as one:
        one.put_state(phi, con)
        one.step(4)
        want = one.get_state()
    sims = [pf.Simulation(p, n, n, n, var, "fp32_mixed") for _ in range(members)]
    try:
        for s in sims:
            s.put_state(phi, con)
        pf.ensemble_step(sims, 4)
        for s in (sims[0], sims[-1]):
            got = s.get_state()
            assert all(np.array_equal(a, b) for a, b in zip(got, want))
    finally:
        for s in sims:
            s.close()


# MiB, and what stays: the reduced forms' W (the carried spectrum S has as many), the
# faithful form's state and derivatives together, and each transform's own fields
@pytest.mark.parametrize("mode,shape,var,dgb", [
    ("fp64_reduced", (64, 64, 64), 11, 0.0),   # 24: streamed, the last that is
    ("fp64_reduced", (64, 64, 64), 12, 0.4),   # 26: W and S
    ("fp64_reduced", (64, 64, 64), 63, 0.0),   # 128: W and S, the last that are
    ("fp64_reduced", (64, 64, 64), 79, 0.4),   # 160: W
    ("fp32_mixed", (64, 64, 64), 24, 0.4),     # 25: W and S
    ("fp32_mixed", (96, 64, 64), 99, 0.0),     # 150: W
    ("fp64_faithful", (64, 64, 64), 5, 0.0),   # 24: streamed
    ("fp64_faithful", (64, 64, 64), 6, 0.4),   # 28: one-kernel x pass
    ("fp64_faithful", (128, 32, 64), 12, 0.4),  # 52: the same, longer lines
    ("fp64_faithful", (96, 64, 64), 5, 0.4),   # 36: three kernels
    ("fp64_faithful", (48, 64, 64), 18, 0.4),  # 57: three kernels
    ("fp64_reduced", (160, 128, 160), 3, 0.4),  # 100, and the chain's one field of 25
    ("fp64_faithful", (160, 128, 160), 3, 0.4)])  # 200, and the chain's one field of 25
def test_spectra_that_stay_cached(pf, oracle, mode, shape, var, dgb):
    _run(pf, oracle, shape, var, mode, 2 if shape[0] < 160 else 1, dgb=dgb)


# The faithful form's one-kernel x pass: every x length at its largest field count and
# either side of the counts and lengths where it takes over from the three kernels.
@pytest.mark.parametrize("shape,var", [((8, 8, 12), 1), ((12, 8, 8), 2), ((16, 8, 8), 16), ((24, 12, 8), 7),
                                       ((32, 8, 8), 16), ((48, 8, 8), 5), ((64, 8, 16), 16), ((96, 8, 8), 11),
                                       ((96, 8, 8), 12), ((128, 8, 8), 16), ((160, 8, 8), 12), ((192, 8, 8), 16),
                                       ((256, 8, 8), 16), ((512, 8, 8), 16), ((64, 8, 8), 17)])
def test_faithful_x_pass(pf, oracle, shape, var):
    _run(pf, oracle, shape, var, "fp64_faithful", 4, dgb=0.4)


# every x length of the one-kernel x pass, one of the three kernels, and short lines of
# more than 2 MiB, whose inverse goes through LDS
@pytest.mark.parametrize("shape,var", [((8, 8, 12), 3), ((12, 8, 8), 5), ((16, 8, 8), 4), ((24, 8, 8), 4),
                                       ((32, 8, 8), 6), ((48, 8, 8), 5), ((64, 8, 8), 4), ((64, 8, 8), 16),
                                       ((96, 8, 8), 12), ((128, 8, 8), 12), ((160, 8, 8), 13), ((192, 8, 8), 12),
                                       ((256, 8, 8), 13), ((512, 8, 8), 12), ((96, 8, 8), 4),
                                       ((24, 64, 48), 4), ((16, 64, 64), 4)])
def test_faithful_calls_of_any_length_agree(pf, shape, var):
    """Steps in calls of 1, 2 and 5, in one call by replayed graphs, and with a restart
    in a new handle from the state of the first four, bit for bit: a call starts from
    the real state and its later steps from x-half lines."""
    phi, con = pf.ic_voronoi(*shape, var, var + 3)
    p = pf.make_params(**dict(PRM, D_gb=0.4))
    got = []
    for runs, graphs in (([[8]], True), ([[8]], False), ([[1] * 8], True), ([[2, 5, 1]], True), ([[4], [4]], True)):
        state = phi, con
        for calls in runs:
            with pf.Simulation(p, *shape, var, "fp64_faithful") as s:
                s.set_graphs(graphs)
                s.put_state(*state)
                for n in calls:
                    s.step(n, diag_every=2)
                state = s.get_state()
        got.append(state)
    for g in got[1:]:
        assert all(np.array_equal(a, b) for a, b in zip(g, got[0]))


# the x lengths of the one-kernel x pass, then every z length with the three kernels
# (more order parameters than the one kernel takes)
@pytest.mark.parametrize("shape,var", [((8, 8, 12), 3), ((12, 8, 8), 5), ((16, 8, 8), 4), ((24, 8, 8), 4),
                                       ((32, 8, 8), 6), ((48, 8, 8), 5), ((64, 8, 8), 4), ((96, 8, 8), 12),
                                       ((128, 8, 8), 12), ((160, 8, 8), 13), ((192, 8, 8), 12), ((256, 8, 8), 13),
                                       ((512, 8, 8), 12)] +
                         [((24, 8, nz), 17) for nz in (8, 12, 16, 24, 32, 48, 64, 96, 128, 160, 192, 256, 512)])
def test_faithful_state_does_not_depend_on_the_rows(pf, shape, var):
    """Steps with no summary row, a row every second step and one every step end in the
    same bits, and so does a restart after an odd number of steps, whose rows fall on
    the other steps."""
    phi, con = pf.ic_voronoi(*shape, var, var + 3)
    p = pf.make_params(**dict(PRM, D_gb=0.4))
    got = []
    for runs, every in (([8], 0), ([8], 1), ([8], 2), ([3, 5], 2)):
        state = phi, con
        for n in runs:
            with pf.Simulation(p, *shape, var, "fp64_faithful") as s:
                s.put_state(*state)
                s.step(n, diag_every=every)
                state = s.get_state()
        got.append(state)
    for g in got[1:]:
        assert all(np.array_equal(a, b) for a, b in zip(g, got[0]))


@pytest.mark.parametrize("mode", ["fp64_faithful", "fp32_mixed"])
@pytest.mark.parametrize("shape,var", [((12, 12, 12), 1), ((8, 8, 12), 15), ((12, 12, 12), 16), ((8, 12, 12), 17),
                                       ((12, 12, 12), 33)])
def test_state_comes_back_point_by_point(pf, mode, shape, var):
    """put_state then get_state, point counts and field counts around the tiles of 128
    points by 16 fields: the faithful form's state as it was, FP32 rounded once more by
    its transforms."""
    rng = np.random.default_rng(var)
    n = shape[2], shape[1], shape[0]
    phi, con = rng.random(n + (var,)), rng.random(n)
    with pf.Simulation(pf.make_params(**PRM), *shape, var, mode) as s:
        ref_phi, ref_con = pf.ic_voronoi(*shape, var, var + 3)
        phi, con = phi.reshape(ref_phi.shape), con.reshape(ref_con.shape)
        s.put_state(phi, con)
        gphi, gcon = s.get_state()
    if mode == "fp64_faithful":
        assert np.array_equal(gphi, phi) and np.array_equal(gcon, con)
    else:
        assert np.abs(gphi - phi).max() <= 2e-6 and np.abs(gcon - con).max() <= 2e-6
