"""What the steps compute does not depend on what the memory they run on held before, on
the GPU: handles made where arrays of NaNs were freed, on grids whose z-column tiles
have padding columns (which have no wavenumbers, and no part in f_int), give the rows
and the state that the oracle gives.

Tolerances: those of the short runs against the oracle (1e-13 for FP64, 2e-6 for
FP32: 30 times the largest differences measured over the parity shapes)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

TOL = {"fp64_reduced": 1e-13, "fp64_faithful": 1e-13, "fp32_mixed": 2e-6}


def _leave_nans():
    """NaNs in freed device memory, in a few large and many small blocks."""
    import torch
    t = [torch.full((1 << 24,), float("nan"), device="cuda") for _ in range(8)]
    t += [torch.full((1 << 14,), float("nan"), device="cuda") for _ in range(200)]
    torch.cuda.synchronize()
    del t
    torch.cuda.empty_cache()


@pytest.mark.parametrize("mode", ["fp32_mixed", "fp64_reduced", "fp64_faithful"])
@pytest.mark.parametrize("shape,var,dgb", [((16, 8, 8), 4, 0.4), ((8, 96, 12), 2, 0.0), ((24, 16, 48), 5, 0.4),
                                           ((12, 24, 64), 3, 0.4), ((96, 8, 16), 4, 0.0), ((8, 24, 160), 3, 0.4)])
def test_rows_and_state_on_memory_that_held_nans(pf, oracle, mode, shape, var, dgb):
    prm = dict(t_step=0.005, grad_coeff_phi=1.0, grad_coeff_c=0.8, D_gb=dgb)
    phi, con = pf.ic_voronoi(*shape, var, var + 3)
    _leave_nans()
    with pf.Simulation(pf.make_params(**prm), *shape, var, mode) as s:
        s.put_state(phi, con)
        first = s.diagnose()
        rows = s.step(4, diag_every=1)
        gphi, gcon = s.get_state()
    od = oracle.run(oracle.make_params(**prm), phi, con, 4)  # advances phi, con
    tol = TOL[mode]
    assert np.abs(gphi - phi).max() <= tol and np.abs(gcon - con).max() <= tol
    for d, o in zip([first] + rows, [od[0]] + list(od)):
        scale = abs(o["f_int"]) + abs(o["f_ch"]) + abs(o["f_eta"]) + 1.0
        for k in ("f_int", "f_ch", "f_eta", "e_tot"):
            assert abs(d[k] - o[k]) <= tol * scale, k
