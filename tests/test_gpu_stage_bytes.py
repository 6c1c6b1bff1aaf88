"""The bytes that pf_stage_bytes gives for a step's stages, on the GPU: over a step they
add up to the passes over the banks that the step's kernels make (a bank: one field's
half spectrum; a real field has the same bytes but for the Nyquist plane).  Whole
numbers: exact up to the rounding of the halves."""
import pytest

pytestmark = pytest.mark.gpu

#      mode, nx, var, D_gb, then banks a step: spectrum passes and real fields by stage
CASES = [
    # one-kernel x pass: C2R in, R2C of state and derivatives out, mob_c
    ("fp64_faithful", 32, 3, 0.4, dict(nonlinear=(12, 1), y_fwd=(16, 0), kspace_update=(18, 0), y_inv=(8, 0))),
    # three kernels: loops 5-10 on real fields, x forward of both, x inverse of the state
    ("fp64_faithful", 96, 3, 0.0, dict(nonlinear=(0, 9), x_r2c=(8, 8), y_fwd=(16, 0), kspace_update=(18, 0),
                                       y_inv=(8, 0), x_c2r=(4, 4))),
    # W in and out, then S with W; the chain's c is counted with its f^ and its field
    ("fp64_reduced", 32, 3, 0.0, dict(nonlinear=(0, 8), y_fwd=(8, 0), kspace_update=(16, 0), y_inv=(8, 0))),
    ("fp32_mixed", 32, 3, 0.4, dict(nonlinear=(0, 9), y_fwd=(8, 0), kspace_update=(21, 0), y_inv=(8, 0))),
]


@pytest.mark.parametrize("mode,nx,var,dgb,want", CASES)
def test_bytes_of_a_step(pf, mode, nx, var, dgb, want):
    ny, nz, es = 8, 12, 4 if mode == "fp32_mixed" else 8
    spec, real = 2 * (nx // 2 + 1) * ny * nz * es, nx * ny * nz * es
    phi, con = pf.ic_voronoi(nx, ny, nz, var, 5)
    with pf.Simulation(pf.make_params(t_step=0.005, D_gb=dgb), nx, ny, nz, var, mode) as s:
        s.put_state(phi, con)
        steps = 4
        s.set_timing(True)
        s.step(steps)
        got = s.stage_times()
    for stage, (nspec, nreal) in want.items():
        t = got[stage]
        n = 1 if stage == "x_c2r" and t["count"] == 1 else steps
        assert t["count"] * t["bytes"] == n * (nspec * spec + nreal * real), stage
