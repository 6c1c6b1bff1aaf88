"""The combined passes at their edges, on the GPU.

  * The faithful form's fused kernels at every z length against the oracle; the x
    lengths give main-block rows shorter than a y tile, and no multiple of one.
  * The point loops of the three-kernel faithful step (few fields on lines over 64
    points, or more than 16 order parameters) take four rows at a time: every
    remainder of var - 1, on either side of it.
  * A device transform from and to real arrays that are aligned for their reals
    only (no complex access is possible there) equals the aligned one bit for bit.

Tolerances: those of the short runs against the oracle (1e-13 for FP64: 30 times
the largest difference measured over the parity shapes)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# (nx, ny, nz, var): every nz; nx / 2 = 4 .. 80 columns a row; var mod 4 = 0 .. 3
SHAPES = [(8, 12, 8, 1), (12, 8, 12, 2), (16, 16, 16, 3), (24, 12, 24, 4), (48, 8, 32, 5), (16, 24, 48, 6),
          (96, 8, 64, 7), (8, 16, 96, 4), (32, 8, 128, 2), (12, 8, 160, 3), (24, 8, 192, 5), (160, 8, 8, 3),
          (8, 8, 256, 3), (8, 8, 512, 2)]


# the three-kernel step: var - 1 = 3 .. 8 and 16 .. 20 rows
POINTS = [(96, 8, 8, 4), (96, 8, 12, 5), (128, 8, 8, 6), (96, 12, 8, 8), (160, 8, 8, 9), (24, 8, 8, 17),
          (16, 8, 12, 18), (64, 8, 8, 19), (32, 8, 8, 20), (8, 8, 8, 21)]


@pytest.mark.parametrize("nx,ny,nz,var", SHAPES + POINTS)
def test_faithful_step_at_every_z_length(pf, oracle, nx, ny, nz, var):
    prm = dict(t_step=0.005, grad_coeff_phi=1.0, grad_coeff_c=0.8, D_gb=0.4)
    phi, con = pf.ic_voronoi(nx, ny, nz, var, 2 * var + 1, iseed=-(nx + nz))
    with pf.Simulation(pf.make_params(**prm), nx, ny, nz, var, "fp64_faithful") as sim:
        sim.put_state(phi, con)
        first = sim.diagnose()
        rows = sim.step(4, diag_every=1)
        gphi, gcon = sim.get_state()
    od = oracle.run(oracle.make_params(**prm), phi, con, 4)  # advances phi, con
    assert np.abs(gphi - phi).max() <= 1e-13 * np.abs(phi).max()
    assert np.abs(gcon - con).max() <= 1e-13 * np.abs(con).max()
    assert len(rows) == 4
    for d, o in zip([first] + rows, [od[0]] + list(od)):
        scale = abs(o["f_int"]) + abs(o["f_ch"]) + abs(o["f_eta"]) + 1.0
        for k in ("f_int", "f_ch", "f_eta", "e_tot"):
            assert abs(d[k] - o[k]) <= 1e-13 * scale, k
        for k in ("c_max", "c_min", "phi_min", "phi_3_max"):
            assert abs(d[k] - o[k]) <= 1e-13, k


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
@pytest.mark.parametrize("layout", [0, 1])
def test_real_arrays_aligned_for_reals_only(pf, prec, layout):
    import torch
    nx, ny, nz, b = 24, 12, 16, 3
    dt, p = (torch.float64, pf.PREC_FP64) if prec == "fp64" else (torch.float32, pf.PREC_FP32)
    n, half = b * nx * ny * nz, b * (nx // 2 + 1) * ny * nz
    g = torch.Generator().manual_seed(5)
    x = torch.randn(n, generator=g, dtype=torch.float64).to(dt).cuda()
    off = torch.zeros(n + 1, dtype=dt, device="cuda")[1:]
    off.copy_(x)
    spec = [torch.zeros(2 * half, dtype=dt, device="cuda") for _ in range(2)]
    back = [torch.zeros(n, dtype=dt, device="cuda"), torch.zeros(n + 1, dtype=dt, device="cuda")[1:]]
    torch.cuda.synchronize()
    for src, sp, dst in zip((x, off), spec, back):
        pf.fft_r2c_device(nx, ny, nz, b, p, src.data_ptr(), sp.data_ptr(), layout, 0.5)
        pf.fft_c2r_device(nx, ny, nz, b, p, sp.data_ptr(), dst.data_ptr(), layout)
    torch.cuda.synchronize()
    assert off.data_ptr() % (2 * x.element_size()) != 0
    assert torch.equal(spec[0], spec[1]) and torch.equal(back[0], back[1])
    assert torch.equal(off, x)  # the source is left alone


# The inverse x pass takes lines of up to 32 complex points (nx <= 64), 64 or 32 of them a
# block, from 2 MiB on through LDS: 1 field of 96 lines, 7 of 96, and enough for 2.2 MiB
# end in a part of a block.
@pytest.mark.parametrize("prec", ["fp64", "fp32"])
@pytest.mark.parametrize("nx", [8, 12, 16, 24, 32, 48, 64, 96])
@pytest.mark.parametrize("batch", [1, 7, 0])
def test_inverse_of_short_lines(pf, prec, nx, batch):
    """Against numpy, with the tolerances of the device transforms' tests; nothing is
    written past the last line."""
    import torch
    ny, nz = 12, 8
    dt, ct, p, tol = ((torch.float64, torch.complex128, pf.PREC_FP64, 1e-13) if prec == "fp64"
                      else (torch.float32, torch.complex64, pf.PREC_FP32, 5e-6))
    batch = batch or int(2.2 * 2 ** 20 / (96 * nx * torch.tensor([], dtype=dt).element_size())) | 1
    rng = np.random.default_rng(nx + batch)
    x = rng.standard_normal((batch, nz, ny, nx))
    spec = torch.tensor(np.fft.rfftn(x, axes=(1, 2, 3)) / (nx * ny * nz)).to(ct).cuda()
    back = torch.full((x.size + 64,), 7.0, dtype=dt, device="cuda")
    torch.cuda.synchronize()
    pf.fft_c2r_device(nx, ny, nz, batch, p, spec.data_ptr(), back.data_ptr(), pf.LAYOUT_XFAST)
    torch.cuda.synchronize()
    back = back.cpu().double().numpy()
    assert np.abs(back[:x.size].reshape(x.shape) - x).max() < tol * np.abs(x).max()
    assert (back[x.size:] == 7.0).all()


# The y pass exchanges the Nyquist planes' lines in rows of their own at three-pass
# lengths (96, 160, 192, 512) and FP32's 256, else (128) in the tile's column order;
# 40 lines end in a part of a tile, and 30 MiB take the accesses of a cached bank.
@pytest.mark.parametrize("prec", ["fp64", "fp32"])
@pytest.mark.parametrize("ny", [96, 128, 160, 192, 256, 512])
@pytest.mark.parametrize("mib", [0, 30])
def test_y_pass_over_the_nyquist_planes(pf, prec, ny, mib):
    """Transform and inverse against numpy, the Nyquist plane on its own scale."""
    import torch
    nx, nz = 12, 8
    dt, ct, p, tol = ((torch.float64, torch.complex128, pf.PREC_FP64, 1e-13) if prec == "fp64"
                      else (torch.float32, torch.complex64, pf.PREC_FP32, 5e-6))
    batch = max(5, (mib << 20) // (nx * ny * nz * torch.tensor([], dtype=dt).element_size()))
    x = np.random.default_rng(ny).standard_normal((batch, nz, ny, nx))
    ref = np.fft.rfftn(x, axes=(1, 2, 3)) / (nx * ny * nz)
    dx = torch.tensor(x, dtype=dt).cuda()
    spec = torch.empty(ref.shape, dtype=ct, device="cuda")
    torch.cuda.synchronize()
    pf.fft_r2c_device(nx, ny, nz, batch, p, dx.data_ptr(), spec.data_ptr(), pf.LAYOUT_XFAST, 1.0 / (nx * ny * nz))
    torch.cuda.synchronize()
    err = np.abs(spec.cpu().numpy() - ref)
    assert err.max() < tol * np.abs(ref).max() and err[..., -1].max() < tol * np.abs(ref[..., -1]).max()
    dx.zero_()
    torch.cuda.synchronize()
    pf.fft_c2r_device(nx, ny, nz, batch, p, spec.data_ptr(), dx.data_ptr(), pf.LAYOUT_XFAST)
    torch.cuda.synchronize()
    assert np.abs(dx.cpu().double().numpy() - x).max() < tol * np.abs(x).max()
