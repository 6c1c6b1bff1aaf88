"""CPU check of the x line's own transform plans (variants 4 and 5 of
csrc/pf_fft2.hpp) against a long-double DFT, with the emulation of
tests/cpu/fft2_emul.cpp, and that a line's threads are lanes of one wave."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"


@pytest.fixture(scope="module")
def plans(tmp_path_factory):
    if not os.path.exists(HIPCC):
        pytest.skip("hipcc not available")
    exe = str(tmp_path_factory.mktemp("xemul") / "xline_emul")
    subprocess.run([HIPCC, "-O1", "-std=c++17", "--offload-host-only", "--offload-arch=gfx950",
                    os.path.join(ROOT, "tests", "cpu", "xline_emul.cpp"), "-o", exe],
                   check=True, capture_output=True, timeout=600)
    out = subprocess.run([exe], check=True, capture_output=True, text=True, timeout=300).stdout
    return {(int(l.split()[0]), int(l.split()[1])): l.split() for l in out.strip().splitlines()}


@pytest.mark.parametrize("v", [4, 5])
@pytest.mark.parametrize("n", [16, 24, 32, 96])
def test_xline_plan_matches_dft(plans, n, v):
    _, _, npass, ef, ei, inplace, nthreads = plans[(n, v)]
    # double-precision butterflies: error grows ~ log n * eps * |x|_1
    assert int(npass) <= 3 and float(ef) < 1e-13 * n and float(ei) < 1e-13 * n
    # the transform is written back into its row without a barrier
    assert inplace == "1" and int(nthreads) <= 64
