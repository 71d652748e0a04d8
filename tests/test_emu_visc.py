"""The accuracy of the viscous flux's quotients, on the CPU: every component of
vflux_n and the internal energy (sd2d_visc.hpp, compiled unchanged with g++) is as
close to 113-bit arithmetic as the same formulas with IEEE divisions, in the rms
over random states, with and without fused multiply-adds."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "sddc_amd", "csrc")


@pytest.mark.parametrize("contract", ["off", "fast"])
def test_viscous_flux_accuracy(tmp_path, contract):
    if shutil.which("g++") is None:
        pytest.skip("g++ is not installed")
    exe = tmp_path / "visc_accuracy"
    r = subprocess.run(["g++", "-std=gnu++20", "-O2", "-mfma", f"-ffp-contract={contract}",
                        "-Wno-unknown-pragmas", "-I", os.path.join(HERE, "emu"), "-I", CSRC,
                        os.path.join(HERE, "emu_visc", "visc_accuracy.cpp"), "-o", str(exe),
                        "-lquadmath"], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-4000:]
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stderr
    rows = [ln.split() for ln in r.stdout.splitlines()]
    assert len(rows) == 8
    for k, a, b in rows:      # 1 %: the order of the sums and of the fusions
        assert float(a) <= 1.01 * float(b), (k, a, b)
