"""The device kernels as the library launches them, checked on the CPU.

tests/emu_kernels/kernels_emu.cpp compiles the kernels' headers unchanged with g++
against the CPU stand-ins of tests/emu/hip/hip_runtime.h, under AddressSanitizer and
UBSan, and launches them with the library's grids, LDS sizes, argument set-up and
buffer sizes: the line, point and mixed stage kernels on the three rotating sets of
maxima (the member's first tile carries them on and clears the third) with the
compact and the full metric table, the viscous kernels, and a traced stage with its
reverse sweep.  What goes out of bounds, misses a barrier or reads what nothing
wrote ends the program or turns the results into NaN.

The results are held to the device tests' bars against the oracle; the line and
the point kernel, and the two metric tables, agree with each other bit for bit (the
norms, summed in another order, to 1e-12)."""
import hashlib
import os
import shutil
import subprocess

import numpy as np
import pytest

from oracle.oracle import Oracle
from tests.test_emu_stage import _case, _run
from tests.util import per_var_error

HERE = os.path.dirname(os.path.abspath(__file__))
REPO = os.path.dirname(HERE)
EMU = os.path.join(HERE, "emu_kernels")
CSRC = os.path.join(REPO, "sddc_amd", "csrc")
SOURCES = [os.path.join(EMU, "kernels_emu.cpp"), os.path.join(HERE, "emu", "hip", "hip_runtime.h"),
           os.path.join(REPO, "include", "sd2d.h")] + \
          [os.path.join(CSRC, f) for f in sorted(os.listdir(CSRC)) if f.endswith(".hpp")]
STEPS, RESID, TRACED, POINT, FULL = 0, 1, 2, 4, 8


@pytest.fixture(scope="module")
def emu():
    """{order: program}"""
    if shutil.which("g++") is None:
        pytest.skip("g++ is not installed")
    h = hashlib.sha256(b"".join(open(p, "rb").read() for p in SOURCES)).hexdigest()[:16]
    exes = {n: os.path.join(EMU, "_build", f"kernels_emu_N{n}_{h}") for n in (3, 4, 5)}
    os.makedirs(os.path.join(EMU, "_build"), exist_ok=True)
    cc = {n: subprocess.Popen(
        ["g++", "-std=c++20", "-O1", "-g", "-fno-omit-frame-pointer", "-fsanitize=address,undefined",
         "-fno-sanitize-recover=undefined", "-pthread", "-Wno-unknown-pragmas", f"-DEMU_N={n}",
         "-I", os.path.join(HERE, "emu"), "-I", CSRC, SOURCES[0], "-o", x + ".tmp"],
        stderr=subprocess.PIPE, text=True) for n, x in exes.items() if not os.path.exists(x)}
    for n, p in cc.items():
        err = p.communicate()[1]
        assert p.returncode == 0, err[-4000:]
        os.replace(exes[n] + ".tmp", exes[n])
    return exes


def _maxima(bits):
    """The running maxima of a set (none of the runs ends with a pair set apart)."""
    assert (bits[2:].view(np.uint64) == np.uint64(2**64 - 1)).all()
    return bits[:2]


def _steps(emu, tmp_path, case, Q0, job, **kw):
    out = _run(emu[case.N], tmp_path, case, Q0, job=STEPS | job, nsteps=3, **kw)
    n = Q0.size
    return (out[:n].reshape(Q0.shape, order="F"), _maxima(out[n:n + 4]),
            out[n + 4:n + 4 + 2 * case.ncell], out[n + 4 + 2 * case.ncell:])


STEP_CASES = [("channel5x4_N3", 3, 0), ("channel5x4_N3", 5, 2), ("ogrid4x8_N4", 5, 0),
              ("ogrid_curved4x8_N4", 3, 0), ("periodic31x2_N4", 3, 3), ("channel7x6_N5", 3, 2),
              ("ogrid2x23_N5", 5, 3)]


@pytest.mark.parametrize("name,k_stage,shape", STEP_CASES)
def test_stage_kernels(emu, tmp_path, name, k_stage, shape):
    case, Q0 = _case(name, k_stage=k_stage)
    o = Oracle(case)
    o.set_state(Q0, [0, 0, 0, 0])
    o.step(3, 2)                      # norms of the third step, the last
    Qo, mo = o.get_state()
    do = o.diag()
    o.close()
    nn = case.N ** 2 * case.ncell
    ref = _steps(emu, tmp_path, case, Q0, 0, tile_shape=shape)
    Q, mx, _, ns = ref
    assert per_var_error(Q - Q0, Qo - Q0)[0].max() <= 1e-11
    np.testing.assert_allclose(mx, np.asarray(mo)[2:4], rtol=1e-13, atol=0)
    np.testing.assert_allclose(np.sqrt(ns / [9 * nn, nn]), [do["resid_rms"], do["divb_rms"]],
                               rtol=1e-10)
    for job in (POINT, FULL):     # (curved cells have the full table either way)
        out = _steps(emu, tmp_path, case, Q0, job, tile_shape=shape)
        for a, b in zip(out[:3], ref[:3]):
            assert np.array_equal(a, b, equal_nan=True), job
        np.testing.assert_allclose(out[3], ns, rtol=1e-12)


@pytest.mark.parametrize("name", ["channel5x4_N3", "ogrid_curved4x8_N4", "channel7x6_N5"])
def test_mixed_kernel(emu, tmp_path, name):
    case, Q0 = _case(name)
    o = Oracle(case)
    o.set_state(Q0, [0, 0, 0, 0])
    o.step(3)
    Qo, _ = o.get_state()
    o.close()
    ref = _steps(emu, tmp_path, case, Q0, 0, precision=1)
    assert per_var_error(ref[0], Qo)[0].max() <= 1e-6
    for a, b in zip(_steps(emu, tmp_path, case, Q0, FULL, precision=1), ref):
        assert np.array_equal(a, b, equal_nan=True)


@pytest.mark.parametrize("name,shape", [("channel5x4_N3", 0), ("ogrid4x8_N4", 0),
                                        ("ogrid_curved4x8_N4", 2), ("channel7x6_N5", 2),
                                        ("ogrid2x23_N5", 3)])
def test_viscous_kernels(emu, tmp_path, name, shape):
    case, Q0 = _case(name, mu=0.02, eta0=0.03)
    n = Q0.size
    o = Oracle(case)
    o.set_state(Q0, [0, 0, 0, 0])
    ro, _ = o.compresid()
    o.set_state(Q0, [0, 0, 0, 0])
    o.step(3)
    Qo, mo = o.get_state()
    o.close()
    out = _run(emu[case.N], tmp_path, case, Q0, job=RESID, tile_shape=shape)
    assert per_var_error(out[:n].reshape(ro.shape, order="F"), ro)[0].max() <= 1e-12
    full = _run(emu[case.N], tmp_path, case, Q0, job=RESID | FULL, tile_shape=shape)
    assert np.array_equal(out, full, equal_nan=True)
    Q, mx, _, _ = _steps(emu, tmp_path, case, Q0, 0, tile_shape=shape)
    assert per_var_error(Q - Q0, Qo - Q0)[0].max() <= 1e-11
    np.testing.assert_allclose(mx, np.asarray(mo)[2:4], rtol=1e-13, atol=0)


@pytest.mark.parametrize("name,shape", [("channel5x4_N3", 2), ("ogrid4x8_N4", 0),
                                        ("ogrid_curved4x8_N4", 0), ("channel7x6_N5", 2),
                                        ("periodic31x2_N4", 3)])
def test_reverse_sweep(emu, tmp_path, name, shape):
    """Central differences of the emulated residual, as test_gpu_adjoint's bar."""
    case, Q0 = _case(name)
    n = Q0.size
    rng = np.random.default_rng(5)
    rbar = np.asfortranarray(rng.standard_normal(Q0.shape))
    V = rng.standard_normal(Q0.shape) * np.abs(Q0).max(axis=(1, 2, 3))[:, None, None, None]

    def run(Q, job=0):
        x = np.concatenate([Q, rbar], axis=3)
        return _run(emu[case.N], tmp_path, case, x, job=TRACED | job, tile_shape=shape)

    out = run(Q0)
    h = 1e-5
    rp, rm = ((run(Q0 + s * h * V)[:n] - (Q0 + s * h * V).ravel(order="F")) for s in (1, -1))
    fd = float(np.dot(rbar.ravel(order="F"), rp - rm)) / (2 * h)
    ad = float(np.dot(out[n:2 * n], V.ravel(order="F")))
    assert abs(ad - fd) <= 1e-6 * abs(fd), (ad, fd)
    assert np.isfinite(out).all()
    assert np.array_equal(run(Q0, FULL), out)
