"""The pinned ring of the state-sized copies (sd2d_xfer.hpp), on the CPU.

tests/emu_xfer/xfer_emu.cpp compiles the header unchanged against stand-ins of
the HIP calls it makes (a stream is a host thread that runs its operations in
order) under ThreadSanitizer: whole copies at the sizes where the path changes,
contexts that come and go while another thread's copy is under way, pinned arrays
of the caller's, and copies too small for the ring."""
import hashlib
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
EMU = os.path.join(HERE, "emu_xfer")
CSRC = os.path.join(os.path.dirname(HERE), "sddc_amd", "csrc")
SOURCES = [os.path.join(EMU, "xfer_emu.cpp"), os.path.join(EMU, "hip", "hip_runtime.h"),
           os.path.join(CSRC, "sd2d_xfer.hpp")]


@pytest.fixture(scope="module")
def xfer_exe():
    if shutil.which("g++") is None:
        pytest.skip("g++ is not installed")
    h = hashlib.sha256(b"".join(open(p, "rb").read() for p in SOURCES)).hexdigest()[:16]
    exe = os.path.join(EMU, "_build", f"xfer_emu_{h}")
    if not os.path.exists(exe):
        os.makedirs(os.path.dirname(exe), exist_ok=True)
        r = subprocess.run(["g++", "-std=c++17", "-O1", "-g", "-fsanitize=thread", "-pthread",
                            "-I", EMU, "-I", CSRC, SOURCES[0], "-o", exe + ".tmp"],
                           capture_output=True, text=True)
        assert r.returncode == 0, r.stderr[-4000:]
        os.replace(exe + ".tmp", exe)
    return exe


@pytest.mark.parametrize("job", ["data", "contexts", "pinned", "small"])
def test_ring(xfer_exe, job):
    r = subprocess.run([xfer_exe, job], capture_output=True, text=True, timeout=300,
                       env=dict(os.environ, TSAN_OPTIONS="halt_on_error=1"))
    assert r.returncode == 0, r.stderr[-4000:]
