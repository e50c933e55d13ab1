"""The LDS slots that the passes of a line FFT exchange their values through
(csrc/fft_device.hpp), replayed on the host for every compiled plan: a slot is
rewritten only by the thread that read it last, which is what lets an exchange
run with one barrier, and every pass finds its inputs (exchange_slots.cpp)."""
import os
import subprocess

from imresh_amd import build

HERE = os.path.dirname(os.path.abspath(__file__))


def test_slots_of_every_plan(tmp_path):
    exe = str(tmp_path / "slots")
    r = subprocess.run([build.hipcc(), "-x", "hip", os.path.join(HERE, "exchange_slots.cpp"), "-o", exe, "-O1",
                        "--offload-arch=gfx950", "-std=c++17", "-w", "-Xclang", "-target-feature", "-Xclang",
                        "-packed-fp32-ops", "-I", build.CSRC, "-I", os.path.join(build.ROOT, "include")],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stdout + r.stderr
    r = subprocess.run([exe], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout + r.stderr
