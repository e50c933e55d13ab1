"""The exact shortcuts of the Poisson sampler (csrc/poisson_device.hpp), which
have to leave every sample unchanged, checked on the host (poisson_exact.cpp)."""
import os
import subprocess

from imresh_amd import build

HERE = os.path.dirname(os.path.abspath(__file__))


def test_shortcuts_are_exact(tmp_path):
    exe = str(tmp_path / "poisson")
    r = subprocess.run(["g++", "-O2", "-std=c++17", "-ffp-contract=off", "-I", build.CSRC,
                        os.path.join(HERE, "poisson_exact.cpp"), "-o", exe], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout + r.stderr
    r = subprocess.run([exe], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout + r.stderr
