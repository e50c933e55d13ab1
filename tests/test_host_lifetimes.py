"""Lifetimes of streams, events and requests in the server and the batch,
checked on the host against a stand-in runtime (host_lifetimes.cpp), the
server's threads under the thread sanitizer."""
import os
import subprocess

from imresh_amd import build

HERE = os.path.dirname(os.path.abspath(__file__))


def test_lifetimes(tmp_path):
    obj, exe = str(tmp_path / "lifetimes.o"), str(tmp_path / "lifetimes")
    threads = ["-Xarch_host", "-fsanitize=thread"]
    for cmd in ([build.hipcc(), "-x", "hip", "--offload-host-only", "--offload-arch=gfx950", "-c", "-g", "-O1",
                 "-std=c++17", "-w", *threads, "-I", build.CSRC, "-I", os.path.join(build.ROOT, "include"),
                 os.path.join(HERE, "host_lifetimes.cpp"), "-o", obj],
                ["/opt/rocm/llvm/bin/clang++", *threads, "-g", obj, "-o", exe, "-lpthread"], [exe]):
        r = subprocess.run(cmd, capture_output=True, text=True, timeout=300)
        assert r.returncode == 0, r.stdout + r.stderr
