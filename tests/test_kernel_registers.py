"""Registers of the built kernels: the compiler keeps every kernel's values in
registers, but for a few.  (A row pass that merged two guarded loops over
arrays it had not initialised spilled 1849 registers, 1.2 KiB per lane, and
still computed the right bits.)"""
import re
import struct
import subprocess
import tempfile

import imresh_amd as im

READELF = "/opt/rocm/llvm/bin/llvm-readelf"
BUNDLE = b"__CLANG_OFFLOAD_BUNDLE__"
# the most today: 6 registers, 28 bytes (Bluestein rows of 16384-point convolutions)
MAX_SPILLS, MAX_SCRATCH = 8, 32


def kernel_metadata(lib):
    """symbol -> (spilled vector registers, scratch bytes per lane)"""
    data, out = open(lib, "rb").read(), {}
    at = data.find(BUNDLE)
    while at >= 0:
        (count,) = struct.unpack_from("<Q", data, at + len(BUNDLE))
        entry = at + len(BUNDLE) + 8
        for _ in range(count):
            offset, size, length = struct.unpack_from("<QQQ", data, entry)
            target = data[entry + 24:entry + 24 + length]
            entry += 24 + length
            if b"gfx950" not in target or size == 0:
                continue
            with tempfile.NamedTemporaryFile() as f:
                f.write(data[at + offset:at + offset + size])
                f.flush()
                text = subprocess.run([READELF, "--notes", f.name], capture_output=True, text=True,
                                      check=True).stdout
            for kernel in re.findall(r"\.private_segment_fixed_size:.*?\.wavefront_size", text, re.S):
                scratch, symbol, spills = (re.search(p, kernel).group(1) for p in (
                    r"\.private_segment_fixed_size: (\d+)", r"\.symbol:\s+(\S+)", r"\.vgpr_spill_count: (\d+)"))
                out[symbol] = int(spills), int(scratch)
        at = data.find(BUNDLE, entry)
    return out


def test_kernels_do_not_spill():
    kernels = kernel_metadata(im.LIB_PATH)
    assert sum("k_row" in k for k in kernels) > 100 and sum("k_col" in k for k in kernels) > 100
    over = {k: v for k, v in kernels.items() if v[0] > MAX_SPILLS or v[1] > MAX_SCRATCH}
    assert not over, over
    columns = {k: v for k, v in kernels.items() if "k_col" in k and v[0] > 0}
    assert not columns, columns


def test_four_step_columns_have_no_projection_kernel():
    # columns of 8192 points project in the four-step pass, whose middle step
    # is the 1024-point kernel: variants of their own would never be launched,
    # yet timed against each other on the first call of a size
    plain = [k for k in kernel_metadata(im.LIB_PATH) if re.search(r"k_col\w+PlanEILi16ELi8192E.*Lb0EEE", k)]
    assert len(plain) == 4   # forward and inverse, complex and real input
