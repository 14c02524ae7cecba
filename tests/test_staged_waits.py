"""The staged K-split fused GEMM's written waits are enough by themselves: what the compiler makes of them needs none of its own.

A stage in LDS is filled by direct loads and read behind a wait that counts the loads in flight.  The compiler follows which array such a load
fills and adds a wait of its own where it finds the written one too lax; a kernel that needs these is right by the compiler's grace only."""
import os
import re
import subprocess

import pytest

import build as native_build


def _kernels(path):
    """The instructions of every instance of the kernel behind its tables' barrier, by rows staged."""
    rows, found = None, {}
    with open(path) as f:
        for line in f:
            m = re.match(r"_ZN2ap17gemms_kbit_kernelILi\d+ELi(\d+)E\w*:", line)
            if m:
                rows = int(m.group(1))
                found[rows] = []
            elif line.startswith(".Lfunc_end"):
                rows = None
            elif rows is not None:
                found[rows].append(line.strip())
    for rows, lines in found.items():
        found[rows] = lines[next(i for i, l in enumerate(lines) if l.startswith("s_barrier")) + 1:]
    return found


@pytest.mark.parametrize("bits", range(3, 9))
def test_no_read_of_a_stage_needs_a_wait_of_the_compiler(bits, tmp_path):
    flags = [f for f in native_build.HIPCC_FLAGS if f not in ("-shared", "-Wall")]
    listing = str(tmp_path / "listing.s")
    subprocess.run([native_build._hipcc(), *flags, "-I", native_build.INCLUDE, "-I", native_build.CSRC, "--cuda-device-only", "-S",
                    f"-DAP_BITS={bits}", os.path.join(native_build.CSRC, "ap_gemms_inst.hip"), "-o", listing], check=True, capture_output=True)
    kernels = _kernels(listing)
    assert sorted(kernels) == [4, 8, 16, 32]
    for rows, lines in kernels.items():
        waits, products, spilled, refills = [], 0, False, 0
        for line in lines:
            if line.startswith("v_mfma") or line.startswith("s_cbranch") or line.startswith(".LBB"):
                # ahead of a product stands one written wait at most (registers that were spilled have waits of their own)
                assert not line.startswith("v_mfma") or len(waits) < 2 or spilled, (bits, rows, waits)
                products += line.startswith("v_mfma")
                waits, spilled = [], False
            elif line.startswith("scratch_"):
                spilled = True
            elif line.startswith("s_waitcnt") and "vmcnt" in line:
                waits.append(line)
            elif line.startswith("buffer_load") and line.endswith("lds"):
                refills += 1
        assert products >= 3 * 16 and refills >= rows       # the listing is that of the kernel: the three forms of a step, a ring refilled
