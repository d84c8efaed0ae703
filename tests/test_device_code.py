"""The walk reads some of its arguments from the kernel's argument segment.

Only a kernel has that segment's address: in a device function that is called
and not inlined the address means nothing, and every pointer read through it
would be wild. Without optimisation the compiler inlines only what it is told
to, so in that form of the device code no function but the kernels may ask
for the address."""
import os
import re
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "amt-bh-benchmark_amd", "csrc")
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="no hipcc")
def test_argument_segment_is_read_in_kernels_only(tmp_path):
    out = tmp_path / "walk.ll"
    subprocess.run([HIPCC, "--offload-arch=gfx950", "-O0", "-std=c++17", "--offload-device-only", "-S", "-emit-llvm",
                    "-ffp-contract=off", "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops", "-o", str(out),
                    os.path.join(CSRC, "bh_walk.hip")], check=True, capture_output=True)
    kernels, others, inside = 0, [], None
    for line in out.read_text().splitlines():
        head = re.match(r"define .*?@([\w.$]+)\(", line)
        if head:
            inside, kernel = head.group(1), "amdgpu_kernel" in line
        elif "call" in line and "llvm.amdgcn.kernarg.segment.ptr" in line:
            kernels += kernel
            if not kernel:
                others.append(inside)
    assert kernels > 0
    assert not others, others
