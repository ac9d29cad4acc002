"""Alignment of the dynamic LDS arrays of the weak-strong kernels: their ordered sums
read 16 bytes at a time, so every such array asks the compiler for 16 bytes (as an
array of doubles it would get 8, and sit on 16 only as long as the arrays before it
happen to end there).  Checked on the compiler's own record of the arrays."""
import os
import re
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_weak_strong_dynamic_lds(tmp_path):
    hipcc, out = "/opt/rocm/bin/hipcc", str(tmp_path / "ws.ll")
    if not os.path.exists(hipcc):
        pytest.skip("hipcc not available")
    subprocess.run([hipcc, "-O0", "-std=c++17", "--offload-arch=gfx950", "--offload-device-only", "-S", "-emit-llvm",
                    "-I" + os.path.join(ROOT, "include"), "-o", out,
                    os.path.join(ROOT, "mtrack_amd", "csrc", "ws.hip")], check=True, capture_output=True)
    with open(out) as f:
        arrays = re.findall(r"^@(\S+) = external .*addrspace\(3\) global \[0 x .*align (\d+)", f.read(), re.M)
    assert arrays
    assert all(int(align) >= 16 for _, align in arrays), arrays
