"""The excitation's normals on the device (mtrack_amd/csrc/qe_dev.h) are the oracle's bit
for bit: the Box-Muller radius and the sine and cosine over all 2^24 inputs each has
(a reciprocal, a square root and two reductions take other steps than the oracle's), and
the five normals of a million macroparticle-turns (Philox keys, counters past 2^32)."""
import os
import subprocess

import pytest

import oracle as o

pytestmark = pytest.mark.gpu
ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_every_input(tmp_path):
    o.lib()
    exe = str(tmp_path / "qe_check")
    subprocess.run(["/opt/rocm/bin/hipcc", "-O3", "-std=c++17", "--offload-arch=gfx950", "-ffp-contract=off", "-Xclang",
                    "-target-feature", "-Xclang", "-packed-fp32-ops", "-I" + os.path.join(ROOT, "mtrack_amd", "csrc"),
                    "-o", exe, os.path.join(ROOT, "tests", "qe_check.hip"), "-ldl"], check=True, capture_output=True)
    print("compiled", flush=True)
    out = subprocess.run([exe, o.LIBPATH], capture_output=True, text=True, timeout=60)
    assert out.returncode == 0, out.stderr
    assert out.stdout.strip() == "radius 0 sine 0 cosine 0 normals 0"
