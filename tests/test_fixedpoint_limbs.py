"""The three limbs in which the turn pass forms its exact dipole sums
(fx_limbs, fx_fold of mtrack_amd/csrc/fixedpoint.h; a host build of the functions
the kernel runs): each double x becomes round(x 2^100), ties to even, checked
against exact rational arithmetic -- single values of every size down to the
quantum and below, of both signs, ties, the largest below the per-particle bounds
min(2^20, 2^27 / Np) -- and the sums of whole work-groups (up to 64 values for each
of 256 lanes) and of bunches of several are the exact sums of those integers.
"""
import os
import struct
import subprocess
from fractions import Fraction

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
TWO100 = 1 << 100
GROUP = 64 * 256


@pytest.fixture(scope="module")
def driver(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("fx") / "fx_limbs_check")
    hipcc = "/opt/rocm/bin/hipcc"
    if not os.path.exists(hipcc):
        pytest.skip("hipcc not available")
    subprocess.run([hipcc, "-x", "hip", "-O2", "--offload-arch=gfx950", "-ffp-contract=off", "-I",
                    os.path.join(ROOT, "mtrack_amd", "csrc"), os.path.join(ROOT, "tests", "fx_limbs_check.cpp"), "-o",
                    exe], check=True, capture_output=True)
    return exe


def signed128(hi, lo):
    v = (int(hi, 16) << 64) | int(lo, 16)
    return v - (1 << 128) if v >> 127 else v


def check(exe, xs, block=GROUP):
    bits = ["%016x" % struct.unpack("<Q", struct.pack("<d", float(x)))[0] for x in xs]
    out = subprocess.run([exe], input="%d %d\n" % (len(xs), block) + "\n".join(bits) + "\n", capture_output=True,
                         text=True, check=True).stdout.split("\n")
    want = [round(Fraction(float(x)) * TWO100) for x in xs]  # Fraction rounds ties to even
    assert [signed128(*line.split()) for line in out[:len(xs)]] == want
    _, hi, lo, vb = out[len(xs)].split()
    assert signed128(hi, lo) == sum(want)
    v, ref = struct.unpack("<d", struct.pack("<Q", int(vb, 16)))[0], float(Fraction(sum(want), TWO100))
    assert abs(v - ref) <= np.spacing(abs(ref)) if ref else v == 0
    return sum(want)


def test_single_values(driver):
    rng = np.random.default_rng(11)
    size = 2.0 ** rng.uniform(-110, 20, 4000)
    check(driver, np.concatenate([size * rng.choice([-1.0, 1.0], 4000), rng.normal(0, 1e-4, 2000),
                                  [0.0, -0.0, 5e-324, -5e-324, 2.0 ** -1022]]), block=7)


def test_ties(driver):
    """Odd multiples of half the quantum, alone and beside bits of the upper limbs,
    and ties of the upper limbs themselves (not ties of the whole integer)."""
    q = 2.0 ** -100
    odd = np.concatenate([np.arange(1.0, 40.0, 2.0), 2.0 ** 39 - np.arange(1.0, 10.0, 2.0), 2.0 ** 52 + np.arange(1.0, 9.0, 2.0)])
    xs = [odd * q / 2, -odd * q / 2]
    for half in (2.0 ** -21, 2.0 ** -61):
        k = np.arange(1.0, 12.0, 2.0)
        xs += [k * half, -k * half, k * half * (1 + 2.0 ** -40), 1 + k * half, k * half + q, -k * half - q]
    check(driver, np.concatenate(xs), block=3)


@pytest.mark.parametrize("np_", [1, 128, 129, GROUP - 1, GROUP, GROUP + 1, 100000])
def test_extremes(driver, np_):
    lim = 134217728.0 / np_ if np_ > 128 else 1048576.0
    top = np.nextafter(lim, 0.0)
    for sign in (1.0, -1.0):
        assert abs(check(driver, [sign * top] * np_)) < (1 << 127)
    check(driver, [top if k % 3 else -top / 7 for k in range(np_)])


def test_carries_between_limbs(driver):
    """Values whose lower limbs are as negative as they get, whose sums borrow from
    the limbs above, and sums that pass through zero."""
    x = 1.0 + 2.0 ** -21 - 2.0 ** -52
    check(driver, [x] * 5000 + [-x] * 5001)
    check(driver, [2.0 ** -61 - 2.0 ** -100] * GROUP)
    check(driver, [-(2.0 ** -21 - 2.0 ** -60)] * GROUP)
