"""Slice dipole sums of the passes against exact integer sums of the coordinates the
device holds: the sum over a slice's macroparticles of round(x 2^100), ties to even,
converted to double (within one unit in the last place and 2^-89 m, half the spacing of
doubles at the low word's 2^64 quanta, which a negative sum's conversion rounds to).
Coordinates just below the per-particle bound min(2^20, 2^27 / Np) of one sign and of
both, far below a metre's last place, in a few slices and beyond the binning range (those join the edge slices);
fewer macroparticles than a work-group, and several work-groups; the statistics pass
(prepare) and the turn's own, with and without excitation.  The transverse wakes that
ask for the sums are too weak to move anything.
"""
from fractions import Fraction

import numpy as np
import pytest

import mtrack_amd as m
from mtrack_amd import confgen as cg

pytestmark = pytest.mark.gpu
TWO100 = 1 << 100
WEAK = [("resonator_%d" % (i + 1), {"Rs": 1e-30, "fres": 8.0, "Qfactor": 1.0, "plane": p})
        for i, p in enumerate(("VER", "HOR"))]


def slices(tau, cfg):
    v = (-tau / cfg.get("sigma_tau") + cfg.get("Nsigma")) / cfg.get("dT") + 1
    return np.clip(np.trunc(v).astype(int), 0, cfg.geti("Ncell") - 1)


def check(ring, cfg, b):
    q, p = ring.get_bunch(b), ring.potentials(b)[0]
    sl = slices(q[0], cfg)
    for row, u in ((4, q[4]), (6, q[2])):
        for s in range(cfg.geti("Ncell")):
            exact = float(Fraction(sum(round(Fraction(float(x)) * TWO100) for x in u[sl == s]), TWO100))
            assert abs(p[row, s] - exact) <= np.spacing(abs(exact)) + 2.0 ** -89, (b, row, s)


@pytest.mark.parametrize("qe", [0, 1])
@pytest.mark.parametrize("np_", [1, 100, 129, 3000])
def test_sums_are_exact(tmp_path, np_, qe):
    print("case", np_, qe, flush=True)
    d = str(tmp_path)
    text = cg.ring_conf(sections={"selffield": {"Ncell": 40, "Nsigma": 5.0},
                                  "tracking": {"NrevTot": 4, "NrevMon": 2, "EnableQuantum": qe},
                                  "ring": {"Lc": cg.small_ring(4), "Iring": 1.0}, "distribution": {"Np": np_}},
                        extra_sections=WEAK)
    cfg = m.Config(cg.write(d + "/dip.conf", text), d + "/")
    g = m.Ring(cfg)
    rng = np.random.default_rng(np_ + qe)
    top = np.nextafter(134217728.0 / np_ if np_ > 128 else 1048576.0, 0.0)
    sizes = [np.full(np_, top), top * rng.choice([-1.0, 1.0], np_), -top * rng.uniform(0.0, 1.0, np_),
             2.0 ** rng.uniform(-105, -50, np_) * rng.choice([-1.0, 1.0], np_)]
    for b in range(cfg.geti("Nbunch")):
        q = np.zeros((6, np_))
        at = rng.choice([-3.0, 5.5, 20.5, 21.5, 47.0], np_)  # slices, two of them outside
        q[0] = -((at - 1) * cfg.get("dT") - cfg.get("Nsigma")) * cfg.get("sigma_tau")
        q[2], q[4] = sizes[b], sizes[b][::-1]
        g.set_bunch(b, q)
    g.prepare()
    for b in range(cfg.geti("Nbunch")):
        check(g, cfg, b)
    g.track(1)
    for b in range(cfg.geti("Nbunch")):
        check(g, cfg, b)
    g.close()
