"""Macroparticles outside the range of the turn's fast forms: on a slice's edge to
the last bits (both the kick's slice and the next histogram's), far beyond the
binning range (slice index past 1e6), phases past the range of the sine's
reduction, beside ordinary ones in the same waves -- first, last, and at the
borders of a work-group's rows, for the variants of the turn with excitation,
dipole histograms and harmonic cavity and for the plain one.

Against the oracle on the same coordinates, two turns: slice counts and counters
bit for bit, every coordinate within 1e-12 of the larger of its own magnitude and
the rms of the ordinary macroparticles (the same operations; the device's sine
and the oracle's differ by one unit in the last place, 1.1e-16, which a turn
multiplies by the voltage and the tune's phase, at most about 1e3).
"""
import numpy as np
import pytest

import mtrack_amd as m
import oracle as o
from mtrack_amd import confgen as cg

pytestmark = pytest.mark.gpu

RES = [("resonator_%d" % (i + 1), {"Rs": rs, "fres": f, "Qfactor": 1.0, "plane": p})
       for i, (p, rs, f) in enumerate((("LON", 5e3, 10.0), ("VER", 2e5, 8.0), ("HOR", 2e5, 8.0)))]
VARIANTS = {"plain": (0, 1, {}), "dipoles": (0, 3, {}), "excitation": (1, 1, {}), "both": (1, 3, {}),
            "cavity": (1, 3, {"EnableIdealHC": 1})}


@pytest.mark.parametrize("np_", [1, 257, 1500])
@pytest.mark.parametrize("name", sorted(VARIANTS))
def test_outside_the_fast_range(tmp_path, name, np_):
    qe, nres, tracking = VARIANTS[name]
    d = str(tmp_path)
    ring = {"Lc": cg.small_ring(4), "Iring": 10.0, "mIdeal": 3, "CHH": 100.0, "CVV": 70.0} if tracking else {
        "Lc": cg.small_ring(4), "Iring": 10.0}
    text = cg.ring_conf(sections={"selffield": {"Ncell": 50, "Nsigma": 5.0},
                                  "tracking": dict(tracking, NrevTot=4, NrevMon=2, EnableQuantum=qe), "ring": ring,
                                  "distribution": {"Np": np_}}, extra_sections=RES[:nres])
    cfg = m.Config(cg.write(d + "/fast.conf", text), d + "/")
    orc, g = o.OracleRing(cfg, o.RNG_PHILOX), m.Ring(cfg)
    sigma, dT = cfg.get("sigma_tau"), cfg.get("dT")
    for b in range(cfg.geti("Nbunch")):
        q = orc.get_bunch(b).copy()
        odd = sorted({0, np_ // 2, min(255, np_ - 1), min(256, np_ - 1), np_ - 1})
        for k, i in enumerate(odd):
            # a slice's edge, its neighbours in the last bit, and far away
            edge = -(((20 + k) - 1) * dT - 5.0) * sigma
            q[0, i] = (edge, np.nextafter(edge, 1), -1e-3, edge, 2e-3)[(k + b) % 5]
        orc.set_bunch(b, q)
        g.set_bunch(b, q)
    orc.prepare()
    g.prepare()
    for _ in range(2):
        orc.track(1)
        g.track(1)
        ho, to = orc.histograms()
        hg, tg = g.histograms()
        assert np.array_equal(ho, hg) and np.array_equal(to, tg)
        for b in range(cfg.geti("Nbunch")):
            a, r = g.get_bunch(b), orc.get_bunch(b)
            ordinary = np.abs(r[0]) < 1e-9
            rms = r[:, ordinary].std(1, keepdims=True) if ordinary.sum() > 1 else np.zeros((6, 1))
            assert np.all(np.abs(a - r) <= 1e-12 * np.maximum(np.abs(r), rms))
    g.close()
