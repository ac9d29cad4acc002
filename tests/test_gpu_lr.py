"""The long-range resonators' phasor scan, slice sums and own-wake convolutions at
the edges of their ranges: fewer buckets than one lane's share (8) and than a
wave has lanes, more than one pass of the scan (512 buckets), rings past 1,365
buckets, more resonators than a block has waves, odd and even slice counts from
two up, slice counts whose own wakes no longer fit the reduction's LDS, samples
kept from less and from more than a turn, and a bunch with macroparticles beyond
the binning range (the recurrence drops them, the selffield keeps them in the
edge slices).

Against the oracle (the recurrence slice by slice) on the same inputs: centroids,
rms, RF phase and voltage within 1e-12, the bound of the other parity tests --
the scan's rounding grows with its depth (about 30 products), the recurrence's
with its length, both far below it.
"""
import numpy as np
import pytest

import mtrack_amd as m
import oracle as o
from mtrack_amd import confgen as cg
from test_gpu_parity import RTOL, stat_errors

pytestmark = pytest.mark.gpu

FB = ("rf_feedback", {"resonator": 1, "averaging_length": 30})
MAIN = ("harmonic_cavity_1", {"m": 1, "Rs": 5e6, "detune": -40e3, "Qfactor": 4e4})
THIRD = ("harmonic_cavity_2", {"m": 3, "Rs": 2e6, "detune": 50e3, "Qfactor": 2e4})
BBR = [("resonator_%d" % (i + 1), {"Rs": rs, "fres": f, "Qfactor": 1.0, "plane": p})
       for i, (p, rs, f) in enumerate((("LON", 5e3, 10.0), ("VER", 2e5, 8.0), ("HOR", 2e5, 8.0)))]


def modes(n, planes):
    return [("longrange_resonator_%d" % (i + 1), {"plane": planes[i % len(planes)], "fres": 0.7 + 0.13 * i, "Rs": 1e5,
                                                  "Qfactor": 3e3}) for i in range(n)]


def fb(length):
    return ("rf_feedback", {"resonator": 1, "averaging_length": length})


CASES = {
    "three_buckets": (3, 2, 2, 5.0, [MAIN, fb(5)]),
    "seven_modes": (20, 20, 41, 5.0, [MAIN, THIRD, fb(30)] + modes(5, ["HOR", "VER", "LON"]) + BBR),
    "long_average": (63, 9, 40, 5.0, [MAIN, fb(1000)]),
    "two_passes": (513, 11, 17, 5.0, [MAIN, THIRD, fb(700)]),
    "old_limit": (1400, 5, 30, 5.0, [MAIN, fb(3000)]),
    "trash": (65, 8, 10, 1.0, [MAIN, fb(30)] + modes(2, ["VER", "HOR"]) + BBR),
    "many_slices": (20, 3, 1000, 5.0, [MAIN, fb(30)] + modes(1, ["VER"]) + BBR),
}


@pytest.mark.parametrize("name", sorted(CASES))
def test_lr_matches_oracle(tmp_path, name):
    h, bunches, ncell, nsig, extra = CASES[name]
    print("case", name, flush=True)
    d = str(tmp_path)
    fill = d + "/fill.txt"
    cg.filling_file(fill, [int(k * h / bunches) for k in range(bunches)], out=(0,))
    text = cg.ring_conf(sections={"selffield": {"Ncell": ncell, "Nsigma": nsig},
                                  "tracking": {"NrevTot": 12, "filling": fill},
                                  "ring": {"Lc": cg.small_ring(h), "Iring": 100.0, "rhorw": 1.7e-8, "beffL1": 0.012,
                                           "beffL2": 0.012, "beffH3": 0.012, "beffV3": 0.012},
                                  "distribution": {"Np": 301}}, extra_sections=extra)
    cfg = m.Config(cg.write(d + "/lr.conf", text), d + "/")
    orc = o.OracleRing(cfg, o.RNG_PHILOX)
    orc.prepare()
    ost, _, orf = orc.track(12)
    g = m.Ring(cfg)
    g.prepare()
    gst, _, grf = g.track(12)
    assert stat_errors(gst, ost).max() <= RTOL
    assert (np.abs(grf - orf) / np.abs(orf)).max() <= RTOL
    ho, to = orc.histograms()
    hg, tg = g.histograms()
    assert np.array_equal(ho, hg) and np.array_equal(to, tg)
    g.close()
