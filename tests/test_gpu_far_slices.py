"""Slices of macroparticles far outside the binning range, where the turn's approximate
slice index is used for its side alone: below and above by 1e6 slices and a few around
it, by 8e6 (where the index's spacing passes the margin of its test), near 2^31 (past
which the conversion of the reference's expression turns over and counts above as
below) and beyond, alone and beside ordinary ones, in the statistics pass and in the
turn's, for the plain variant and those with dipole histograms and excitation.  Slice
counts and counters against the oracle, bit for bit, over three turns."""
import numpy as np
import pytest

import mtrack_amd as m
import oracle as o
from mtrack_amd import confgen as cg
from variants import L20

pytestmark = pytest.mark.gpu

RES = [("resonator_%d" % (i + 1), {"Rs": rs, "fres": f, "Qfactor": 1.0, "plane": p})
       for i, (p, rs, f) in enumerate((("LON", 5e3, 10.0), ("VER", 2e5, 8.0), ("HOR", 2e5, 8.0)))]
FAR = [1e6 - 3, 1e6 - 0.5, 1e6, 1e6 + 0.5, 1e6 + 2, 3e6 + 0.25, 8e6, 8e6 + 0.5, 1e8, 1e9, 2.147e9, 2147483000.0,
       2147483640.0, 2147483647.0, 2147483648.0, 2147483649.0, 2147483660.0, 2.2e9, 1e10]


@pytest.mark.parametrize("name,qe,nres", [("plain", 0, 1), ("dipoles", 0, 3), ("excitation", 1, 1), ("both", 1, 3)])
@pytest.mark.parametrize("np_", [len(FAR), 300])
def test_side_of_far_slices(tmp_path, name, qe, nres, np_):
    print("case", name, np_, flush=True)
    d = str(tmp_path)
    text = cg.ring_conf(sections={"selffield": {"Ncell": 50, "Nsigma": 5.0},
                                  "tracking": {"NrevTot": 4, "NrevMon": 2, "EnableQuantum": qe},
                                  "ring": {"Lc": L20, "Iring": 10.0}, "distribution": {"Np": np_}},
                        extra_sections=RES[:nres])
    cfg = m.Config(cg.write(d + "/far.conf", text), d + "/")
    orc, g = o.OracleRing(cfg, o.RNG_PHILOX), m.Ring(cfg)
    for b in range(cfg.geti("Nbunch")):
        q = orc.get_bunch(b).copy()
        v = np.array(FAR) * (1.0 if b % 2 else -1.0) + (b // 2) * 0.125
        q[0, np.arange(len(FAR)) * (np_ // len(FAR))] = -((v - 1) * cfg.get("dT") - cfg.get("Nsigma")) * cfg.get("sigma_tau")
        orc.set_bunch(b, q)
        g.set_bunch(b, q)
    orc.prepare()
    g.prepare()
    for turn in range(4):
        ho, to = orc.histograms()
        hg, tg = g.histograms()
        assert np.array_equal(ho, hg) and np.array_equal(to, tg), turn
        if turn < 3:
            orc.track(1)
            g.track(1)
    g.close()
