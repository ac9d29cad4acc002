"""The interval of the current scan (NrevScan) by its magnitude: the reference takes
the turn number modulo it, (rev + 1) % NrevScan == 0 (src/tracking.c:43-59), which a
negative interval satisfies on the same turns as its magnitude.  The scan's steps and the
resistive wall's trigger, which counts turns since the last step, against the oracle
(the signed remainder) over 60 turns, past the trigger's fifty: within 1e-12, the bound
of the other parity tests; the trigger also without a current scan to end each turn.
"""
import numpy as np
import pytest

import mtrack_amd as m
import oracle as o
from mtrack_amd import confgen as cg
from test_gpu_parity import RTOL, stat_errors
from variants import BBR_L, L20, RW

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("scan_type", [1, 2])
@pytest.mark.parametrize("every", [7, -7, -55])
def test_signed_interval(tmp_path, scan_type, every):
    print("case", scan_type, every, flush=True)
    d = str(tmp_path)
    text = cg.ring_conf(sections={"selffield": {"Ncell": 40, "Nsigma": 5.0},
                                  "tracking": {"NrevTot": 60, "NrevMon": 10, "EnableRW_long": 1, "Nmlt": 2,
                                               "triggerRW": 1},
                                  "ring": dict(RW, Lc=L20, Iring=40.0), "distribution": {"Np": 200}},
                        extra_sections=[BBR_L, ("scan", {"scan_type": scan_type, "Nscan": 60, "NrevScan": every,
                                                         "scan_start": 20.0, "scan_step": 10.0})])
    cfg = m.Config(cg.write(d + "/scan.conf", text), d + "/")
    orc, g = o.OracleRing(cfg, o.RNG_PHILOX), m.Ring(cfg)
    orc.prepare()
    g.prepare()
    ost, gst = orc.track(60)[0], g.track(60)[0]
    assert stat_errors(gst, ost).max() <= RTOL
    g.close()
