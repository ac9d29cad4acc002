"""The fused electron-side launch of the weak-strong turn (phase 2 of one turn,
phase 1 of the next, the resistive wall from a ring of dipole rows) at the edges
of its ranges: one bunch, more bunches than a block has lanes, the deepest
history (30 turns, the row being written beside it), the history message's cut
at 5,000 doubles, the trigger's change of wake at turn 50, and calls of uneven
length, whose last launch ends the turn that a longer call would have carried
into the next.

Against the oracle within 1e-12 of each output's largest magnitude (the bound of
the other weak-strong tests: the same operations in the same order but for
the device's sin); calls of uneven length against one call bit for bit.
"""
import numpy as np
import pytest

import mtrack_amd as m
import oracle as o
from mtrack_amd import confgen as cg

pytestmark = pytest.mark.gpu
RTOL = 1e-12


def write(d, h, bunches, nmlt, trigger=0, fbii=0):
    fill = d + "/fill.txt"
    cg.filling_file(fill, [int(k * h / bunches) for k in range(bunches)], out=())
    text = cg.ring_conf(sections={
        "tracking": {"BunchModel": "STRONG", "EnableFBII": fbii, "NrevTot": 100, "NrevMon": 7, "EnableRW_long": 1,
                     "Nmlt": nmlt, "EnableQuantum": 0, "triggerRW": trigger, "filling": fill},
        "ring": {"Lc": cg.small_ring(h), "Iring": 20.0, "rhorw": 1.7e-8, "beffL1": 0.012, "beffL2": 0.012,
                 "beffH3": 0.012, "beffV3": 0.012},
        "distribution": {"Np": 2000, "Nslc": 20}})
    return m.Config(cg.write(d + "/ws.conf", text), d + "/")


@pytest.mark.parametrize("h,bunches,nmlt,trigger,turns", [
    (20, 1, 3, 0, 12), (20, 20, 28, 0, 40), (416, 416, 2, 0, 8), (416, 300, 28, 0, 35), (20, 7, 1, 1, 55)])
def test_step_matches_oracle(tmp_path, h, bunches, nmlt, trigger, turns):
    cfg = write(str(tmp_path), h, bunches, nmlt, trigger)
    print("case", h, bunches, nmlt, trigger, turns, flush=True)
    orc = o.OracleWS(cfg, 1)
    ref = orc.track(turns)
    g = m.WeakStrong(cfg)
    got = g.track(turns)
    for a, b in zip(got, ref[:4]):
        a, b = np.asarray(a), np.asarray(b)
        err = np.abs(a - b).max(axis=tuple(range(a.ndim - 1))) / np.maximum(np.abs(b).max(axis=tuple(range(b.ndim - 1))),
                                                                            1e-300)
        assert err.max() <= RTOL
    for ib in (0, g.Nb - 1):
        a, b = g.slices(ib), orc.slices(ib)
        assert np.all(np.abs(a - b).max(1) <= RTOL * np.abs(b).max(1))


@pytest.mark.parametrize("fbii", [0, 1])
def test_calls_of_uneven_length(tmp_path, fbii):
    cfg = write(str(tmp_path), 20, 7, 4, fbii=fbii)
    a, b = m.WeakStrong(cfg), m.WeakStrong(cfg)
    whole = a.track(15)
    parts = [b.track(n) for n in (1, 2, 5, 1, 6)]
    for k in range(4):
        assert np.array_equal(whole[k], np.concatenate([p[k] for p in parts]))
    for ib in range(a.Nb):
        assert np.array_equal(a.slices(ib), b.slices(ib))
