"""Weak-strong bunches whose resistive wall has no past turn to act from (Nmlt below 0,
which the configuration accepts): no kicks, the same bits as with the wall off."""
import numpy as np
import pytest

import mtrack_amd as m
from mtrack_amd import confgen as cg

pytestmark = pytest.mark.gpu


def conf(d, rw, nmlt):
    cg.filling_file(d + "/fill.txt", range(7), out=())
    text = cg.ring_conf(sections={
        "tracking": {"BunchModel": "STRONG", "EnableFBII": 0, "NrevTot": 20, "NrevMon": 5, "EnableRW_long": rw,
                     "Nmlt": nmlt, "EnableQuantum": 0, "filling": d + "/fill.txt"},
        "ring": {"Lc": cg.small_ring(20), "Iring": 20.0, "rhorw": 1.7e-8, "beffL1": 0.012, "beffL2": 0.012,
                 "beffH3": 0.012, "beffV3": 0.012},
        "distribution": {"Np": 2000, "Nslc": 20}})
    return m.Config(cg.write(d + "/ws%d_%d.conf" % (rw, nmlt), text), d + "/")


@pytest.mark.parametrize("nmlt", [-1, -2, -5])
def test_no_history(tmp_path, nmlt):
    d = str(tmp_path)
    a, b = m.WeakStrong(conf(d, 1, nmlt)), m.WeakStrong(conf(d, 0, 3))
    for x, y in zip(a.track(12), b.track(12)):
        assert np.array_equal(x, y)
    for k in range(a.Nb):
        assert np.array_equal(a.slices(k), b.slices(k))
