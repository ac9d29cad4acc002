"""The ion-parallel train at the edges of its loops: slice counts below, at and past
a group of four and a chunk of eight, up to the capacity; bunches with fewer ions than
a block, so that a block's ions have many creators, and a block's last lanes with none.

Against the bunch-by-bunch relay, which looks its fields up by another formula and
adds in another order, on the same field tables: within 1e-12 of each output's largest
magnitude over two turns (a field at 1e-16 per slice, at most fifty slices a bunch and
thirty bunches of them in a row).
"""
import numpy as np
import pytest

import mtrack_amd as m
from mtrack_amd import confgen as cg

pytestmark = pytest.mark.gpu
RTOL = 1e-12


@pytest.mark.parametrize("nslc,bunches", [(1, 2), (1, 30), (2, 11), (3, 30), (4, 30), (7, 5), (8, 30), (11, 30),
                                          (24, 30)])
def test_slice_counts(tmp_path, nslc, bunches):
    d = str(tmp_path)
    cg.filling_file(d + "/fill.txt", list(range(bunches)), out=())
    text = cg.ring_conf(sections={
        "tracking": {"BunchModel": "STRONG", "EnableFBII": 1, "NrevTot": 100, "NrevMon": 1, "EnableRW_long": 0,
                     "EnableQuantum": 0, "filling": d + "/fill.txt"},
        "ring": {"Lc": cg.small_ring(40), "Iring": 20.0},
        "distribution": {"Np": 2000, "Nslc": nslc}})
    cfg = m.Config(cg.write(d + "/ws.conf", text), d + "/")
    print("case", nslc, bunches, flush=True)
    out = []
    for serial in (False, True):
        w = m.WeakStrong(cfg, serial_train=serial)
        out.append(list(w.track(2)) + [w.slices(k).T for k in range(bunches)])
        w.close()
    for a, b in zip(*out):
        a, b = np.asarray(a), np.asarray(b)
        # one slice a side has no field (0 / 0 in its spacing): not a number in both
        assert np.array_equal(np.isnan(a), np.isnan(b))
        a, b = np.nan_to_num(a), np.nan_to_num(b)
        err = np.abs(a - b).max(axis=tuple(range(a.ndim - 1)))
        top = np.abs(b).max(axis=tuple(range(b.ndim - 1)))
        assert np.all(err <= RTOL * np.maximum(top, 1e-300))
