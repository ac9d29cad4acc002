"""What the ion-parallel train's comparisons with the bunch-by-bunch relay rest on: that
there are ions.  The electrons of a slice make them, and the slices reach from -7 sigma
up in steps of 0.3, so with few slices a side only a large distribution has electrons
in the last ones (four: one of 200,000; none of 2,000 below six).  In every case here the
sums and slices are numbers, every bunch's cloud is charged and every bunch after the
first is kicked (somewhere by far more than the 1e-12 the two forms agree to), for
slice counts with both remainders of a group of four that an odd count has, after one
chunk of eight, two, three and six.  Three slices to seven have no ions (one slice a
side: no field either, 0 / 0 in its spacing); parity of the train there is unpinned.
"""
import numpy as np
import pytest

import mtrack_amd as m
from mtrack_amd import confgen as cg

pytestmark = pytest.mark.gpu
RTOL = 1e-12


def train(d, nslc, bunches, fbii=1, **form):
    cg.filling_file(d + "/fill.txt", list(range(bunches)), out=())
    text = cg.ring_conf(sections={
        "tracking": {"BunchModel": "STRONG", "EnableFBII": fbii, "NrevTot": 100, "NrevMon": 1, "EnableRW_long": 0,
                     "EnableQuantum": 0, "filling": d + "/fill.txt"},
        "ring": {"Lc": cg.small_ring(40), "Iring": 20.0},
        "distribution": {"Np": 200000, "Nslc": nslc}})
    w = m.WeakStrong(m.Config(cg.write(d + "/ws%d.conf" % fbii, text), d + "/"), **form)
    ion = np.asarray(w.track(2)[2])
    sl = np.stack([w.slices(k) for k in range(bunches)])
    w.close()
    return ion, sl


@pytest.mark.parametrize("nslc,bunches", [(4, 30), (5, 9), (6, 9), (7, 5), (8, 30), (10, 2), (11, 30), (24, 30)])
def test_sums_and_kicks_are_there(tmp_path, nslc, bunches):
    print("case", nslc, bunches, flush=True)
    d = str(tmp_path)
    ion, sl = train(d, nslc, bunches)
    rion, rsl = train(d, nslc, bunches, serial_train=True)
    _, bare = train(d, nslc, bunches, fbii=0)
    assert np.isfinite(ion).all() and np.isfinite(sl).all()
    assert np.all(ion[..., 2] > 0)  # every bunch's cloud
    assert np.all(np.abs(ion - rion).max((0, 1)) <= RTOL * np.abs(rion).max((0, 1)))
    top = np.abs(rsl).max((0, 2))
    assert np.all(np.abs(sl - rsl).max((0, 2)) <= RTOL * np.maximum(top, 1e-300))
    kicked = np.abs(sl - bare)[:, 5].max(1)  # z' of every bunch
    assert kicked[0] == 0 and np.all(kicked[1:] > 0) and kicked.max() > 1000 * RTOL * top[5], kicked / top[5]


def test_without_ions(tmp_path):
    """Nothing in the train without ions: no charge in its sums, no kicks."""
    d = str(tmp_path)
    for nslc in (2, 3):
        bare = train(d, nslc, 9, fbii=0)[1]
        for serial in (False, True):
            ion, sl = train(d, nslc, 9, serial_train=serial)
            assert not ion[..., 2].any() and np.array_equal(sl, bare)
