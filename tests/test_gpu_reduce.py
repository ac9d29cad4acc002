"""The per-bunch reduction's convolutions and the one-pass resistive-wall sum at the
edges of their ranges, the sum as a matrix product, and the turn count a block of launches keeps itself.

Slice counts around the lanes a group of slices gets (16, 8, 4, 2 and 1 of a block
of 256 or 512 lanes) and around the eight and sixteen terms read at a time, one
bunch and more bunches than take the wide block; the wide and the narrow block give
the same bits (a ring alone and in an ensemble past the line).  Resistive wall: one
bunch, every bucket, more (row, bunch) pairs than lanes, the trigger's change at
turn 50 inside and at the ends of calls; as a matrix product buckets below, at and
past its tiles of 16, few and many slices of its sum, one ring.  Against the oracle within 1e-12, the
bound of the other parity tests: the same terms added in another order.
"""
import numpy as np
import pytest

import mtrack_amd as m
import oracle as o
from mtrack_amd import confgen as cg
from test_gpu_parity import RTOL, stat_errors

pytestmark = pytest.mark.gpu

RES = [("resonator_%d" % (i + 1), {"Rs": rs, "fres": f, "Qfactor": 1.0, "plane": p})
       for i, (p, rs, f) in enumerate((("LON", 5e3, 10.0), ("VER", 2e5, 8.0), ("HOR", 2e5, 8.0)))]
WALL = {"rhorw": 1.7e-8, "beffL1": 0.012, "beffL2": 0.012, "beffH3": 0.012, "beffV3": 0.012}


def conf(d, name, h, bunches, np_, ncell=0, nmlt=0, **tracking):
    fill = "%s/%s.fill" % (d, name)
    cg.filling_file(fill, [int(k * h / bunches) for k in range(bunches)], out=(0,))
    secs = {"tracking": dict({"NrevTot": 100, "NrevMon": 7, "EnableRW_long": int(nmlt > 0), "Nmlt": max(nmlt, 1),
                              "filling": fill}, **tracking),
            "ring": dict(WALL, Lc=cg.small_ring(h), Iring=0.5 * bunches), "distribution": {"Np": np_}}
    if ncell:
        secs["selffield"] = {"Ncell": ncell, "Nsigma": 5.0}
    return m.Config(cg.write("%s/%s.conf" % (d, name), cg.ring_conf(sections=secs, extra_sections=RES if ncell else ())),
                    d + "/")


def check(cfg, calls, **options):
    orc, g = o.OracleRing(cfg, o.RNG_PHILOX), m.Ring(cfg, **options)
    orc.prepare()
    g.prepare()
    for n in calls:
        ost, oam, _ = orc.track(n)
        gst, gam, _ = g.track(n)
        assert stat_errors(gst, ost).max() <= RTOL
        assert np.all(np.abs(gam - oam) <= RTOL * np.abs(oam).max())
    if cfg.geti("Ncell"):
        ho, to = orc.histograms()
        hg, tg = g.histograms()
        assert np.array_equal(ho, hg) and np.array_equal(to, tg)
    g.close()


@pytest.mark.parametrize("ncell", [2, 3, 15, 16, 17, 31, 33, 65, 127, 129, 257, 513])
@pytest.mark.parametrize("bunches", [1, 260])
def test_convolutions(tmp_path, ncell, bunches):
    print("case", ncell, bunches, flush=True)
    check(conf(str(tmp_path), "conv", 300, bunches, 67, ncell=ncell), [4])


@pytest.mark.parametrize("h,bunches,nmlt,calls", [(20, 1, 1, [30]), (416, 1, 3, [9]), (20, 20, 60, [70]),
                                                  (416, 416, 5, [10]), (33, 7, 2, [7, 42, 1, 1, 9])])
def test_wall_sum(tmp_path, h, bunches, nmlt, calls):
    print("case", h, bunches, nmlt, flush=True)
    check(conf(str(tmp_path), "wall", h, bunches, 31, nmlt=nmlt, triggerRW=1), calls)


@pytest.mark.parametrize("h,bunches,nmlt", [(3, 3, 1), (15, 4, 2), (16, 16, 11), (17, 5, 12), (130, 13, 25),
                                            (416, 416, 40)])
def test_wall_product(tmp_path, h, bunches, nmlt):
    print("case", h, bunches, nmlt, flush=True)
    check(conf(str(tmp_path), "product", h, bunches, 31, nmlt=nmlt, triggerRW=1), [2 * nmlt, 7], force_gemm=True)


def test_wide_and_narrow_blocks_agree(tmp_path):
    d = str(tmp_path)
    small, large = conf(d, "a", 20, 20, 900, ncell=100, nmlt=3), conf(d, "b", 300, 260, 300, ncell=100, nmlt=3)
    alone, both = m.Ring(small), m.Ensemble([small, large])
    for r in (alone, both):
        r.set_chunk(2)
        r.prepare()
    a, b = alone.track(12)[0], both.track(12)[0]
    assert np.array_equal(a, both.ring_rows(0, b))
    for k in (0, 19):
        assert np.array_equal(alone.get_bunch(k), both.get_bunch(k))
    alone.close()
    both.close()
