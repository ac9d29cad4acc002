"""The tables mbt_ring_potentials returns for the bunches of an ensemble whose rings
have longitudinal long-range resonators, transverse ones alone, or none: the ring's own
bit for bit (the dipole rows for the rings that make dipole sums when alone), the
long-range row zero where no longitudinal resonator is and not elsewhere, whichever ring
was read before."""
import numpy as np
import pytest

import mtrack_amd as m
from variants import write_variant

pytestmark = pytest.mark.gpu
MEMBERS = ["lr_fb", "wakes", "lr_hv", "scan"]


def test_ensemble_potentials(tmp_path):
    cfgs = []
    for name in MEMBERS:
        d = str(tmp_path / name)
        cfgs.append(m.Config(write_variant(name, d, selffield={"Ncell": 40}, tracking={"NrevMon": 10}), d + "/"))
    ens = m.Ensemble(cfgs)
    ens.prepare()
    ens.track(7)
    for k, cfg in enumerate(cfgs):
        g = m.Ring(cfg)
        g.set_chunk(ens.chunk())
        g.prepare()
        g.track(7)
        for ib in (0, cfg.geti("Nbunch") - 1):
            a, b = ens.potentials(ens.first[k] + ib), g.potentials(ib)
            rows = range(7) if MEMBERS[k] in ("wakes", "lr_hv") else (0, 1, 2, 3, 5)
            assert all(np.array_equal(a[0][q], b[0][q]) for q in rows), (MEMBERS[k], ib)
            assert np.array_equal(a[1], b[1]), (MEMBERS[k], ib)
            assert np.any(a[0][1] != 0.0) == (MEMBERS[k] == "lr_fb"), (MEMBERS[k], ib)
        g.close()
    ens.close()
