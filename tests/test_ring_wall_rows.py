"""A ring whose resistive wall would have no row of dipole history (Nmlt below -1, which
the configuration reader accepts) is refused before any device call: the turn writes its
dipoles to the history's rows."""
import pytest

import mtrack_amd as m
from variants import write_variant


@pytest.mark.parametrize("nmlt", [-2, -3, -100])
def test_refused(tmp_path, nmlt):
    d = str(tmp_path)
    cfg = m.Config(write_variant("wakes", d, tracking={"Nmlt": nmlt}), d + "/")
    assert cfg.geti("Nmlt") == nmlt
    with pytest.raises(m.MbtError, match="Nmlt"):
        m.Ring(cfg)
    with pytest.raises(m.MbtError, match="Nmlt"):
        m.Ensemble([cfg])
