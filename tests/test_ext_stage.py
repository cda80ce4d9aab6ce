"""The 2-D stage by element tile: one tile, several tiles, the widest node
lists, radiating boundaries whose interior neighbour is in another tile, and
EXTERNAL_STEP called after internal steps, against the oracle bit for bit."""
import numpy as np
import pytest

from helpers import ELEM2, NODE2, compare, wheel_mesh

pytestmark = pytest.mark.gpu

STATE = ["el", "d", "ua", "va", "el1", "d1"]


def _model(name):
    import myfvcomcode_amd as F
    if name == "wheel":            # a node of 12 triangles: sub-edge lists of 24
        return wheel_mesh()
    nx, ny = {"one_tile": (5, 4), "two_tiles": (9, 9), "tiles": (61, 31)}[name]
    m = F.Model.build(1, nx=nx, ny=ny, kb=6, n_seamounts=1)
    nob = m.hdr.iobcn              # every boundary condition, along tiles' borders too
    m.set_obc_type([(k % 10) + 1 for k in range(nob)])
    return m


@pytest.mark.parametrize("name", ["one_tile", "two_tiles", "tiles", "wheel"])
def test_stage_parity(built, name):
    import myfvcomcode_amd as F
    from oracle import Oracle
    m = _model(name)
    dev, orc = F.DeviceModel(m), Oracle(m)
    print("case: %s (%d elements), external / internal / external steps" % (name, m.n), flush=True)
    dev.external_step(1)
    orc.external_step(1)
    worst, bad = compare(dev, orc, m, STATE, 0.0)
    assert not bad, bad
    dev.run(3)
    orc.run(3)
    worst, bad = compare(dev, orc, m, NODE2 + ELEM2 + ["u", "t1"], 0.0)
    assert not bad, bad
    # the external step's constants are those that the internal step left
    for iext in (1, 2, 3):
        dev.external_step(iext)
        orc.external_step(iext)
    worst, bad = compare(dev, orc, m, STATE, 0.0)
    assert not bad, bad
