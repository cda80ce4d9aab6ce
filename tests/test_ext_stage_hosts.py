"""The 2-D stage on tables that a host has set otherwise than the grid builder
does, against the oracle bit for bit."""
import numpy as np
import pytest

from helpers import compare

pytestmark = pytest.mark.gpu

STATE = ["el", "d", "ua", "va", "el1", "d1"]


def _model(types):
    import myfvcomcode_amd as F
    m = F.Model.build(1, nx=61, ny=31, kb=6, n_seamounts=1)
    m.set_obc_type([types[k % len(types)] for k in range(m.hdr.iobcn)])
    return m


def _parity(m, what):
    import myfvcomcode_amd as F
    from oracle import Oracle
    print("case: %s (%d elements), 3 external steps" % (what, m.n), flush=True)
    dev, orc = F.DeviceModel(m), Oracle(m)
    for iext in (1, 2, 3):
        dev.external_step(iext)
        orc.external_step(iext)
    worst, bad = compare(dev, orc, m, STATE, 0.0)
    assert not bad, bad
    assert np.ptp(dev.get("ua")) > 0
    return dev


@pytest.mark.parametrize("radiating", [5, 6, 7, 8])
def test_next_obc_is_an_obc_node(built, radiating):
    """Nodes that radiate from a clamped neighbour on the boundary: its
    elevation is the clamped one."""
    m = _model([3, radiating, 4])
    m.field("next_obc")[1::3] = m.field("i_obc_n")[0::3][:len(m.field("next_obc")[1::3])]
    _parity(m, "TYPE_OBC %d beside 3" % radiating)
