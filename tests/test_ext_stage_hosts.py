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


def test_boundary_marks_of_any_value(built):
    """ISBC enters the edge terms as a number; an ISBCE other than 1, 2 and 3
    marks nothing."""
    m = _model([1])
    rng = np.random.default_rng(4)
    c = rng.permutation(np.arange(1, m.hdr.ne + 1))
    for k, v in enumerate((3, -1, 7, 4, 2)):
        m.field("isbc")[c[40 * k:40 * (k + 1)]] = v
    e = rng.permutation(np.flatnonzero(m.field("isbce")[1:] == 0) + 1)
    for k, v in enumerate((4, 5, 6, 7, -2, -1)):
        m.field("isbce")[e[20 * k:20 * (k + 1)]] = v
    dev = _parity(m, "ISBC and ISBCE of any value")
    assert np.isfinite(dev.get("ua")).all()


@pytest.mark.parametrize("types", [[1], [5, 2, 8, 3, 9]])
def test_flux_to_a_cell_without_the_node(built, types):
    """OBC nodes whose flux defects go to boundary cells elsewhere (each
    node's cells exchanged with those of the node across the boundary)."""
    m = _model(types)
    adjc = m.field("adjc_obc").reshape(2, -1)
    adjc[:, 1:-1] = adjc[:, 1:-1][:, ::-1].copy()
    assert (m.field("isbce")[adjc[adjc > 0]] == 2).any()
    _parity(m, "TYPE_OBC %s, cells exchanged" % types)
