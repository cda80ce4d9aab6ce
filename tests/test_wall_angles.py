"""The wall projection's SIN and COS of the wall angle: two calls of the C
library in the oracle as in the HIP path.  A call of sincos differs in the
last bit at some angles; the 41x23-node mesh here has a wall element at one."""
import math

import numpy as np
import pytest

import myfvcomcode_amd as F
from helpers import ELEM2, ELEM3, NODE2, NODE3, compare


def _model():
    return F.Model.build(1, nx=41, ny=23, kb=6, n_seamounts=1)


def test_oracle_projects_by_sin_and_cos(built):
    from oracle import Oracle
    m = _model()
    orc = Oracle(m)
    rng = np.random.default_rng(2)
    u, v = rng.standard_normal(m.n + 1), rng.standard_normal(m.n + 1)
    orc.put("uaf", u)
    orc.put("vaf", v)
    orc.routine("bcond_gcn2")
    walls = np.flatnonzero(m.field("isbce") == 1)
    assert len(walls) == 104
    for e in walls:
        s, c = math.sin(m.field("alpha")[e]), math.cos(m.field("alpha")[e])
        assert orc.get("uaf")[e] == u[e] * (s * s) - v[e] * s * c, e
        assert orc.get("vaf")[e] == -u[e] * s * c + v[e] * (c * c), e


@pytest.mark.gpu
def test_parity_at_such_an_angle(built):
    from oracle import Oracle
    m = _model()
    print("case: 41x23 nodes, 2 external and 4 internal steps", flush=True)
    dev, orc = F.DeviceModel(m), Oracle(m)
    for iext in (1, 2):
        dev.external_step(iext)
        orc.external_step(iext)
    worst, bad = compare(dev, orc, m, ["el", "d", "ua", "va", "el1", "d1"], 0.0)
    assert not bad, bad
    dev.run(4)
    orc.run(4)
    worst, bad = compare(dev, orc, m, NODE2 + ELEM2 + ELEM3 + NODE3, 0.0)
    assert not bad, bad
