"""The forms of the step's kernels that depend on the mesh's size: layers
split over workgroups or whole columns, VDIF_Q by block of columns or a lane a
column, for all columns or for those that the learned closure rejects."""
import numpy as np
import pytest

import myfvcomcode_amd as F
from helpers import ELEM2, ELEM3, NODE2, NODE3, compare

pytestmark = pytest.mark.gpu

FAMILIES = ["adv_ts", "adv_q", "viscofh", "vdif_q", "vdif_ts", "adjust1_brough", "adjust2", "baropg", "step_end",
            "closure_features", "closure_apply"]
TURB = ["km", "kh", "kq", "q2", "q2l", "l"]


def _params(dev):
    """Weights that reject a column if its depth is above the median: one
    hidden unit a layer, KM = KH from 2.5e-3 up to far above the limit of 1."""
    x = dev.closure_samples()[0][:, 4]
    c, s = float(np.median(x)), 40.0
    w1, b1 = np.zeros((64, 5), np.float32), np.zeros(64, np.float32)
    w2, b2 = np.zeros((64, 64), np.float32), np.zeros(64, np.float32)
    w3, b3 = np.zeros((2, 64), np.float32), np.full(2, -6.0, np.float32)
    w1[0, 4], b1[0] = s, -s * c
    w2[0, 0] = 8.0
    w3[:, 0] = 32.0
    return np.concatenate([a.ravel() for a in (w1, b1, w2, b2, w3, b3)])


def _check_subset(m, params, devs):
    """One step with `params` on every handle of devs (in the same state): the
    columns that it rejects get what they get where all are rejected, the
    others keep their turbulence; the handles agree to the bit."""
    ref = F.DeviceModel(m)
    for n in ("u", "v", "el", "ua", "va"):
        assert np.array_equal(devs[0].get(n), devs[1].get(n)), n
    before = {n: devs[0].get(n).reshape(m.kb, -1) for n in TURB}
    ref.run(2)
    for n in TURB + ["u", "t1", "el"]:
        assert np.array_equal(ref.get(n), devs[0].get(n)), n
    reject = params.copy()
    reject[-2:] = 30.0
    ref.set_closure(1, reject)
    ref.run(1)
    assert ref.closure_fallbacks() == (m.m, m.m)
    for d in devs:
        d.set_closure(1, params)
        d.run(1)
    nf, nc = devs[0].closure_fallbacks()
    assert nc == m.m and 0.1 * nc < nf < 0.9 * nc
    kept = np.ones(m.m + 1, bool)
    got = {n: devs[0].get(n).reshape(m.kb, -1) for n in TURB}
    for n in ("kq", "q2", "q2l", "l"):
        kept &= (got[n] == before[n]).all(axis=0)
    kept[0] = True
    assert (~kept).sum() == nf
    for n in TURB:
        assert np.array_equal(got[n][:, ~kept], ref.get(n).reshape(m.kb, -1)[:, ~kept]), n
        for d in devs[1:]:
            assert np.array_equal(d.get(n), devs[0].get(n)), n
    assert (got["km"][:, kept][:, 1:] <= 1.0).all()


# by block of columns, and a lane a column (above 45 levels)
@pytest.mark.parametrize("kb", [12, 45, 46])
def test_rejected_columns_only(built, kb):
    m = F.Model.build(1, nx=61, ny=31, kb=kb, n_seamounts=3)
    print("case: 61x31 nodes, KB=%d, half of the columns rejected" % kb, flush=True)
    devs = [F.DeviceModel(m) for _ in range(2)]
    for f in FAMILIES:
        devs[1].set_block(f, 64)
    for d in devs:
        d.run(2)
    _check_subset(m, _params(devs[0]), devs)


def test_whole_columns_on_a_large_mesh(built):
    """105,625 nodes, 209,952 elements: no kernel splits its layers with
    workgroups of 64, only VISCOF_H and the closure's features do with 256;
    VDIF_Q takes a lane a column."""
    from oracle import Oracle
    m = F.Model.build(1, nx=325, ny=325, kb=41, n_seamounts=20)
    devs = [F.DeviceModel(m) for _ in range(2)]
    for f in FAMILIES:
        devs[1].set_block(f, 64)
    print("case: 325x325 nodes, KB=41, 2 steps", flush=True)
    orc = Oracle(m)
    orc.run(2)
    print("case: oracle done", flush=True)
    for d in devs:
        d.run(2)
        worst, bad = compare(d, orc, m, NODE2 + ELEM2 + ELEM3 + NODE3, 0.0)
        assert not bad, bad
    _check_subset(m, _params(devs[0]), devs)


# 128 elements fill one tile of the 2-D stage; 144 need two, with nodes that
# both have and one of them stores
@pytest.mark.parametrize("nx,tiles", [(9, 1), (10, 2)])
def test_first_tile_border(built, nx, tiles):
    from oracle import Oracle
    m = F.Model.build(1, nx=nx, ny=9, kb=6, n_seamounts=1)
    assert (m.n > 128) == (tiles == 2)
    m.set_obc_type([(k % 10) + 1 for k in range(m.hdr.iobcn)])
    print("case: %d elements in %d tiles" % (m.n, tiles), flush=True)
    dev, orc = F.DeviceModel(m), Oracle(m)
    for iext in (1, 2):
        dev.external_step(iext)
        orc.external_step(iext)
    dev.run(3)
    orc.run(3)
    worst, bad = compare(dev, orc, m, NODE2 + ELEM2 + ELEM3 + NODE3, 0.0)
    assert not bad, bad
