"""The internal step where the tiles of the fused tracer and q2 kernels carry
the most: tiles whose nodes and rings exceed two waves, the widest rings,
sigma columns that differ from node to node, and the deepest columns,
against the oracle bit for bit."""
import numpy as np
import pytest

from helpers import ELEM2, ELEM3, NODE2, NODE3, compare, wheel_mesh

pytestmark = pytest.mark.gpu


def _stretched(nx=33, ny=97, kb=6):
    """Nodes eight times as far apart in x as in y: a tile of 128 triangles is
    about 3 by 22 cells, up to 133 nodes with their rings."""
    import myfvcomcode_amd as F
    c = F.Model.case_defaults(0)
    d = c.dx
    x = np.tile(np.arange(nx) * 8.0 * d, ny)
    y = np.repeat(np.arange(ny) * d, nx)
    i = (np.arange(ny - 1)[:, None] * nx + np.arange(nx - 1)[None, :] + 1).ravel()
    rows = np.concatenate([np.stack([i, i + nx, i + 1], 1), np.stack([i + 1, i + nx, i + nx + 1], 1)])
    m = F.Model.from_mesh(x, y, rows, 15.0 + 5.0 * np.cos(x / x.max() * 3.0), kb, [], c.p)
    vx, vy = m.field("vx"), m.field("vy")
    m.field("el")[1:] = 0.05 * np.cos(np.pi * vx[1:] / vx.max()) * np.cos(np.pi * vy[1:] / vy.max())
    m.field3("t1")[:-1, 1:] = 15.0 + np.linspace(3.0, 0.0, kb - 1)[:, None] + 0.2 * np.sin(vy[1:] / (5.0 * d))
    m.field3("s1")[:-1, 1:] = 30.0 + 0.3 * np.sin(vx[1:] / (30.0 * d))
    m.cold_start()
    return m


def _sigma_by_node(kb=8):
    """The estuary channel with a power law whose exponent varies by node."""
    import myfvcomcode_amd as F
    m = F.Model.build(0, nx=41, ny=21, kb=kb)
    p = 1.0 + 0.3 * np.sin(np.arange(m.field3("z").shape[1]) * 0.37)
    z = -((np.arange(kb) / (kb - 1.0))[:, None] ** p[None, :])

    def fill(names, z):
        zz, dz, dzz = np.zeros_like(z), np.zeros_like(z), np.zeros_like(z)
        zz[:-1] = 0.5 * (z[:-1] + z[1:])
        zz[-1] = 2.0 * zz[-2] - zz[-3]
        dz[:-1] = z[:-1] - z[1:]
        dzz[:-1] = zz[:-1] - zz[1:]
        for n, v in zip(names, (z, zz, dz, dzz)):
            m.field3(n)[:, 1:] = v[:, 1:]

    fill(("z", "zz", "dz", "dzz"), z)
    nv = m.field("nv").reshape(3, -1)[:, 1:]
    z1 = np.zeros((kb, nv.shape[1] + 1))
    z1[:, 1:] = (z[:, nv[0]] + z[:, nv[1]] + z[:, nv[2]]) / 3.0
    fill(("z1", "zz1", "dz1", "dzz1"), z1)
    m.cold_start()
    return m


def _deep():
    """The most layers the device takes, under an open boundary."""
    import myfvcomcode_amd as F
    return F.Model.build(1, nx=13, ny=9, kb=64, n_seamounts=1)


CASES = {"stretched": _stretched, "wheel": wheel_mesh, "sigma": _sigma_by_node, "deep": _deep,
         # up to 45 levels VDIF_Q takes blocks of columns here, past them a lane a column
         "wheel_45": lambda: wheel_mesh(kb=45), "sigma_46": lambda: _sigma_by_node(kb=46),
         "wheel_47": lambda: wheel_mesh(kb=47)}


@pytest.mark.parametrize("name", list(CASES))
def test_internal_parity(built, name):
    import myfvcomcode_amd as F
    from oracle import Oracle
    m = CASES[name]()
    print("case: %s (%d elements), 4 internal steps" % (name, m.n), flush=True)
    dev, orc = F.DeviceModel(m), Oracle(m)
    dev.run(4)
    orc.run(4)
    worst, bad = compare(dev, orc, m, NODE2 + ELEM2 + ELEM3 + NODE3, 0.0)
    assert not bad, bad
    assert np.isfinite(dev.get("t1")).all() and np.ptp(dev.get("t1")) > 0
