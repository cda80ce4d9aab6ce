"""get_state / put_state of arrays below, around and far above the size from
which the copies are cut into chunks for several threads: what is put is got,
to the bit, and nothing beside it changes."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny,kb", [
    (21, 11, 4),       # a few KiB
    (181, 120, 12),    # T1 just below 2 MiB, U above
    (181, 121, 12),    # T1 just above 2 MiB
    (301, 201, 25),    # T1 12 MB, U 24 MB: several chunks a thread and a remainder
])
def test_put_get_round_trip(built, nx, ny, kb):
    import myfvcomcode_amd as F
    m = F.Model.build(1, nx=nx, ny=ny, kb=kb, n_seamounts=1)
    dev = F.DeviceModel(m)
    rng = np.random.default_rng(nx * 1000 + ny)
    names = ["el", "ua", "t1", "u", "v", "q2"]
    want = {}
    for n in names:
        size = len(dev.get(n))
        buf = rng.standard_normal(size + 1)
        want[n] = buf[1:]                       # off the allocation's alignment
        print("case: %s, %d bytes" % (n, 8 * size), flush=True)
        dev.put(n, want[n])
    s1 = dev.get("s1")
    for n in names:
        assert np.array_equal(dev.get(n), want[n]), n
    assert np.array_equal(dev.get("s1"), s1)
