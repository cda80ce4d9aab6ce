"""New wind from one thread while another enqueues steps on the same handle."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_wind_set_while_steps_are_enqueued(built):
    import myfvcomcode_amd as F
    from myfvcomcode_amd.restart import STATE
    m = F.Model.build(1, nx=61, ny=31, kb=6, n_seamounts=1)
    n1 = m.n + 1
    rng = np.random.default_rng(7)
    winds = [np.concatenate([8.0 + rng.standard_normal(n1), 2.0 + rng.standard_normal(n1)]) for _ in range(3)]
    print("case: wind from one thread, eager steps from another", flush=True)
    dev = F.DeviceModel(m)
    dev.set_forcing("wind", winds[0])       # from here on every external step forms its own stress
    stop, steps = threading.Event(), [0]

    def enqueue():
        while not stop.is_set() and steps[0] < 400:
            dev.internal_step()
            steps[0] += 1

    t = threading.Thread(target=enqueue)
    t.start()
    for _ in range(5):
        dev.set_forcing("wind", winds[0])
        dev.set_forcing("wind", winds[1])   # the last one
    stop.set()
    t.join()
    dev.synchronize()
    # a handle that is given the same state and winds, one after another
    ref = F.DeviceModel(m)
    ref.set_forcing("wind", winds[0])
    ref.run(steps[0])
    ref.set_forcing("wind", winds[1])
    for name in STATE:
        ref.put(name, dev.get(name))
    for d in (dev, ref):
        d.set_forcing("wind", winds[2])
        d.run(1)
    for name in ("el", "ua", "va", "u", "v"):
        assert np.array_equal(dev.get(name), ref.get(name)), name
