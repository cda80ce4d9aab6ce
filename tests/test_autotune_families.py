"""Which kernel families the autotuner tries: those of the step that have a
choice of workgroup size; and the calls that set such choices."""
import pytest

import myfvcomcode_amd as F

pytestmark = pytest.mark.gpu


# up to 45 levels VDIF_Q takes blocks of columns on a small mesh, whose
# workgroups have one size; past them a lane a column
@pytest.mark.parametrize("kb,lanes", [(9, False), (45, False), (46, True)])
def test_autotuned_families(built, kb, lanes):
    m = F.Model.build(1, nx=21, ny=11, kb=kb, n_seamounts=1)
    dev = F.DeviceModel(m)
    print("case: autotune, KB=%d" % kb, flush=True)
    rep = dev.autotune(1)
    assert set(rep) == {"adv_ts", "adv_q", "viscofh", "vdif_ts", "adjust1_brough", "adjust2", "baropg",
                        "step_end"} | ({"vdif_q"} if lanes else set())
    assert all(size in (64, 128, 256) and us > 0.0 for size, us in rep.values())


def test_concurrency_and_block_arguments(built):
    m = F.Model.build(0, nx=21, ny=7, kb=6)
    dev = F.DeviceModel(m)
    print("case: set_concurrency, set_block", flush=True)
    for mode in (0, 1, 2, 3):
        dev.set_concurrency(mode)
    for mode in (-1, 4):
        with pytest.raises(RuntimeError):
            dev.set_concurrency(mode)
    for size in (64, 128, 256):
        dev.set_block("adv_ts", size)
    for size in (0, 32, 512):
        with pytest.raises(RuntimeError):
            dev.set_block("adv_ts", size)
