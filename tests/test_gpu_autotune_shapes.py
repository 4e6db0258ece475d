"""What gprm_autotune leaves behind: small point launches keep the four-wave
variant that a context takes for them by default, whichever shape was found;
only a shape that the caller sets holds for every launch.  Seen from the work
units of a small call, whose size follows the launch's waves."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _units(sp, q, r):
    sp.profile_enable(True)
    sp.indicator_dev(q, r)
    units = sp.profile_read().units_done
    sp.profile_enable(False)
    return units


def test_small_launches_after_autotune(workload_dir):
    import torch

    import gpuprm_amd
    d = workload_dir(3)
    sp = gpuprm_amd.RobotConfigspace(d, 0.01, 1 << 20)
    sp.init(0, 1)
    shape = sp.get_launch_shape()
    assert shape.waves == 5
    M = int(np.fromfile(d + "/pairs/M.bin", np.int32)[0])
    n = 24 * (shape.grid * shape.block // 64) // M * 64  # the largest small launch
    g = torch.Generator(device="cuda").manual_seed(1)
    q = (torch.rand(7, 1 << 20, device="cuda", generator=g) * 2 - 1) * np.pi
    small = q[:, :n].contiguous()
    r = torch.zeros(n, dtype=torch.int32, device="cuda")
    default = _units(sp, small, r)
    codes = r.clone()
    found, _ = sp.autotune(q, reps=2)
    print("autotune found", found.as_dict(), flush=True)
    assert _units(sp, small, r) == default
    assert torch.equal(r, codes)
    sp.set_launch_shape(256, 5, 128)
    assert _units(sp, small, r) > default  # more waves, so smaller units
    assert torch.equal(r, codes)
