"""The full tests' iteration history, whose first entries are in LDS: how many
depends on the launch (16 for a few blocks, the fewer the more blocks share a
CU, none where the image leaves no room) and the rest is in memory.  Launches
of two groups to a full grid, every launch shape, two scenes; codes must be the
oracle's, also those of pairs that run through all iterations."""
import numpy as np
import pytest

import gpuprm_amd
from oracle.oracle import OracleScene

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("block,waves", [(256, 5), (256, 4), (1024, 4)])
@pytest.mark.parametrize("workload", [1, 3])
def test_history_in_lds_and_memory(workload_dir, workload, block, waves):
    import torch
    d = workload_dir(workload)
    sp = gpuprm_amd.RobotConfigspace(d, 0.01, 1 << 16)
    sp.init(0, 1)
    sp.set_launch_shape(block, waves, 64)
    o = OracleScene(d)
    nd = sp.dim()
    rng = np.random.default_rng(7)
    Q = rng.uniform(-np.pi, np.pi, size=(nd, 40000)).astype(np.float32)
    want = o.indicator_batch(Q[:, :6000].copy(), nthreads=8)
    assert (want != 0).any() and (want == 0).any()
    full = None
    for n in (40000, 6000, 1500, 300, 65):
        print("history: workload %d, %d x %d, n %d" % (workload, block, waves, n), flush=True)
        r = torch.zeros(n, dtype=torch.int32, device="cuda")
        sp.indicator_dev(torch.from_numpy(Q[:, :n].copy()).cuda(), r)
        got = r.cpu().numpy()
        full = got if full is None else full
        assert np.array_equal(got[:6000], want[:n])
        assert np.array_equal(got, full[:n])
    QE = np.clip(Q[:, :500] + rng.uniform(-0.4, 0.4, size=(nd, 500)), -np.pi, np.pi).astype(np.float32)
    re = torch.zeros(500, dtype=torch.int32, device="cuda")
    sp.indicator2_dev(torch.from_numpy(Q[:, :500].copy()).cuda(), torch.from_numpy(QE).cuda(), re)
    wante, _ = o.indicator2(Q[:, :500].copy(), QE, nthreads=8)
    assert np.array_equal(re.cpu().numpy() != 0, wante != 0)
