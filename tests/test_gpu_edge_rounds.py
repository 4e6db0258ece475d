"""Large calls of a fresh context that take several rounds: the first window
enqueued before the largest testnum is known (more than 2^28 / 16 pair tests
in it), and pair masks in rounds whose preparation runs beside the round
before.  A larger call of the same context replaces the buffers between its
rounds.  A part of the edges is re-decided by the oracle."""
import numpy as np
import pytest

from oracle.oracle import OracleScene

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("wl,n,lo,hi", [(3, 80000, 0.05, 0.25), (2, 24000, 1.0, 2.4)])
def test_rounds_of_large_calls(workload_dir, wl, n, lo, hi):
    import torch

    import gpuprm_amd
    d = workload_dir(wl)
    sp = gpuprm_amd.RobotConfigspace(d, 0.01, 1 << 16)
    sp.init(0, 1)
    o = OracleScene(d)
    M = int(np.fromfile(d + "/pairs/M.bin", np.int32)[0])
    nd = sp.dim()
    rng = np.random.default_rng(31 * wl)
    for times in (1, 2):  # the second call twice the edges, and longer ones
        k = n * times
        assert (16 * k * M > 1 << 28) == (wl == 3)  # the first window goes ahead
        QS = rng.uniform(-np.pi, np.pi, size=(nd, k)).astype(np.float32)
        u = rng.normal(size=(nd, k))
        QE = (QS + u / np.linalg.norm(u, axis=0) * rng.uniform(lo, hi * times, k)).astype(np.float32)
        res = torch.full((k,), 7, dtype=torch.int32, device="cuda")
        print("edge rounds: workload %d, %d edges" % (wl, k), flush=True)
        st = sp.indicator2_dev(torch.from_numpy(QS).cuda(), torch.from_numpy(QE).cuda(), res)
        assert st.samples_total * M > 1 << 28 and st.rounds >= 2
        sub = slice(0, k, 40)
        want, _ = o.indicator2(QS[:, sub].copy(), QE[:, sub].copy(), nthreads=8)
        assert np.array_equal(res.cpu().numpy()[sub] != 0, want != 0)
        assert 0.02 < (want != 0).mean() < 0.95
