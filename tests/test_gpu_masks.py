"""Edge checks with pair masks (the kinematics kernel leaves out the pairs
whose bounds hold for a whole group of items) and the level windows of an
edge's samples: decisions must be the oracle's for edges around every window
and row boundary, for degenerate edges, and for a call large enough that the
single-scene path writes masks (multi-scene calls always do)."""
import numpy as np
import pytest

from oracle.oracle import OracleScene

pytestmark = pytest.mark.gpu

# testnums at which runs, rows and windows change (kRunShort, rows of 16,
# edge_levels)
TESTNUMS = [1, 2, 3, 7, 8, 9, 15, 16, 17, 31, 32, 33, 63, 64, 65, 255, 256, 257, 511, 512, 513, 1000, 2047, 2048, 2049]


def _edges(rng, ndof, dq, testnums, each):
    """`each` random edges of every testnum T (length (T - 1/2) dq, so that
    rounding cannot move T), in mixed order."""
    T = np.repeat(testnums, each)
    rng.shuffle(T)
    A = rng.uniform(-3.0, 3.0, size=(ndof, len(T)))
    d = rng.normal(size=A.shape)
    B = A + d / np.linalg.norm(d, axis=0) * (T - 0.5) * dq
    return A.astype(np.float32), B.astype(np.float32), T


@pytest.mark.parametrize("wl", [1, 2, 3, 5])
def test_batch_edges_every_window(workload_dir, wl):
    import torch

    import gpuprm_amd
    d = workload_dir(wl)
    dq = 0.002
    sp = gpuprm_amd.RobotConfigspace(d, dq, 1 << 16)
    sp.init(0, 1)
    o = OracleScene(d, dq)
    rng = np.random.default_rng(90 + wl)
    nd = sp.dim()
    QS, QE, T = _edges(rng, nd, dq, TESTNUMS, 12)
    # edges of no length
    QE[:, :3] = QS[:, :3]
    want, tot = o.indicator2(QS, QE, nthreads=8)
    b = gpuprm_amd.SceneBatch([sp])
    qs, qe = torch.from_numpy(QS).cuda(), torch.from_numpy(QE).cuda()
    res = torch.full((QS.shape[1],), 7, dtype=torch.int32, device="cuda")
    print("masks: workload %d, %d edges" % (wl, QS.shape[1]), flush=True)
    _, samples = b.indicator2_dev([qs], [qe], [res])
    assert samples == tot
    got = res.cpu().numpy()
    bad = np.flatnonzero((got != 0) != (want != 0))
    assert bad.size == 0, (T[bad[:10]], got[bad[:10]], want[bad[:10]])
    res.fill_(7)
    st = sp.indicator2_dev(qs, qe, res)
    assert st.samples_total == tot and 0 < st.samples_scheduled <= tot
    assert np.array_equal(res.cpu().numpy() != 0, want != 0)
    assert 0 < (want != 0).sum() < len(want)


@pytest.mark.parametrize("wl,n,length", [(3, 16384, 0.6), (2, 16384, 1.2)])
def test_large_call_with_masks(workload_dir, wl, n, length):
    """At least 2^27 pair tests: masks in the single-scene path.  Every 8th
    edge re-decided by the oracle."""
    import torch

    import gpuprm_amd
    d = workload_dir(wl)
    sp = gpuprm_amd.RobotConfigspace(d, 0.01, 1 << 16)
    sp.init(0, 1)
    o = OracleScene(d)
    nd = sp.dim()
    rng = np.random.default_rng(17 * wl)
    QS = rng.uniform(-np.pi, np.pi, size=(nd, n)).astype(np.float32)
    dirn = rng.normal(size=(nd, n))
    QE = (QS + dirn / np.linalg.norm(dirn, axis=0) * length * rng.uniform(0.6, 1.0, n)).astype(np.float32)
    res = torch.full((n,), 7, dtype=torch.int32, device="cuda")
    print("masks: workload %d, %d edges" % (wl, n), flush=True)
    sp.indicator2_dev(torch.from_numpy(QS).cuda(), torch.from_numpy(QE).cuda(), res)
    sub = slice(0, n, 8)
    want, _ = o.indicator2(QS[:, sub].copy(), QE[:, sub].copy(), nthreads=8)
    assert np.array_equal(res.cpu().numpy()[sub] != 0, want != 0)
    assert 0.1 < (want != 0).mean() < 0.95


def test_undefined_edges_keep_their_group(workload_dir):
    """An edge with a NaN coordinate, among ordinary ones of the same rows:
    the others' decisions stay the oracle's, with masks and without."""
    import torch

    import gpuprm_amd
    d = workload_dir(2)
    sp = gpuprm_amd.RobotConfigspace(d, 0.01, 1 << 16)
    sp.init(0, 1)
    o = OracleScene(d)
    rng = np.random.default_rng(5)
    QS, QE, _ = _edges(rng, 6, 0.01, [1, 5, 8, 16, 60], 40)
    bad = np.arange(0, QS.shape[1], 7)
    QE[2, bad] = np.nan
    ok = np.setdiff1d(np.arange(QS.shape[1]), bad)
    want, _ = o.indicator2(QS[:, ok].copy(), QE[:, ok].copy(), nthreads=8)
    qs, qe = torch.from_numpy(QS).cuda(), torch.from_numpy(QE).cuda()
    for batch in (True, False):
        res = torch.full((QS.shape[1],), 7, dtype=torch.int32, device="cuda")
        if batch:
            gpuprm_amd.SceneBatch([sp]).indicator2_dev([qs], [qe], [res])
        else:
            sp.indicator2_dev(qs, qe, res)
        assert np.array_equal(res.cpu().numpy()[ok] != 0, want != 0), batch
