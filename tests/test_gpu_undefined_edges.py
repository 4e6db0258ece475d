"""Edges with NaN or infinite coordinates among ordinary ones: the call's sample
total counts the ordinary edges' samples (it also sizes the launches' buffers),
and their decisions stay the oracle's, through device and host arrays."""
import numpy as np
import pytest

from oracle.oracle import OracleScene

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("value", [np.nan, np.inf, -np.inf, 3.0e38])
def test_totals_beside_undefined_edges(workload_dir, value):
    import torch

    import gpuprm_amd
    d = workload_dir(2)
    sp = gpuprm_amd.RobotConfigspace(d, 0.01, 1 << 16)
    sp.init(0, 1)
    rng = np.random.default_rng(12)
    n = 3000  # several blocks of the prologue
    QS = rng.uniform(-np.pi, np.pi, size=(6, n)).astype(np.float32)
    QE = (QS + rng.normal(0, 0.1, size=QS.shape)).astype(np.float32)
    bad = np.array([0, 1, 63, 64, 1023, 1024, 2047, 2999])
    QE[3, bad] = value
    ok = np.setdiff1d(np.arange(n), bad)
    want, total = OracleScene(d).indicator2(QS[:, ok].copy(), QE[:, ok].copy(), nthreads=8)
    res = torch.full((n,), 7, dtype=torch.int32, device="cuda")
    print("undefined edges: %r" % value, flush=True)
    st = sp.indicator2_dev(torch.from_numpy(QS).cuda(), torch.from_numpy(QE).cuda(), res)
    # an edge of undefined length is one sample, one of infinite length none
    assert st.samples_total == total + (len(bad) if np.isnan(value) else 0)
    assert np.array_equal(res.cpu().numpy()[ok] != 0, want != 0)
    before = sp.get_numthreads_all()
    r = np.full(n, 7, np.int32)
    sp.indicator2(QS.ravel(), QE.ravel(), r, n, n)
    assert sp.get_numthreads_all() - before == total
    assert np.array_equal(r[ok] != 0, want != 0)


def test_totals_of_any_number_of_edges(workload_dir):
    """One block of the prologue and several, large calls before small ones, the
    library's stream and a caller's: the oracle's totals and decisions."""
    import torch

    import gpuprm_amd
    d = workload_dir(1)
    sp = gpuprm_amd.RobotConfigspace(d, 0.01, 1 << 16)
    sp.init(0, 1)
    o = OracleScene(d)
    rng = np.random.default_rng(3)
    stream = torch.cuda.Stream()
    for n in (5000, 1, 1025, 1024, 1023, 2, 2049, 64):
        QS = rng.uniform(-np.pi, np.pi, size=(4, n)).astype(np.float32)
        QE = (QS + rng.normal(0, 0.03, size=QS.shape)).astype(np.float32)
        want, total = o.indicator2(QS, QE, nthreads=8)
        longest = int((np.sqrt(((QE - QS) ** 2).sum(axis=0)) / 0.01).max()) + 1
        qs, qe = torch.from_numpy(QS).cuda(), torch.from_numpy(QE).cuda()
        for st in (None, stream):
            res = torch.full((n,), 7, dtype=torch.int32, device="cuda")
            torch.cuda.synchronize()
            s = sp.indicator2_dev(qs, qe, res, None if st is None else st.cuda_stream)
            assert s.samples_total == total and abs(s.max_testnum - longest) <= 1, n
            assert np.array_equal(res.cpu().numpy() != 0, want != 0), n
