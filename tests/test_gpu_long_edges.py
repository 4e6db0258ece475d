"""Edges of more samples than a launch holds: the launches cut an edge's ranks
(single-scene calls at 2^24 items, multi-scene steps at 2^19).  An edge whose
last few samples alone collide is blocked, the edge that ends just before them
is free with every sample tested, and short edges beside them keep the
oracle's decisions.  Which samples collide is asked of the point checks."""
import numpy as np
import pytest

from oracle.oracle import OracleScene

pytestmark = pytest.mark.gpu


def _codes(sp, a, b, first, last, T):
    """Point codes of samples [first, last) of T of the edge a, b, with the edge
    checks' float operations."""
    import torch
    c1 = np.arange(first, last, dtype=np.int32).astype(np.float32) / np.float32(T - 1)
    c2 = np.float32(1) - c1
    q = torch.from_numpy((c1[None, :] * a[:, None] + c2[None, :] * b[:, None]).astype(np.float32)).cuda()
    r = torch.zeros(last - first, dtype=torch.int32, device="cuda")
    sp.indicator_dev(q, r)
    return r.cpu().numpy()


def _edges(sp, T):
    """(start, end that collides in its last samples only, end just short of
    that, edge length): along one line, T samples to the first end."""
    rng = np.random.default_rng(4)
    nd = sp.dim()
    while True:
        a = rng.uniform(-2.5, 2.5, nd).astype(np.float32)
        d = rng.normal(size=nd)
        d = (d / np.linalg.norm(d)).astype(np.float32)
        at = lambda t: (a + np.float32(t) * d).astype(np.float32)
        code = _codes(sp, at(2.0), a, 0, 2001, 2001)
        k = int(np.argmax(code != 0))
        if code[0] != 0 or k < 500:
            continue
        lo, hi = 2.0 * (k - 1) / 2000, 2.0 * k / 2000  # free, blocked
        for _ in range(14):
            mid = 0.5 * (lo + hi)
            if _codes(sp, at(mid), a, 0, 2, 2)[1] == 0:
                lo = mid
            else:
                hi = mid
        return a, at(hi), at(lo - 1e-3), hi


@pytest.mark.parametrize("T,batch", [((1 << 24) + (1 << 23), False), (1 << 21, True)])
def test_edge_longer_than_a_launch(workload_dir, T, batch):
    import torch

    import gpuprm_amd
    d = workload_dir(1)
    a, hit, free, length = _edges(gpu_space(d, 0.01), T)
    dq = float(np.float32(length / T))
    sp = gpu_space(d, dq)
    rng = np.random.default_rng(6)
    short = rng.uniform(-3.0, 3.0, size=(4, 40)).astype(np.float32)
    u = rng.normal(size=short.shape)
    ends = (short + u / np.linalg.norm(u, axis=0) * rng.uniform(0.5, 60.0, 40) * dq).astype(np.float32)
    want, _ = OracleScene(d, dq).indicator2(short, ends, nthreads=8)
    QS = np.concatenate([hit[:, None], a[:, None], short], axis=1)
    QE = np.concatenate([a[:, None], free[:, None], ends], axis=1)
    qs, qe = torch.from_numpy(QS).cuda(), torch.from_numpy(QE).cuda()
    res = torch.full((QS.shape[1],), 7, dtype=torch.int32, device="cuda")
    print("long edges: %d samples, batch %d" % (T, batch), flush=True)
    if batch:
        _, total = gpuprm_amd.SceneBatch([sp]).indicator2_dev([qs], [qe], [res])
    else:
        # the free edge alone: every sample scheduled, in more launches than levels
        st = sp.indicator2_dev(qs[:, 1:2].contiguous(), qe[:, 1:2].contiguous(), res[1:2])
        Tf, levels = st.max_testnum, 3
        while Tf > 512 * 4 ** (levels - 3):
            levels += 1
        assert st.samples_scheduled == st.samples_total == Tf and st.rounds > levels
        assert res[1].item() == 0
        st = sp.indicator2_dev(qs, qe, res)
        total = st.samples_total
        assert abs(st.max_testnum - T) < 0.01 * T
        hits = sum(int((_codes(sp, QS[:, 0], QE[:, 0], i, min(i + (1 << 22), st.max_testnum), st.max_testnum) != 0).sum())
                   for i in range(0, st.max_testnum, 1 << 22))
        assert 0 < hits < 0.01 * T
        frees = [_codes(sp, QS[:, 1], QE[:, 1], i, min(i + (1 << 22), Tf), Tf).any() for i in range(0, Tf, 1 << 22)]
        assert not any(frees)
    got = res.cpu().numpy()
    assert total > 1.9 * T
    assert got[0] != 0 and got[1] == 0
    assert np.array_equal(got[2:] != 0, want != 0)


def test_edges_of_several_slices(workload_dir):
    """Windows of about 1,024 ranks (a compaction block's slice) and of many
    slices, short edges between them: the oracle's decisions, and every sample
    of the free edges scheduled."""
    import torch

    import gpuprm_amd
    d = workload_dir(1)
    dq = 2e-5
    sp = gpu_space(d, dq)
    rng = np.random.default_rng(8)
    T = np.array([1364, 1365, 1366, 1367, 1381, 2731, 4095, 4097, 30000, 100003] * 6 + [3, 17, 200] * 40)
    rng.shuffle(T)
    QS = rng.uniform(-3.0, 3.0, size=(4, len(T)))
    u = rng.normal(size=QS.shape)
    QE = QS + u / np.linalg.norm(u, axis=0) * (T - 0.5) * dq
    QS, QE = QS.astype(np.float32), QE.astype(np.float32)
    want, total = OracleScene(d, dq).indicator2(QS, QE, nthreads=8)
    assert 0 < (want != 0).sum() < len(want)
    qs, qe = torch.from_numpy(QS).cuda(), torch.from_numpy(QE).cuda()
    res = torch.full((len(T),), 7, dtype=torch.int32, device="cuda")
    print("slices: %d edges" % len(T), flush=True)
    st = sp.indicator2_dev(qs, qe, res)
    assert st.samples_total == total and np.array_equal(res.cpu().numpy() != 0, want != 0)
    free = torch.from_numpy(np.flatnonzero(want == 0)).cuda()
    st = sp.indicator2_dev(qs[:, free].contiguous(), qe[:, free].contiguous(), res[:len(free)])
    assert st.samples_scheduled == st.samples_total and not res[:len(free)].any()
    res.fill_(7)
    gpuprm_amd.SceneBatch([sp]).indicator2_dev([qs], [qe], [res])
    assert np.array_equal(res.cpu().numpy() != 0, want != 0)


def gpu_space(d, dq):
    import gpuprm_amd
    sp = gpuprm_amd.RobotConfigspace(d, dq, 1 << 16)
    sp.init(0, 1)
    return sp
