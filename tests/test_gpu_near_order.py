"""What gprm_radius_neighbours leaves in its arrays, without the wrapper's own
sort: pairs by query and, for queries of at most 1,024 matches, by node, also
across the scan's chunks of 1,024 queries; the first `cap` of them where there
are more, and nothing beyond."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _search(nodes, queries, D, cap):
    import torch

    import gpuprm_amd
    nd, n = nodes.shape
    nq = queries.shape[1]
    lo, hi = np.full(nd, -np.pi, np.float32), np.full(nd, np.pi, np.float32)
    fp = C.POINTER(C.c_float)
    dn, dq = (torch.from_numpy(np.ascontiguousarray(a)).cuda() for a in (nodes, queries))
    out = torch.full((3, cap + 64), -7, dtype=torch.int32, device="cuda")
    total = C.c_longlong(-1)
    torch.cuda.synchronize()
    rc = gpuprm_amd.lib().gprm_radius_neighbours(
        nd, C.c_void_p(dn.data_ptr()), n, n, C.c_void_p(dq.data_ptr()), nq, nq, lo.ctypes.data_as(fp),
        hi.ctypes.data_as(fp), D, C.c_void_p(out[0].data_ptr()), C.c_void_p(out[1].data_ptr()),
        C.c_void_p(out[2].data_ptr()), cap, C.byref(total), None)
    assert rc == 0
    q, node, d2 = out.cpu().numpy()
    assert (out[:, min(cap, total.value):] == -7).all()
    return total.value, q, node, d2.view(np.float32)


def _brute(nodes, queries, D):
    s = np.zeros((queries.shape[1], nodes.shape[1]), np.float32)
    for i in range(nodes.shape[0]):
        diff = nodes[i][None, :] - queries[i][:, None]
        s = s + diff * diff
    q, n = np.nonzero(s < np.float32(D) * np.float32(D))  # by query, then node
    return q.astype(np.int32), n.astype(np.int32), s[q, n]


@pytest.mark.parametrize("nq", [1, 1023, 1024, 1025, 2048, 5000])
def test_pairs_come_sorted(nq):
    rng = np.random.default_rng(nq)
    nodes = rng.uniform(-np.pi, np.pi, size=(4, 3000)).astype(np.float32)
    queries = rng.uniform(-np.pi, np.pi, size=(4, nq)).astype(np.float32)
    q, n, d2 = _brute(nodes, queries, 0.7)
    assert len(q) >= nq // 4
    print("near order: %d queries, %d pairs" % (nq, len(q)), flush=True)
    total, gq, gn, gd = _search(nodes, queries, 0.7, len(q) + 100)
    k = len(q)
    assert total == k
    assert np.array_equal(gq[:k], q) and np.array_equal(gn[:k], n)
    assert np.array_equal(gd[:k].view(np.int32), d2.view(np.int32))
    for cap in (0, 1, k // 2, k - 1, k):  # fewer slots than pairs
        total, gq, gn, gd = _search(nodes, queries, 0.7, cap)
        assert total == k
        assert np.array_equal(gq[:cap], q[:cap]) and np.array_equal(gn[:cap], n[:cap])


@pytest.mark.parametrize("matches", [1023, 1024, 1025, 2500])
def test_queries_of_many_matches(matches):
    """One dense query between sparse ones: in node order up to 1,024 matches,
    the same pairs in any order beyond, the other queries' places unmoved."""
    rng = np.random.default_rng(matches)
    dense = rng.uniform(-0.05, 0.05, size=(3, matches))
    sparse = rng.uniform(1.0, 3.0, size=(3, 500))
    nodes = np.concatenate([dense, sparse], axis=1)[:, rng.permutation(matches + 500)].astype(np.float32)
    queries = np.concatenate([rng.uniform(1.0, 3.0, size=(3, 40)), np.zeros((3, 1)),
                              rng.uniform(1.0, 3.0, size=(3, 40))], axis=1).astype(np.float32)
    q, n, d2 = _brute(nodes, queries, 0.4)
    assert (q == 40).sum() == matches
    total, gq, gn, gd = _search(nodes, queries, 0.4, len(q))
    assert total == len(q) and np.array_equal(gq[:total], q)
    if matches > 1024:
        o = np.lexsort((gn[:total], gq[:total]))
        gn, gd = gn[o], gd[o]
    assert np.array_equal(gn[:total], n)
    assert np.array_equal(gd[:total].view(np.int32), d2.view(np.int32))
