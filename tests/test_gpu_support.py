"""The full tests' support scan (kernels.hip, support) against the oracle's
hill climb where the two could part: exact ties (boxes and configurations
along the axes), flat and degenerate polytopes, rows that miss edges (the
climb stops short of the support vertex there), equal vertices, and vertex
counts around the scan's limit.  Codes and decisions must be the oracle's."""
import tempfile

import numpy as np
import pytest

import scenes
from oracle.oracle import OracleScene

pytestmark = pytest.mark.gpu


def _box(h):
    return np.array([[x, y, z] for x in (-h, h) for y in (-h, h) for z in (-h, h)], np.float32)


def _complete(n):
    return [[j for j in range(n) if j != i] for i in range(n)]


BOX_EDGES = [[i ^ 1, i ^ 2, i ^ 4] for i in range(8)]


def _sphere(n):
    i = np.arange(n) + 0.5
    t, p = np.arccos(1 - 2 * i / n), np.pi * (1 + 5 ** 0.5) * i
    return np.stack([np.cos(p) * np.sin(t), np.sin(p) * np.sin(t), np.cos(t)], axis=1).astype(np.float32) * np.float32(0.3)


def _hull(V):
    from scipy.spatial import ConvexHull
    nb = [set() for _ in V]
    for a, b, c in ConvexHull(V).simplices:
        nb[a] |= {b, c}
        nb[b] |= {a, c}
        nb[c] |= {a, b}
    return [sorted(int(x) for x in s) for s in nb]


def _shapes(kind):
    """(vertices, neighbour rows) of the obstacles' shape."""
    if kind == "box":
        return _box(0.25), BOX_EDGES
    if kind == "box_complete":
        return _box(0.25), _complete(8)
    if kind == "box_missing_edge":
        rows = [list(r) for r in BOX_EDGES]
        rows[0].remove(1)
        rows[1].remove(0)
        return _box(0.25), rows
    if kind == "ring_rows":  # every row names one neighbour only
        return _box(0.25), [[(i + 1) % 8] for i in range(8)]
    if kind == "point":
        return np.zeros((1, 3), np.float32), [[0]]
    if kind == "segment":
        return np.array([[-0.4, 0, 0], [0.4, 0, 0]], np.float32), [[1], [0]]
    if kind == "square":
        return _box(0.3)[[0, 1, 3, 2]], [[1, 3], [0, 2], [1, 3], [0, 2]]
    if kind == "equal_vertices":
        V = _box(0.25)
        return np.concatenate([V, V[:1]]), _complete(9)
    if kind == "thin":
        return _box(0.25) * np.array([1, 1e-4, 1], np.float32), BOX_EDGES
    n = int(kind[6:])
    V = _sphere(n)
    return V, _hull(V) if n > 3 else _complete(n)


KINDS = ["box", "box_complete", "box_missing_edge", "ring_rows", "point", "segment", "square", "equal_vertices", "thin",
         "sphere4", "sphere5", "sphere17", "sphere31", "sphere32", "sphere33"]


@pytest.mark.parametrize("kind", KINDS)
def test_support_matches_climb(workload_dir, kind):
    import torch

    import gpuprm_amd
    base = scenes.read_dir(workload_dir(1))
    rng = np.random.default_rng(len(kind) + sum(map(ord, kind)))
    V, rows = _shapes(kind)
    nobs = int((base["sys"] == 0).sum())
    vo, eo = np.concatenate([[0], np.cumsum(base["n"])]), np.concatenate([[0], np.cumsum(base["m"])])
    parts = {k: [] for k in ("n", "m", "vertices", "dsp", "cnt", "dest")}
    for k in range(len(base["n"])):
        if k < nobs:
            # every second obstacle stays on the axes, at a coarse grid
            # position: exact ties with configurations along the axes
            R = np.eye(3) if k % 2 else np.linalg.qr(rng.normal(size=(3, 3)))[0]
            c = np.round(rng.uniform(-2, 2, 3) * 4) / 4
            v, r = (V @ R.T + c).astype(np.float32), rows
        else:
            v = base["vertices"].reshape(-1, 3)[vo[k]:vo[k + 1]]
            d, cn, de = base["dsp"][vo[k]:vo[k + 1]], base["cnt"][vo[k]:vo[k + 1]], base["dest"][eo[k]:eo[k + 1]]
            r = [list(de[a:a + b]) for a, b in zip(d, cn)]
        cnt = np.array([len(x) for x in r], np.int32)
        parts["n"].append(len(v))
        parts["m"].append(int(cnt.sum()))
        parts["vertices"].append(v.ravel())
        parts["cnt"].append(cnt)
        parts["dsp"].append(np.concatenate([[0], np.cumsum(cnt)[:-1]]).astype(np.int32))
        parts["dest"].append(np.concatenate([np.asarray(x, np.int32) for x in r]))
    s = dict(base, n=np.array(parts["n"], np.int32), m=np.array(parts["m"], np.int32),
             **{k: np.concatenate(parts[k]) for k in ("vertices", "dsp", "cnt", "dest")})
    d = scenes.write_dir(s, tempfile.mkdtemp(prefix="gprm_support_"))
    o = OracleScene(d)
    sp = gpuprm_amd.RobotConfigspace(d, 0.01, 1 << 16)
    sp.init(0, 1)
    Q = rng.uniform(-np.pi, np.pi, size=(4, 6000)).astype(np.float32)
    Q[:, :2000] = np.round(Q[:, :2000] / (np.pi / 4)) * (np.pi / 4)  # along the axes
    Q[:, 0] = 0.0
    Q = np.clip(Q, s["mins"][:, None], s["maxs"][:, None]).astype(np.float32)
    r = torch.zeros(Q.shape[1], dtype=torch.int32, device="cuda")
    print("support: %s" % kind, flush=True)
    sp.indicator_dev(torch.from_numpy(Q).cuda(), r)
    want = o.indicator_batch(Q, nthreads=8)
    assert np.array_equal(r.cpu().numpy(), want)
    small = np.array([sp.indicator(Q[:, k].copy()) for k in range(0, 2400, 50)])
    assert np.array_equal(small, want[0:2400:50])
    QE = np.clip(Q[:, :400] + rng.uniform(-0.4, 0.4, size=(4, 400)), -np.pi, np.pi).astype(np.float32)
    re = torch.zeros(400, dtype=torch.int32, device="cuda")
    sp.indicator2_dev(torch.from_numpy(Q[:, :400].copy()).cuda(), torch.from_numpy(QE).cuda(), re)
    wante, _ = o.indicator2(Q[:, :400].copy(), QE, nthreads=8)
    assert np.array_equal(re.cpu().numpy() != 0, wante != 0)
