"""Support scan on polytopes with faces of more than three vertices: after
rounding to floats the face's vertices are not quite in one plane, so the
certificate's cone coefficients come out slightly negative.  Prisms of 3 to 14
corners (28 vertices), turned, exact and with their vertices moved by up to
1e-3, and rows of a triangulation (whose diagonals lie in the faces).  Codes
must be the oracle's."""
import tempfile

import numpy as np
import pytest

import scenes
from oracle.oracle import OracleScene

pytestmark = pytest.mark.gpu


def _prism(k):
    a = 2 * np.pi * np.arange(k) / k
    ring = np.stack([0.3 * np.cos(a), 0.25 * np.sin(a)], axis=1)
    V = np.concatenate([np.c_[ring, np.full(k, -0.3)], np.c_[ring, np.full(k, 0.3)]])
    nb = [set() for _ in V]
    for i in range(k):
        j = (i + 1) % k
        for u, v in ((i, j), (k + i, k + j), (i, k + i), (i, k + j)):  # sides, with a diagonal each
            nb[u].add(v)
            nb[v].add(u)
        if 1 < i < k - 1:  # both ends as fans
            for base in (0, k):
                nb[base].add(base + i)
                nb[base + i].add(base)
    return V, [sorted(x) for x in nb]


@pytest.mark.parametrize("moved", [0.0, 1e-7, 1e-5, 1e-3])
@pytest.mark.parametrize("corners", [3, 4, 6, 9, 14])
def test_prisms(workload_dir, corners, moved):
    import torch

    import gpuprm_amd
    base = scenes.read_dir(workload_dir(1))
    rng = np.random.default_rng(corners + int(moved * 1e8))
    V, rows = _prism(corners)
    nobs = int((base["sys"] == 0).sum())
    vo, eo = np.concatenate([[0], np.cumsum(base["n"])]), np.concatenate([[0], np.cumsum(base["m"])])
    parts = {k: [] for k in ("n", "m", "vertices", "dsp", "cnt", "dest")}
    for k in range(len(base["n"])):
        if k < nobs:
            R = np.linalg.qr(rng.normal(size=(3, 3)))[0]
            c = rng.uniform(-2, 2, 3)
            v, r = ((V + rng.uniform(-moved, moved, V.shape)) @ R.T + c).astype(np.float32), rows
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
    d = scenes.write_dir(s, tempfile.mkdtemp(prefix="gprm_faces_"))
    sp = gpuprm_amd.RobotConfigspace(d, 0.01, 1 << 16)
    sp.init(0, 1)
    Q = rng.uniform(-np.pi, np.pi, size=(4, 8000)).astype(np.float32)
    Q = np.clip(Q, s["mins"][:, None], s["maxs"][:, None]).astype(np.float32)
    r = torch.zeros(Q.shape[1], dtype=torch.int32, device="cuda")
    print("prism of %d corners, moved %g" % (corners, moved), flush=True)
    sp.indicator_dev(torch.from_numpy(Q).cuda(), r)
    assert np.array_equal(r.cpu().numpy(), OracleScene(d).indicator_batch(Q, nthreads=8))
