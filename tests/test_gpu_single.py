"""Single configurations (the small call's kernel, whose first wave computes
the joints side by side) against the oracle and the batched kernels: random
ones, joints exactly on their limits, and one joint out of its limits at each
place."""
import numpy as np
import pytest

import gpuprm_amd
import scenes
from oracle.oracle import OracleScene

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("workload", [1, 2, 3])
def test_single_configurations(workload_dir, workload):
    d = workload_dir(workload)
    sp = gpuprm_amd.RobotConfigspace(d, 0.01, 1 << 12)
    sp.init(0, 1)
    nd = sp.dim()
    s = scenes.read_dir(d)
    rng = np.random.default_rng(workload)
    Q = rng.uniform(-np.pi, np.pi, size=(nd, 64 + 4 * nd)).astype(np.float32)
    Q = np.clip(Q, s["mins"][:, None], s["maxs"][:, None]).astype(np.float32)
    for j in range(nd):
        at = 64 + 4 * j
        Q[j, at], Q[j, at + 1] = s["mins"][j], s["maxs"][j]
        Q[j, at + 2] = np.nextafter(s["mins"][j], np.float32(-np.inf))
        Q[j, at + 3] = np.nextafter(s["maxs"][j], np.float32(np.inf))
    want = OracleScene(d).indicator_batch(Q, nthreads=8)
    got = np.array([sp.indicator(Q[:, k].copy()) for k in range(Q.shape[1])])
    assert np.array_equal(got, want)
    assert np.array_equal(sp.indicator_batch(Q), want)
