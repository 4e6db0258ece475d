"""Point checks around the sizes where the launch changes its shape (few pairs
a wave: four waves per SIMD; many: six rounds of units): the codes must be
those of one explicit shape over the whole range, and the oracle's on a part."""
import numpy as np
import pytest

import gpuprm_amd
from oracle.oracle import OracleScene

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("workload", [1, 3])
def test_codes_across_shapes(workload_dir, workload):
    import torch
    d = workload_dir(workload)
    sp = gpuprm_amd.RobotConfigspace(d, 0.01, 1 << 20)
    sp.init(0, 1)
    shape = sp.get_launch_shape()
    waves = shape.grid * shape.block // 64
    M = int(np.fromfile(d + "/pairs/M.bin", np.int32)[0])
    sizes = []
    for per_wave in (24, 200):
        edge = per_wave * waves // M * 64  # the last size of the lower side
        sizes += [edge - 63, edge, edge + 1, edge + 65]
    sizes = [n for n in sizes if n <= 1 << 21]
    rng = np.random.default_rng(workload)
    Q = rng.uniform(-np.pi, np.pi, size=(sp.dim(), max(sizes))).astype(np.float32)
    q = torch.from_numpy(Q).cuda()
    got = []
    for n in sizes:
        print("point shapes: workload %d, n %d" % (workload, n), flush=True)
        r = torch.full((n + 64,), 77, dtype=torch.int32, device="cuda")
        sp.indicator_dev(q[:, :n].contiguous(), r)
        assert bool((r[n:] == 77).all())
        got.append(r[:n].clone())
    sp.set_launch_shape(256, 5, 128)
    want = torch.zeros(max(sizes), dtype=torch.int32, device="cuda")
    sp.indicator_dev(q, want)
    for n, g in zip(sizes, got):
        assert torch.equal(g, want[:n])
    k = 4000
    assert np.array_equal(want[:k].cpu().numpy(), OracleScene(d).indicator_batch(Q[:, :k].copy(), nthreads=8))
