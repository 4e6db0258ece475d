"""The surrogate's gradients over the edges of their splits: chunks of 32 rows
(4 loaded ahead), splits of K (1 .. 32 of the two wide layers, 1 .. 128 of the
first; their blocks are regrouped eight splits at a time), one partial row per
forward block, against the numpy oracle (oracle/mlp.py).

Tolerance: the oracle's "bf16" mode rounds where the kernels round.  Left are
orders of float32 sums (relative 1e-5 or less) and the values that such a
difference takes over a BF16 rounding boundary, each by 2^-8 relative: if all
values did, a gradient would be off by 2^-8 = 3.9e-3 relative; they are a few
percent, so 4e-3 holds with room for three layers' worth."""
import numpy as np
import pytest

from oracle import mlp

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 33, 64, 65, 129, 255, 257, 512, 2048, 2304, 4097, 8192, 8256, 16385])
def test_gradients_over_split_edges(n):
    import torch
    import gpuprm_amd
    rng = np.random.default_rng(n)
    s = gpuprm_amd.Surrogate(ndof=6, batch=n, seed=2)
    p = s.get_params()
    Q = rng.uniform(-np.pi, np.pi, size=(6, n)).astype(np.float32)
    codes = np.where(rng.uniform(size=n) < 0.4, -1, 0).astype(np.int32)
    q, c = torch.from_numpy(Q).cuda(), torch.from_numpy(codes).cuda()
    g, L = s.gradients(q, c)
    want, want_L = mlp.gradients(p, mlp.inputs(Q), (codes != 0).astype(np.float32), "bf16")
    offs = np.cumsum([0] + mlp.SIZES)
    errs = [float(np.linalg.norm(g[a:b] - want[a:b]) / max(np.linalg.norm(want[a:b]), 1e-30))
            for a, b in zip(offs[:-1], offs[1:])]
    print("loss %.7f vs %.7f, gradient rel errors %s" % (L, want_L, " ".join("%.1e" % e for e in errs)))
    assert max(errs) < 4e-3, errs
    assert abs(L - want_L) < 1e-4 * max(1.0, abs(want_L))
    # the same call again: the same bits (the sums' orders are fixed)
    g2, L2 = s.gradients(q, c)
    assert np.array_equal(g, g2) and L == L2
