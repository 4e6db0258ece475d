"""Inference over the edges of its tiles: 64 rows a tile, 256 blocks, two tiles
of a block in flight (the second absent or ragged, an odd number of tiles per
block), 1 to 16 joints, against the numpy oracle (oracle/mlp.py).

Tolerance: the oracle's "bf16" mode rounds where the kernel rounds; what is
left is the order of float32 sums of at most 256 terms and, where such a
difference crosses a BF16 rounding boundary, one step (2^-8 relative) of single
activations.  256 activations with weights of about 1/16 that each differ by
2^-8 of an activation of at most about 1, at random, move z by
16 * 2^-8 / 16 = 4e-3 at the very most, if all were to round differently;
few percent do, which leaves about 1e-3, and sigmoid takes a quarter: 2.5e-4.
Twice that is the bound.  A row's result depends on nothing but the row, so the
same rows in other tiles have to give the same bits."""
import numpy as np
import pytest

from oracle import mlp

pytestmark = pytest.mark.gpu

T = 64 * 256  # rows of one tile in every block of a 256-unit device


@pytest.mark.parametrize("n", [1, 63, 64, 65, T, T + 1, 2 * T - 1, 2 * T + 1, 3 * T + 64, 5 * T - 65])
@pytest.mark.parametrize("nd", [4, 16])
def test_rows_over_tile_edges(n, nd):
    import torch
    import gpuprm_amd
    rng = np.random.default_rng(n + nd)
    s = gpuprm_amd.Surrogate(ndof=nd, batch=64, seed=3)
    off = n + 5
    Q = rng.uniform(-np.pi, np.pi, size=(nd, off)).astype(np.float32)
    q = torch.from_numpy(Q).cuda()
    prob = torch.full((n + 64,), -1.0, dtype=torch.float32, device="cuda")
    s.predict(q, prob[:n], offset=off)
    assert bool((prob[n:] == -1.0).all())
    # rows of the first, middle and last tiles, against the oracle
    rows = np.unique(np.concatenate([np.arange(min(n, 130)), np.arange(n // 2, min(n, n // 2 + 130)),
                                     np.arange(max(0, n - 130), n)]))
    want, _ = mlp.forward(s.get_params(), mlp.inputs(np.ascontiguousarray(Q[:, rows])), "bf16")
    got = prob[:n].cpu().numpy()
    print("max |dp| %.2e" % float(np.max(np.abs(got[rows] - want))))
    assert float(np.max(np.abs(got[rows] - want))) < 5e-4
    # the same rows from a call of their own (other tiles and blocks)
    again = torch.zeros(rows.size, dtype=torch.float32, device="cuda")
    s.predict(torch.from_numpy(np.ascontiguousarray(Q[:, rows])).cuda(), again)
    assert np.array_equal(again.cpu().numpy(), got[rows])
