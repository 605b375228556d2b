"""The B-spline operator apply around its block of 256 rows: orders at the order
of the spline (every row at an edge of the matrix) and around the block, odd
numbers of pencils, beta zero or not; an infinity reaches the rows whose band
holds its column and no other.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,k", [(6, 4), (8, 8), (9, 8), (17, 5), (63, 6), (96, 8), (255, 8),
                                 (256, 8), (257, 8), (600, 12)])
@pytest.mark.parametrize("d", [0, 1, 2])
def test_rows_and_pencils(gpu, n, k, d):
    import torch
    import suzerain_amd as sa
    op = sa.BsplineOp.channel(n, k, 2.0)
    D = op.dense(d)
    rng = np.random.default_rng(n * k + d)
    for nrhs, beta in ((1, 0.0), (3, 0.75 + 2j), (37, 1.0)):
        x = rng.standard_normal((nrhs, n)) + 1j * rng.standard_normal((nrhs, n))
        y = rng.standard_normal((nrhs, n)) + 1j * rng.standard_normal((nrhs, n))
        alpha = 0.5 - 2j
        xd, yd = torch.from_numpy(x).to(gpu), torch.from_numpy(y.copy()).to(gpu)
        op.accumulate(d, alpha, xd, beta, yd)
        want = alpha * (x @ D.T) + beta * y
        # at most 2k - 1 terms of one rounding each, then alpha and beta:
        # (2k + 8) units of 2^-53 of the sum of magnitudes, both sides
        bound = (2 * k + 8) * 2.0 ** -52 * (2 * abs(alpha) * (np.abs(x) @ np.abs(D).T) +
                                            2 * abs(beta) * np.abs(y) + 1e-300)
        assert (np.abs(yd.cpu().numpy() - want) <= bound).all()
    c = n // 2
    x[:] = 1.0
    x[0, c] = np.inf
    xd, yd = torch.from_numpy(x).to(gpu), torch.zeros((nrhs, n), dtype=torch.complex128,
                                                      device=gpu)
    op.accumulate(d, 1.0, xd, 0.0, yd)
    ok = np.isfinite(yd.cpu().numpy())
    i = np.arange(n)
    reached = (i - op.ku[d] <= c) & (c <= i + op.kl[d])
    assert (ok[0] == ~reached).all() and ok[1:].all()
