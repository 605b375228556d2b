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


@pytest.mark.parametrize("real", [False, True])
@pytest.mark.parametrize("n,k", [(8, 8), (33, 6), (255, 8), (257, 5)])
def test_strides_and_types(gpu, n, k, real):
    """Elements and pencils apart (increments of 1, 2 and 3, gaps between the
    pencils), real and complex: the results, and the gaps as they were."""
    import torch
    import suzerain_amd as sa
    from suzerain_amd._lib import load, cplx
    op = sa.BsplineOp.channel(n, k, 2.0)
    rng = np.random.default_rng(n + k)
    dt = np.float64 if real else np.complex128
    stream = torch.cuda.current_stream().cuda_stream
    for nrhs, incx, incy, gap in ((1, 1, 2, 0), (1, 3, 1, 0), (5, 2, 3, 0), (7, 1, 1, 5),
                                  (19, 3, 2, 4)):
        ldx, ldy = n * incx + gap, n * incy + gap
        fill = lambda m: rng.standard_normal(m) + (0 if real else 1j * rng.standard_normal(m))
        x, y = fill(nrhs * ldx).astype(dt), fill(nrhs * ldy).astype(dt)
        X = np.stack([x[p * ldx:p * ldx + n * incx:incx] for p in range(nrhs)])
        Y = np.stack([y[p * ldy:p * ldy + n * incy:incy] for p in range(nrhs)])
        for d in (0, 2):
            for beta in (0.0, -1.5):
                alpha = 0.75 if real else 0.75 - 2j
                xd, yd = torch.from_numpy(x).to(gpu), torch.from_numpy(y.copy()).to(gpu)
                f = (load().sz_bsplineop_accumulate_batched if real
                     else load().sz_bsplineop_accumulate_complex_batched)
                assert f(op._w, d, nrhs, alpha if real else cplx(alpha), xd.data_ptr(), incx,
                         ldx, beta if real else cplx(beta), yd.data_ptr(), incy, ldy,
                         stream) == 0
                got = yd.cpu().numpy()
                D = op.dense(d)
                want = y.copy()
                # (the bound of test_rows_and_pencils)
                for p in range(nrhs):
                    at = slice(p * ldy, p * ldy + n * incy, incy)
                    want[at] = alpha * (D @ X[p]) + beta * Y[p]
                    bound = (2 * k + 8) * 2.0 ** -52 * (
                        2 * abs(alpha) * (np.abs(D) @ np.abs(X[p])) +
                        2 * abs(beta) * np.abs(Y[p]) + 1e-300)
                    assert (np.abs(got[at] - want[at]) <= bound).all(), (nrhs, d, beta, p)
                    got[at] = want[at]
                np.testing.assert_array_equal(got, want)     # the gaps
