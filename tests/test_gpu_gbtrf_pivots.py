"""Pivot choice of the LDS-window factorization, a row a lane (kl < 64) and by
strides: ties (the first of equal magnitudes wins), a NaN in and below the
pivot row, an infinity, a zero column.  Compared with the oracle bit for bit.
"""
import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", ["z", "c"])
@pytest.mark.parametrize("kl,ku", [(0, 3), (1, 1), (17, 11), (63, 20), (64, 10)])
def test_pivots_match_oracle(gpu, kl, ku, precision):
    import torch
    import suzerain_amd as sa
    rng = np.random.default_rng(10 * kl + ku)
    N, ldab, nb = 90, 2 * kl + ku + 1, 5
    ab = np.zeros((nb, N, ldab), dtype=np.complex128 if precision == "z" else np.complex64)
    for j in range(N):
        lo, hi = max(0, j - ku), min(N, j + kl + 1)
        r = kl + ku + np.arange(lo, hi) - j
        ab[:, j, r] = (rng.integers(-2, 3, (nb, hi - lo)) +
                       1j * rng.integers(-2, 3, (nb, hi - lo)))
    ab[1:, :, kl + ku] += 9.0
    ab[2, 20, kl + ku:] = 0.0                            # zero pivot column
    ab[3, 30, min(kl + ku + 1, ldab - 1)] = np.nan
    ab[4, 30, kl + ku] = np.inf
    abd = torch.from_numpy(ab).to(gpu)
    ipiv, info = sa.gbtrf(abd, kl, ku, precision=precision)
    lu, ipiv, info = abd.cpu().numpy(), ipiv.cpu().numpy(), info.cpu().numpy()
    for s in range(nb):
        ref = ab[s].reshape(-1).copy()
        with np.errstate(all="ignore"):
            rinfo, rpiv = oracle.zgbtrf(N, kl, ku, ref, ldab)
        assert info[s] == rinfo
        np.testing.assert_array_equal(ipiv[s], rpiv)
        np.testing.assert_array_equal(lu[s], ref.reshape(N, ldab))
