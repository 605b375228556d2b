"""The register-resident triangular solves where they can go wrong: orders
around the 64-row window, the block of four rows and the eight columns
requested ahead; bands at the edges of one and two registers a lane; far
pivots, zeros in the right hand side (whose columns are left out), singular
systems left as they are.  Compared with the oracle bit for bit; the widest
bands, and the smallest orders, take the LDS kernel.
"""
import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu

# (kl, ku): none, one-sided, kl + ku = 60 | 61 | 63 | 64 | 124 | 125 | 127 | 128,
# kl = 56 | 57 | 63 | 64
BANDS = [(0, 0), (0, 5), (3, 0), (2, 3), (30, 30), (34, 27), (63, 0), (24, 40),
         (34, 34), (56, 68), (57, 60), (62, 62), (63, 62), (63, 64), (64, 64), (1, 126)]


def _factored(rng, nb, N, kl, ku, precision):
    """Random L multipliers at most 1 in size, a U whose solves stay bounded,
    and pivots anywhere in reach."""
    ldab = 2 * kl + ku + 1
    kv = kl + ku
    z = rng.standard_normal((nb, N, ldab)) + 1j * rng.standard_normal((nb, N, ldab))
    z /= 2.0 * np.sqrt(kv + 1.0)
    z[:, :, kv] += np.exp(2j * np.pi * rng.random((nb, N)))
    j = np.arange(N)
    piv = j + rng.integers(0, kl + 1, (nb, N)) * (rng.random((nb, N)) < 0.5)
    piv = np.minimum(piv, N - 1).astype(np.int32) + 1
    return z.astype(np.complex64 if precision == "c" else np.complex128), piv


@pytest.mark.parametrize("precision", ["z", "c"])
@pytest.mark.parametrize("kl,ku", BANDS)
def test_solves_at_the_window_edges(gpu, kl, ku, precision):
    import torch
    import suzerain_amd as sa
    rng = np.random.default_rng(100 * kl + ku)
    nb, nrhs = 3, 2
    ldab = 2 * kl + ku + 1
    for N in (1, 3, 4, 5, 8, 9, 63, 64, 65, 66, 127, 128, 129, 195):
        lu, piv = _factored(rng, nb, N, kl, ku, precision)
        b = (rng.standard_normal((nb, nrhs, N)) +
             1j * rng.standard_normal((nb, nrhs, N))).astype(lu.dtype)
        b[rng.random(b.shape) < 0.1] = 0.0
        b[:, 1, N // 2:] = 0.0
        lud, pd = torch.from_numpy(lu).to(gpu), torch.from_numpy(piv).to(gpu)
        for trans in "NTC":
            bd = torch.from_numpy(b).to(gpu)
            sa.gbtrs(trans, lud, kl, ku, pd, bd, precision=precision)
            got = bd.cpu().numpy()
            for s in range(nb):
                for r in range(nrhs):
                    want = oracle.zgbtrs(trans, N, kl, ku, lu[s].reshape(-1).copy(), ldab,
                                         piv[s], b[s, r].copy())
                    np.testing.assert_array_equal(got[s, r], want, err_msg=str((trans, N, s, r)))


@pytest.mark.parametrize("precision", ["z", "c"])
@pytest.mark.parametrize("kl,ku", [(0, 0), (0, 70), (4, 4), (40, 30)])
def test_smallest_orders_in_small_and_large_batches(gpu, kl, ku, precision):
    """The smallest orders take the LDS kernel, up to a larger order for more
    than 1,024 systems: a large batch and its parts give the same bits, and the
    oracle's, on either side of each line."""
    import torch
    import suzerain_amd as sa
    rng = np.random.default_rng(7 * kl + ku)
    nb, nrhs, ldab = 1025, 2, 2 * kl + ku + 1
    for N in (1, 2, 3, 5, 6, 8, 9, 11, 12, 23, 24):
        lu, piv = _factored(rng, nb, N, kl, ku, precision)
        b = (rng.standard_normal((nb, nrhs, N)) +
             1j * rng.standard_normal((nb, nrhs, N))).astype(lu.dtype)
        lud, pd = torch.from_numpy(lu).to(gpu), torch.from_numpy(piv).to(gpu)
        for trans in "NTC":
            bd = torch.from_numpy(b).to(gpu)
            parts = bd.clone()
            sa.gbtrs(trans, lud, kl, ku, pd, bd, precision=precision)
            for i in (slice(0, 1024), slice(1024, nb)):
                sa.gbtrs(trans, lud[i], kl, ku, pd[i], parts[i], precision=precision)
            got = bd.cpu().numpy()
            np.testing.assert_array_equal(parts.cpu().numpy(), got, err_msg=str((trans, N)))
            for s in (0, nb - 1):
                for r in range(nrhs):
                    want = oracle.zgbtrs(trans, N, kl, ku, lu[s].reshape(-1).copy(), ldab,
                                         piv[s], b[s, r].copy())
                    np.testing.assert_array_equal(got[s, r], want, err_msg=str((trans, N, s)))


@pytest.mark.parametrize("trans", ["N", "T"])
def test_singular_system_keeps_its_right_hand_side(gpu, trans):
    import torch
    import suzerain_amd as sa
    N, kl, ku = 70, 5, 7
    rng = np.random.default_rng(3)
    ab = np.zeros((2, N, 2 * kl + ku + 1), dtype=np.complex128)
    ab[:, :, kl + ku] = 2.0
    ab[1, 66, kl + ku] = 0.0
    b = rng.standard_normal((2, 1, N)) + 0j
    x = torch.from_numpy(b).to(gpu)
    _, info = sa.gbsv(trans, torch.from_numpy(ab).to(gpu), kl, ku, x)
    assert info.cpu().tolist() == [0, 67]
    got = x.cpu().numpy()
    np.testing.assert_array_equal(got[0], b[0] / 2.0)
    np.testing.assert_array_equal(got[1], b[1])
