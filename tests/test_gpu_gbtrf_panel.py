"""The panel factorization (four columns at a time) of the channel band shapes, alone
and with U^T y = b solved on the way,
where it can go wrong: orders around its block of four columns, its 64-column
window and its last rows; pivots far enough to reach the columns beyond the
window; zero pivots; and infinities, whose updates must leave the columns no
interchange has reached as they are.  Compared with the oracle bit for bit
(a NaN equals a NaN), as LAPACK's column-by-column loop orders the sums.
"""
import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu

SHAPES = [(34, 34), (24, 24), (34, 20)]


def _bands(rng, nb, N, kl, ku, dom):
    ldab = 2 * kl + ku + 1
    ab = np.zeros((nb, N, ldab), dtype=np.complex128)
    for j in range(N):
        lo, hi = max(0, j - ku), min(N, j + kl + 1)
        r = kl + ku + np.arange(lo, hi) - j
        ab[:, j, r] = (rng.standard_normal((nb, hi - lo)) +
                       1j * rng.standard_normal((nb, hi - lo)))
    ab[:, :, kl + ku] += dom
    return ab


def _check(gpu, ab, kl, ku, precision):
    import torch
    import suzerain_amd as sa
    if precision == "c":
        ab = ab.astype(np.complex64)
    N, ldab = ab.shape[1:]
    abd = torch.from_numpy(ab).to(gpu)
    ipiv, info = sa.gbtrf(abd, kl, ku, precision=precision)
    lu, ipiv, info = abd.cpu().numpy(), ipiv.cpu().numpy(), info.cpu().numpy()
    for s in range(ab.shape[0]):
        ref = ab[s].reshape(-1).copy()
        with np.errstate(all="ignore"):
            rinfo, rpiv = oracle.zgbtrf(N, kl, ku, ref, ldab)
        assert info[s] == rinfo
        np.testing.assert_array_equal(ipiv[s], rpiv)
        np.testing.assert_array_equal(lu[s], ref.reshape(N, ldab))
    return ipiv


ORDERS = [1, 2, 3, 4, 5, 35, 37, 63, 64, 65, 68, 69, 70, 71, 72, 73, 76, 103, 135]


@pytest.mark.parametrize("precision", ["z", "c"])
@pytest.mark.parametrize("kl,ku", SHAPES)
@pytest.mark.parametrize("N", ORDERS)
def test_orders_around_the_blocks(gpu, N, kl, ku, precision):
    rng = np.random.default_rng(1000 * kl + ku + N)
    _check(gpu, _bands(rng, 3, N, kl, ku, 0.0), kl, ku, precision)
    _check(gpu, _bands(rng, 2, N, kl, ku, 20.0), kl, ku, precision)


@pytest.mark.parametrize("precision", ["z", "c"])
@pytest.mark.parametrize("kl,ku", SHAPES)
def test_far_pivots_and_ties(gpu, kl, ku, precision):
    """The last sub-diagonal dominates (every pivot kl rows away, so every
    fill-in column is used), then entries of equal magnitude (the first wins)
    and magnitudes that differ in the low word only."""
    rng = np.random.default_rng(kl + ku)
    N = 150
    ab = _bands(rng, 3, N, kl, ku, 0.0)
    ab[0, :, 2 * kl + ku] *= 50.0
    ab[1] = np.where(ab[1] != 0, np.sign(ab[1].real), 0)
    ab[2] = np.where(ab[2] != 0, 1 + 1e-12 * ab[2].real, 0)
    for j in range(N):                       # entries past the last row stay zero
        ab[:, j, kl + ku + N - j:] = 0
    piv = _check(gpu, ab, kl, ku, precision)
    assert (piv[0] - np.arange(1, N + 1)).max() == kl


@pytest.mark.parametrize("kl,ku", SHAPES)
def test_infinities_and_zero_columns(gpu, kl, ku):
    """An infinite entry, a NaN off the diagonal, a NaN in a pivot row and a
    column of zeros, each in a system of its own."""
    rng = np.random.default_rng(7 * kl + ku)
    N = 120
    ab = _bands(rng, 5, N, kl, ku, 20.0)
    ab[0, 50, kl + ku + 2] = np.inf
    ab[1, 41, kl + ku + 5] = np.nan
    ab[2, 62, kl + ku] = complex(np.nan, 1.0)
    ab[3, 33, :] = 0.0
    ab[4, 70, kl + ku] = 5e-324              # 1/pivot overflows
    ab[4, 70, kl + ku + 1:] = 0.0
    _check(gpu, ab, kl, ku, "z")


def _fused_entries():
    """The factorization with U^T y = b, and the L^T sweep that completes it."""
    import ctypes as C
    from suzerain_amd._lib import load
    lib = load()
    i32, i64, vp = C.c_int, C.c_longlong, C.c_void_p
    ut, lt = lib.sz_internal_zgbtrf_ut, lib.sz_internal_zgbtrs_lt
    ut.restype = lt.restype = i32
    ut.argtypes = [i32, i32, i32, vp, i32, i64, vp, i64, vp, vp, i64, i32, vp]
    lt.argtypes = [i32, i32, i32, vp, i32, i64, vp, i64, vp, i64, vp, i32, vp]
    return ut, lt


def _check_fused(gpu, rng, ab, kl, ku):
    """Factors, pivots and info against ZGBTRF, and the solutions of the systems
    without a zero pivot against ZGBTRS 'T'.  Right hand sides a stride apart
    that leaves a gap, which stays as it is."""
    import ctypes as C
    import torch
    ut, lt = _fused_entries()
    nb, N, ldab = ab.shape
    b = rng.standard_normal((nb, N + 3)) + 1j * rng.standard_normal((nb, N + 3))
    abd, bd = torch.from_numpy(ab).to(gpu), torch.from_numpy(b).to(gpu)
    ipiv = torch.zeros((nb, N), dtype=torch.int32, device=gpu)
    info = torch.full((nb,), -1, dtype=torch.int32, device=gpu)
    stream = C.c_void_p(torch.cuda.current_stream().cuda_stream)
    assert ut(N, kl, ku, abd.data_ptr(), ldab, ldab * N, ipiv.data_ptr(), N,
              info.data_ptr(), bd.data_ptr(), N + 3, nb, stream) == 0
    assert lt(N, kl, ku, abd.data_ptr(), ldab, ldab * N, ipiv.data_ptr(), N,
              bd.data_ptr(), N + 3, info.data_ptr(), nb, stream) == 0
    lu, piv, x = abd.cpu().numpy(), ipiv.cpu().numpy(), bd.cpu().numpy()
    info = info.cpu().numpy()
    np.testing.assert_array_equal(x[:, N:], b[:, N:])
    for s in range(nb):
        ref = ab[s].reshape(-1).copy()
        rinfo, rpiv = oracle.zgbtrf(N, kl, ku, ref, ldab)
        assert info[s] == rinfo
        np.testing.assert_array_equal(piv[s], rpiv)
        np.testing.assert_array_equal(lu[s], ref.reshape(N, ldab))
        if rinfo == 0:
            want = oracle.zgbtrs("T", N, kl, ku, ref, ldab, rpiv, b[s, :N].copy())
            np.testing.assert_array_equal(x[s, :N], want, err_msg=str((N, s)))
    return piv, info


@pytest.mark.parametrize("kl,ku", SHAPES)
@pytest.mark.parametrize("N", ORDERS)
def test_fused_orders_around_the_blocks(gpu, N, kl, ku):
    """As test_orders_around_the_blocks, with U^T y = b on the way: a partial
    last block's y, and the right hand sides handed over from the columns beyond
    the window."""
    rng = np.random.default_rng(2000 * kl + ku + N)
    _check_fused(gpu, rng, _bands(rng, 3, N, kl, ku, 0.0), kl, ku)
    _check_fused(gpu, rng, _bands(rng, 2, N, kl, ku, 20.0), kl, ku)


@pytest.mark.parametrize("kl,ku", SHAPES)
@pytest.mark.parametrize("N", [74, 150])
def test_fused_far_pivots_and_singular_systems(gpu, N, kl, ku):
    """Every pivot kl rows away; a zero column between two ordinary systems,
    whose solutions it must not touch; a zero last column."""
    rng = np.random.default_rng(3 * kl + ku + N)
    ab = _bands(rng, 6, N, kl, ku, 0.0)
    ab[0, :, 2 * kl + ku] *= 50.0
    for j in range(N):                       # entries past the last row stay zero
        ab[0, j, kl + ku + N - j:] = 0
    ab[2, 30, :] = 0.0
    ab[4, N - 1, :] = 0.0
    piv, info = _check_fused(gpu, rng, ab, kl, ku)
    assert (piv[0] - np.arange(1, N + 1)).max() == kl
    assert [i > 0 for i in info] == [False, False, True, False, True, False]


@pytest.mark.parametrize("kl,ku", SHAPES)
def test_arrays_aligned_as_c_double_complex(gpu, kl, ku):
    """Band storage and right hand sides 8 bytes off a 16-byte boundary, which
    C's double complex allows: the panel kernel's 16-byte transfers to LDS are
    not for them.  The factorization still gives the oracle's bits; the fused
    one declines, and has written nothing."""
    import ctypes as C
    import torch
    from suzerain_amd._lib import load
    lib, vp = load(), C.c_void_p
    f_ut, _ = _fused_entries()
    rng = np.random.default_rng(kl + 2 * ku)
    N, nb, ldab = 77, 2, 2 * kl + ku + 1
    ab = _bands(rng, nb, N, kl, ku, 0.0)
    b = rng.standard_normal((nb, N)) + 1j * rng.standard_normal((nb, N))

    def device(a, off):                      # a's doubles from element `off` on
        flat = a.reshape(-1).view(np.float64)
        d = torch.zeros(flat.size + 2, dtype=torch.float64, device=gpu)
        assert d.data_ptr() % 16 == 0
        d[off:off + flat.size] = torch.from_numpy(flat).to(gpu)
        return d, d.data_ptr() + 8 * off

    def host(d, off, a):
        return d[off:off + 2 * a.size].cpu().numpy().view(np.complex128).reshape(a.shape)

    stream = vp(torch.cuda.current_stream().cuda_stream)
    ipiv = torch.zeros((nb, N), dtype=torch.int32, device=gpu)
    info = torch.zeros((nb,), dtype=torch.int32, device=gpu)
    for oa, ob in ((1, 0), (0, 1)):
        ad, ap = device(ab, oa)
        bd, bp = device(b, ob)
        assert f_ut(N, kl, ku, ap, ldab, ldab * N, ipiv.data_ptr(), N, info.data_ptr(),
                    bp, N, nb, stream) == 1
        torch.cuda.synchronize()
        np.testing.assert_array_equal(host(ad, oa, ab), ab)
        np.testing.assert_array_equal(host(bd, ob, b), b)
    ad, ap = device(ab, 1)
    assert lib.sz_zgbtrf_batched(N, kl, ku, ap, ldab, ldab * N, ipiv.data_ptr(), N,
                                 info.data_ptr(), nb, stream) == 0
    torch.cuda.synchronize()
    lu = host(ad, 1, ab)
    for s in range(nb):
        ref = ab[s].reshape(-1).copy()
        rinfo, rpiv = oracle.zgbtrf(N, kl, ku, ref, ldab)
        assert int(info[s]) == rinfo == 0
        np.testing.assert_array_equal(ipiv[s].cpu().numpy(), rpiv)
        np.testing.assert_array_equal(lu[s], ref.reshape(N, ldab))
