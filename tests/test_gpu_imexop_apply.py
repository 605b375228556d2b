"""The matrix-free operator where its launch can go wrong: orders around the
wavefront and around the two block sizes, one and many systems a block (uneven
last shares), narrow and wide bands (whose first and last rows reach the zeros
kept around a field), an infinity in x, beta zero or not, an absent field.
Compared with the oracle bit for bit (a NaN equals a NaN).
"""
import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu

SCEN = (3000.0, 0.7, 1.5, 0.3, 1.4)
PHI = complex(-2.5e-3, 1.0e-4)


@pytest.mark.parametrize("n,k,nsys", [(9, 4, 1), (9, 8, 2600), (24, 8, 1100), (63, 6, 3),
                                      (64, 8, 700), (65, 5, 7), (96, 8, 515), (192, 8, 5),
                                      (253, 8, 2), (254, 8, 2), (255, 8, 2), (300, 12, 3),
                                      (384, 8, 1), (385, 8, 300), (480, 4, 2)])
def test_apply_matches_oracle(gpu, n, k, nsys):
    import torch
    import suzerain_amd as sa
    from suzerain_amd.imexop import Imexop
    rng = np.random.default_rng(1000 * n + k)
    op = sa.BsplineOp.channel(n, k, 3.0)
    dt = np.stack([op.D_T(d) for d in range(3)])
    ops = oracle.Ops(bands=(dt, op.kl, op.ku, op.max_kl, op.max_ku))
    imx = Imexop(op, *SCEN)
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(gpu)
    refs = rng.uniform(-1, 1, (26, n))
    km, kn = rng.uniform(-30, 30, nsys), rng.uniform(-30, 30, nsys)
    x = rng.standard_normal((5, nsys, n)) + 1j * rng.standard_normal((5, nsys, n))
    y = rng.standard_normal((5, nsys, n)) + 1j * rng.standard_normal((5, nsys, n))
    x[1, nsys // 2, min(5, n - 1)] = np.inf
    check = sorted({0, 1, nsys // 2, nsys - 1} |
                   set(rng.integers(0, nsys, 6).tolist())) if nsys > 8 else range(nsys)
    off = dev(np.arange(nsys, dtype=np.int64) * n)
    refd, kmd, knd = dev(refs), dev(km), dev(kn)
    for beta, present in ((0.5 - 2j, (True,) * 5), (0.0, (True,) * 5),
                          (0.5 - 2j, (True, True, False, True, True))):
        xd, yd = dev(x), dev(y)
        imx.accumulate(PHI, kmd, knd, refd, [xd[f] if present[f] else None for f in range(5)],
                       beta, [yd[f] if present[f] else None for f in range(5)], nsys=nsys,
                       inoff=off, outoff=off)
        got = yd.cpu().numpy()
        for s in check:
            if s >= nsys:
                continue
            want = np.ascontiguousarray(y[:, s])
            with np.errstate(all="ignore"):
                oracle.imexop_accumulate(PHI, km[s], kn[s], SCEN, refs, ops,
                                         np.ascontiguousarray(x[:, s]), beta, want,
                                         present=present)
            np.testing.assert_array_equal(got[:, s], want, err_msg=str((s, beta, present)))


@pytest.mark.parametrize("n", [24, 96, 260])
def test_strided_profiles_and_scattered_pencils(gpu, n):
    """Profiles a stride apart and pencils at offsets of their own, input and
    output at different ones, in place where they are the same: the same bits as
    the contiguous call, and nothing else written."""
    import torch
    import suzerain_amd as sa
    from suzerain_amd.imexop import Imexop
    rng = np.random.default_rng(n)
    nsys, beta = 37, 0.5 - 2j
    imx = Imexop(sa.BsplineOp.channel(n, 8, 3.0), *SCEN)
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(gpu)
    crand = lambda *s: rng.standard_normal(s) + 1j * rng.standard_normal(s)
    refs = rng.uniform(-1, 1, (26, n))
    km, kn = dev(rng.uniform(-30, 30, nsys)), dev(rng.uniform(-30, 30, nsys))
    x, y = crand(5, nsys, n), crand(5, nsys, n)
    want = dev(y)
    imx.accumulate(PHI, km, kn, dev(refs), dev(x), beta, want)
    want = want.cpu().numpy()
    strided = dev(refs.T).T                          # (26, n), stride(1) = 26
    assert strided.stride(1) == 26
    place = lambda: rng.permutation(2 * nsys)[:nsys] * (n + 3)
    io, oo = place(), place()
    xb, yb = crand(5, 2 * nsys * (n + 3)), crand(5, 2 * nsys * (n + 3))
    for s in range(nsys):
        xb[:, io[s]:io[s] + n] = x[:, s]
        yb[:, oo[s]:oo[s] + n] = y[:, s]
    yd = dev(yb)
    imx.accumulate(PHI, km, kn, strided, list(dev(xb)), beta, list(yd), nsys=nsys,
                   inoff=dev(io), outoff=dev(oo))
    for s in range(nsys):
        yb[:, oo[s]:oo[s] + n] = want[:, s]
    np.testing.assert_array_equal(yd.cpu().numpy(), yb)
    xd = dev(x)                                      # y = (M + phi L) x + beta x
    imx.accumulate(PHI, km, kn, dev(refs), xd, beta, xd)
    other = dev(x)
    imx.accumulate(PHI, km, kn, dev(refs), dev(x), beta, other)
    np.testing.assert_array_equal(xd.cpu().numpy(), other.cpu().numpy())
