"""Every length run as two register passes, as the z and as the x length, with
line counts that leave tiles and line pairs partly filled, and with extents
below the 3/2 rule's (fewer retained modes).  Against numpy's pocketfft, within
the bound of a length-n transform's rounding: a few eps log2(n) of the largest
result."""
import numpy as np
import pytest

from test_gpu_fft import backward_numpy, dealiased_wave, forward_numpy

pytestmark = pytest.mark.gpu

LENGTHS = (12, 18, 24, 36, 48, 54, 72, 96, 108, 144, 162, 192, 216, 288, 384)


@pytest.mark.parametrize("Ny,short", [(1, 0), (5, 0), (16, 3), (33, 1)])
@pytest.mark.parametrize("n", LENGTHS)
def test_two_pass_lengths(gpu, n, Ny, short):
    import torch
    from suzerain_amd.fft import PencilFFT
    for dNx, dNz in ((n, 18), (12, n)):
        Nx, Nz = max(2 * dNx // 3 - short, 2), max(2 * dNz // 3 - short, 2)
        print(f"case Ny={Ny} Nx={Nx} dNx={dNx} Nz={Nz} dNz={dNz}", flush=True)
        rng = np.random.default_rng(n + Ny)
        W, keep = dealiased_wave(rng, 2, Ny, Nx, dNx, Nz, dNz)
        fft = PencilFFT(Ny, Nx, dNx, Nz, dNz)
        tol = 4 * np.finfo(float).eps * np.log2(dNx * dNz)
        junk = W + (~keep)[None, :, :, None]          # dealiased modes count as zero
        Pd = torch.full((2, Ny, dNz, dNx), np.nan, dtype=torch.float64, device=gpu)
        fft.wave_to_physical(torch.from_numpy(junk).to(gpu), Pd)
        want = backward_numpy(W, dNx, dNz)
        assert np.abs(Pd.cpu().numpy() - want).max() <= tol * np.abs(want).max()
        P = rng.standard_normal((2, Ny, dNz, dNx))
        Wd = torch.full(W.shape, np.nan + 0j, dtype=torch.complex128, device=gpu)
        fft.physical_to_wave(torch.from_numpy(P).to(gpu), Wd)
        want = forward_numpy(P, keep)
        got = Wd.cpu().numpy()
        assert np.abs(got - want).max() <= tol * np.abs(want).max()
        assert (got[:, ~keep] == 0).all()
