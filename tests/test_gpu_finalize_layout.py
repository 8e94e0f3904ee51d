"""Every word that device-resident finalize leaves in the buffer: float32 images from float index
f * fstride * npix on, complex images where no real part lies, everything else untouched
(fft_and_repacking_routines.cpp:106-116), on odd and even sizes, more correlations than images, and
twice in one context (the kept FFT plan).

Tolerance: an FP32 transform of N points errs by about 2^-24 sqrt(log2 N) of the image's rms; 1e-5
of the peak covers every size here."""
import numpy as np
import pytest
import torch

from common import make_spec, round_to, set_options, small_obs
from bullseye_amd.binding import Binding
from bullseye_amd.library_loader import load_library

pytestmark = pytest.mark.gpu


def expected(before, n):
    """The buffer as float32 words, and which of them finalize writes."""
    F, cube, P, ny, nx = before.shape
    npix, fstride = ny * nx, cube * P
    words = before.astype(np.complex64).reshape(F, fstride, npix).copy()
    img = np.fft.fftshift(np.fft.ifft2(np.fft.ifftshift(
        before.reshape(F, fstride, ny, nx)[:, :n].astype(np.complex128), axes=(-2, -1))),
        axes=(-2, -1)) * npix
    words[:, :n] = img.reshape(F, n, npix)
    flat = words.reshape(-1).view(np.float32).copy()
    for f in range(F):
        o = fstride * npix * f
        flat[o:o + n * npix] = img[f].real.reshape(-1)
    return flat, np.abs(img).max()


@pytest.mark.parametrize("npix", [33, 64])
@pytest.mark.parametrize("mode,cube,facets", [("grid_single_pol", 1, 1), ("facet_duel_pol", 1, 3),
                                              ("facet_duel_pol", 3, 2), ("facet_4_cor", 2, 3)])
def test_finalize_words(mode, cube, facets, npix):
    print("case finalize words", mode, cube, facets, npix, flush=True)
    obs = round_to(small_obs(mode, seed=2), "mixed")
    spec = make_spec(obs, mode, npix=npix, n_facets=facets, precision="mixed", cube=cube)
    lib = load_library("GPU", "mixed")
    set_options(lib, device_resident=1)
    b = Binding("mixed", obs, spec, device=torch.device("cuda:0"))
    torch.cuda.synchronize()
    buf = b.keep["output_buffer"]
    try:
        assert lib.initLibrary(b.byref()) == 0, lib.bullseye_last_error()
        for seed in (1, 2):
            g = torch.Generator(device="cuda:0").manual_seed(seed)
            torch.view_as_real(buf).normal_(0.0, 1.0, generator=g)
            want, peak = expected(buf.cpu().numpy(), cube)
            torch.cuda.synchronize()
            assert lib.finalize(b.byref()) == 0, lib.bullseye_last_error()
            got = torch.view_as_real(buf).reshape(-1).cpu().numpy()
            np.testing.assert_allclose(got, want, rtol=0, atol=1e-5 * peak)
    finally:
        lib.releaseLibrary()
        set_options(lib)
