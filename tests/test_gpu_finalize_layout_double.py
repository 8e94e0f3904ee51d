"""test_gpu_finalize_layout on the double build: a complex value is four float32 words there, so one
facet's real parts lie in other facets' words, and a double can lose one half to a real part.

Tolerance: the images are FP64 transforms rounded to float32 (2^-24) or left as FP64 (an FP64
transform errs by about 2^-53 sqrt(log2 N) of the rms; 1e-12 of the peak)."""
import numpy as np
import pytest
import torch

from common import make_spec, round_to, set_options, small_obs
from bullseye_amd.binding import Binding
from bullseye_amd.library_loader import load_library

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("npix", [33, 64])
@pytest.mark.parametrize("mode,cube,facets", [("grid_single_pol", 1, 1), ("facet_duel_pol", 1, 5),
                                              ("facet_duel_pol", 3, 4), ("facet_4_cor", 2, 6)])
def test_finalize_words(mode, cube, facets, npix):
    print("case finalize words double", mode, cube, facets, npix, flush=True)
    obs = round_to(small_obs(mode, seed=2), "double")
    spec = make_spec(obs, mode, npix=npix, n_facets=facets, precision="double", cube=cube)
    lib = load_library("GPU", "double")
    set_options(lib, device_resident=1)
    b = Binding("double", obs, spec, device=torch.device("cuda:0"))
    buf = b.keep["output_buffer"]
    torch.view_as_real(buf).normal_(0.0, 1.0)
    before = buf.cpu().numpy()
    torch.cuda.synchronize()
    try:
        assert lib.initLibrary(b.byref()) == 0, lib.bullseye_last_error()
        assert lib.finalize(b.byref()) == 0, lib.bullseye_last_error()
        got = torch.view_as_real(buf).reshape(-1).cpu().numpy()
    finally:
        lib.releaseLibrary()
        set_options(lib)
    F, _, P, ny, nx = before.shape
    n, block = cube, cube * P * npix * npix   # images a facet; floats between facets' real parts
    img = np.fft.fftshift(np.fft.ifft2(np.fft.ifftshift(
        before.reshape(F, cube * P, ny, nx)[:, :n], axes=(-2, -1))), axes=(-2, -1)) * npix * npix
    peak = np.abs(img).max()
    words = before.reshape(F, cube * P, ny, nx).copy()
    words[:, :n] = img
    want = words.reshape(-1).view(np.float64)
    real = np.zeros(2 * want.size, bool)
    floats = got.view(np.float32)
    for f in range(F):
        at = slice(f * block, f * block + n * npix * npix)
        np.testing.assert_allclose(floats[at], img[f].real.reshape(-1), rtol=2.0 ** -23,
                                   atol=1e-12 * peak)
        real[at] = True
    kept = ~real.reshape(-1, 2).any(1)   # doubles without a real part in either half
    assert 0 < kept.sum() < kept.size
    np.testing.assert_allclose(got[kept], want[kept], rtol=0, atol=1e-12 * peak)
    half = real.reshape(-1, 2)
    high = half[:, 0] & ~half[:, 1]      # (little endian) the high half still holds the value
    if high.any():
        mixed = got[high].view(np.uint32).reshape(-1, 2)[:, 1]
        full = want[high].view(np.uint32).reshape(-1, 2)[:, 1]
        assert np.abs(mixed.astype(np.int64) - full.astype(np.int64)).max() <= 1
