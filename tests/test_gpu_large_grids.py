"""Grids of more than 2^32 cells: clearing, publishing and normalising them takes more work items
than one axis of a launch holds.  Every facet has the same centre, so every facet's grid is the
same; a second pass after a reset gives the first one again."""
import ctypes

import numpy as np
import pytest
import torch

from common import make_spec, round_to, set_options, small_obs
from bullseye_amd.binding import Binding
from bullseye_amd.library_loader import PATH_FP32_KAHAN, load_library

pytestmark = pytest.mark.gpu

FACETS, NPIX = 260, 4096   # 4.36e9 cells, 70 GB of grid


def test_every_facet_alike():
    print("case large grids", flush=True)
    obs = round_to(small_obs("facet_single_pol", n_ant=6, n_time=5), "mixed")
    spec = make_spec(obs, "facet_single_pol", precision="mixed", npix=64, cell=2.0,
                     n_facets=FACETS)
    spec.facet_centres = np.array([obs.phase_centre] * FACETS)
    out = torch.zeros((FACETS, NPIX, NPIX), dtype=torch.complex64, device="cuda:0")
    b = Binding("mixed", obs, spec, device=torch.device("cuda:0"))
    b.params.nx = b.params.ny = NPIX
    b.params.output_buffer = out.data_ptr()
    torch.cuda.synchronize()
    lib = load_library("GPU", "mixed")
    set_options(lib, compute_path=PATH_FP32_KAHAN, device_resident=1)
    assert lib.initLibrary(b.byref()) == 0, lib.bullseye_last_error()
    try:
        for _ in range(2):
            assert lib.bullseye_reset_grids() == 0, lib.bullseye_last_error()
            out.fill_(7.0)   # what is not published shows
            torch.cuda.synchronize()
            assert lib.facet_single_pol(b.byref()) == 0, lib.bullseye_last_error()
            assert lib.normalize(b.byref()) == 0, lib.bullseye_last_error()
            first = out[0].cpu().numpy()
            assert np.abs(first).max() > 0
            peak = np.abs(first).max()
            for f in (127, 128, 254, 255, 256, FACETS - 1):
                # one sample's place in the order of the atomics: test_gpu_parity's bars
                assert np.abs(out[f].cpu().numpy() - first).max() <= 2e-5 * peak, f
    finally:
        lib.releaseLibrary()
        set_options(lib)
        del out, b
        torch.cuda.empty_cache()
