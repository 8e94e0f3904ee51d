"""The one-stream-per-wavefront kernel (4 correlations, FP32 paths, half support 3) against the
oracle where its steps and runs break: streams of fewer samples than a wavefront, exactly one step,
one more, runs longer than a run may be, spans that begin and end inside a quad (heavy flagging),
fast tracks that move every sample, several grid slices.

Bars as in test_gpu_parity: FP32 products and compensated sums 1e-6 rms of the peak, plain FP32 sums
2e-6."""
import ctypes

import numpy as np
import pytest

from common import make_spec, rel_err, round_to, run_library, set_options, small_obs
from bullseye_amd.binding import Binding
from bullseye_amd.library_loader import PATH_FP32, PATH_FP32_KAHAN, load_library
from oracle import oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("path", [PATH_FP32_KAHAN, PATH_FP32])
@pytest.mark.parametrize("mode", ["grid_4_cor", "facet_4_cor", "facet_4_cor_corrections"])
@pytest.mark.parametrize("n_time,n_chan,flags,cell,cube", [
    (1, 1, 0.0, 20.0, 1), (1, 3, 0.0, 20.0, 1), (3, 21, 0.5, 20.0, 1), (2, 32, 0.0, 2.0, 1),
    (5, 13, 0.7, 2.0, 1), (40, 7, 0.2, 40.0, 1), (9, 48, 0.05, 5.0, 3)])
def test_wave4(mode, path, n_time, n_chan, flags, cell, cube):
    print("case wave4", mode, path, n_time, n_chan, flags, cell, cube, flush=True)
    obs = round_to(small_obs(mode, seed=11, n_ant=7, n_time=n_time, n_chan=n_chan,
                             flag_fraction=flags), "mixed")
    spec = make_spec(obs, mode, npix=150, cell=cell, precision="mixed", cube=cube)
    ref = Binding("double", obs, spec)
    want_norm = oracle.run(ref, mode)
    lib = load_library("GPU", "mixed")
    # one segment per baseline, every channel of a slice together
    set_options(lib, compute_path=path, rows_per_stream=n_time, channels_per_stream=n_chan)
    b = Binding("mixed", obs, spec)
    norm = run_library(lib, b, mode)
    rms, peak = rel_err(b.output, ref.output)
    print("rms %.3e peak %.3e" % (rms, peak))
    assert np.abs(ref.output).max() > 0
    tol = 1e-6 if path == PATH_FP32_KAHAN else 2e-6
    assert rms <= tol and peak <= 20 * tol, (rms, peak)
    np.testing.assert_allclose(norm, want_norm, rtol=1e-9)
