"""The width-specialised AA gridder of one and two correlations (several streams a wavefront)
against the oracle where its steps, quads and runs break: steps of a number of lanes that is no
multiple of four, streams of less than a quad and of less than a step, heavy flagging, fast tracks
that move every sample, several grid slices, every width and path; and the walk order, measured
by a wavefront a baseline, against its definition.

Bars as in test_gpu_parity: FP32 products and compensated sums 1e-6 rms of the peak, plain FP32 sums
2e-6, FP64 sums of FP32 data 1e-7."""
import ctypes

import numpy as np
import pytest

from common import make_spec, rel_err, round_to, run_library, set_options, small_obs
from bullseye_amd.binding import Binding
from bullseye_amd.library_loader import (PATH_FP32, PATH_FP32_KAHAN, PATH_FP64, bullseye_stats,
                                         load_library)
from oracle import oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("path", [PATH_FP32_KAHAN, PATH_FP32, PATH_FP64])
@pytest.mark.parametrize("support", [1, 2, 3, 4, 5])
@pytest.mark.parametrize("mode,n_time,n_chan,flags,cell,cube", [
    ("grid_duel_pol", 1, 3, 0.0, 20.0, 1), ("facet_duel_pol", 9, 13, 0.5, 2.0, 1),
    ("facet_duel_pol", 40, 7, 0.1, 40.0, 3), ("facet_single_pol", 5, 21, 0.6, 5.0, 1)])
def test_runs(mode, path, support, n_time, n_chan, flags, cell, cube):
    print("case runs", mode, path, support, n_time, n_chan, flags, cell, cube, flush=True)
    obs = round_to(small_obs(mode, seed=17, n_ant=7, n_time=n_time, n_chan=n_chan,
                             flag_fraction=flags), "mixed")
    spec = make_spec(obs, mode, npix=150, cell=cell, support=support, precision="mixed",
                     cube=cube)
    ref = Binding("double", obs, spec)
    want_norm = oracle.run(ref, mode)
    lib = load_library("GPU", "mixed")
    set_options(lib, compute_path=path, rows_per_stream=n_time, channels_per_stream=n_chan)
    b = Binding("mixed", obs, spec)
    norm = run_library(lib, b, mode)
    rms, peak = rel_err(b.output, ref.output)
    print("rms %.3e peak %.3e" % (rms, peak))
    assert np.abs(ref.output).max() > 0
    tol = {PATH_FP32_KAHAN: 1e-6, PATH_FP32: 2e-6, PATH_FP64: 1e-7}[path]
    assert rms <= tol and peak <= 20 * tol, (rms, peak)
    np.testing.assert_allclose(norm, want_norm, rtol=1e-9)


@pytest.mark.parametrize("n_time,n_chan,f_hi", [(1, 4, 1.42e9), (2, 5, 1.42e9), (33, 2, 1.42e9),
                                                (34, 64, 1.401e9), (70, 3, 1.9e9)])
def test_walk_order(n_time, n_chan, f_hi):
    print("case walk order", n_time, n_chan, f_hi, flush=True)
    mode = "grid_single_pol"
    obs = round_to(small_obs(mode, seed=5, n_ant=6, n_time=n_time, n_chan=n_chan, f_hi=f_hi),
                   "mixed")
    lib = load_library("GPU", "mixed")
    set_options(lib, compute_path=PATH_FP32_KAHAN)
    b = Binding("mixed", obs, make_spec(obs, mode, npix=150, precision="mixed"))
    run_library(lib, b, mode)
    st = bullseye_stats()
    assert lib.bullseye_get_stats(ctypes.byref(st)) == 0
    cm = (n_chan - 1) // 2
    rl, rl2 = 1.0 / obs.wavelengths.ravel()[cm:cm + 2]
    time_steps, chan_steps = [], []
    for key in set(zip(obs.ant1, obs.ant2)):
        rows = [r for r in range(obs.uvw.shape[0]) if (obs.ant1[r], obs.ant2[r]) == key][:33]
        uv = obs.uvw[rows, :2]
        time_steps += list(np.abs(np.diff(uv * rl, axis=0)).sum(axis=1))
        chan_steps += list(np.abs(uv).sum(axis=1) * abs(rl2 - rl))
    want = bool(time_steps) and np.mean(time_steps) < np.mean(chan_steps)
    assert bool(st.time_inner) == bool(want)
