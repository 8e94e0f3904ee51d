"""Degridding calls large enough for the kernels that large calls take (csrc/degrid.hip, launch_t)
against the same rows in pieces small enough for sixteen lanes a sample, which
test_gpu_degrid_shapes pins to the oracle: one sample's visibilities depend on no other sample, so
a call and its pieces agree to the rounding of a footprint's sum, and the pieces' ends do not
show.  Each side lies within test_gpu_degrid's bars of the exact sums, the two within their sum
of each other."""
import numpy as np
import pytest

from common import make_spec, rel_err, round_to, wproj_spec
from bullseye_amd import synth
from bullseye_amd.binding import Binding
from bullseye_amd.library_loader import PATH_FP32, PATH_FP32_KAHAN, PATH_FP64
from test_gpu_degrid import degrid, open_lib, tolerance

pytestmark = pytest.mark.gpu

FP32, FP64 = ("mixed", PATH_FP32_KAHAN), ("double", PATH_FP64)


def check(obs, spec, halves, mode, precision, path, pieces):
    rng = np.random.default_rng(5)
    lib = open_lib(precision, path, halves)
    whole = Binding(precision, obs, spec)
    shape = whole.output.shape
    model = (rng.normal(size=shape) + 1j * rng.normal(size=shape)).astype(np.complex64)
    assert lib.initLibrary(whole.byref()) == 0, lib.bullseye_last_error()
    try:
        got = degrid(lib, whole, mode, model)
        edges = [obs.rows * i // pieces for i in range(pieces + 1)]
        want = np.concatenate([degrid(lib, Binding(precision, obs, spec, rows=(a, b)), mode, model)
                               for a, b in zip(edges, edges[1:])])
    finally:
        lib.releaseLibrary()
        lib.bullseye_set_wplane_support(None, 0)
    assert np.abs(want).max() > 0
    assert np.array_equal(got == 0, want == 0)
    rms, peak = rel_err(got, want)
    print("rms %.3e peak %.3e" % (rms, peak))
    tol = tolerance(precision, path)
    assert rms <= 2 * tol[0] and peak <= 2 * tol[1], (rms, peak)


def observation(mode, samples, n_chan, precision, n_ant=33, seed=7):
    nbl = n_ant * (n_ant - 1) // 2
    n_time = -(-samples // (nbl * n_chan))
    jones = 0.05 if mode == "facet_4_cor_corrections" else None
    obs = synth.simulate(n_ant=n_ant, array_size_m=1000.0, n_time=n_time, n_chan=n_chan,
                         n_corr=1 if mode == "grid_single_pol" else 4, n_src=1,
                         jones_sigma=jones, seed=seed)
    rng = np.random.default_rng(seed)
    obs.weights = rng.uniform(0.5, 2.0, obs.weights.shape).astype(np.float32)
    return round_to(obs, precision)


@pytest.mark.parametrize("mode,case,halves,samples", [
    ("grid_single_pol", FP32, [0, 1, 2, 3], 1 << 17),
    ("grid_single_pol", FP32, [0, 3, 4, 15, 31], 3 << 17),
    ("grid_single_pol", ("mixed", PATH_FP32), [4, 7], 3 << 17),
    ("grid_single_pol", FP64, [3, 8, 31], 1 << 18),
    ("facet_duel_pol", FP32, [1, 3], 1 << 17),
    ("facet_duel_pol", FP32, [3, 4, 7], 1 << 20),
    ("grid_duel_pol", FP64, [2, 9], 1 << 20),
    ("facet_4_cor_corrections", FP32, [1, 2, 3], 1 << 17),
    ("grid_4_cor", FP32, [3, 5], 1 << 21),
])
def test_wproj_large_calls(mode, case, halves, samples):
    print("case degrid route w", mode, case, halves, samples, flush=True)
    obs = observation(mode, samples, 37, case[0])
    S = max(halves)
    spec, halves = wproj_spec(obs, mode, case[0], S=S, OS=4, planes=len(halves), halves=halves,
                              npix=256)
    check(obs, spec, halves, mode, *case, pieces=2)


@pytest.mark.parametrize("case", [FP32, FP64])
@pytest.mark.parametrize("mode", ["facet_duel_pol", "facet_4_cor_corrections"])
@pytest.mark.parametrize("support", [1, 2, 3, 4, 5])
def test_aa_large_calls(support, mode, case):
    samples = 5120 * (2 if mode == "facet_duel_pol" else 4)
    print("case degrid route aa", support, mode, case, samples, flush=True)
    obs = observation(mode, samples, 7, case[0], n_ant=9)
    spec = make_spec(obs, mode, precision=case[0], npix=97, support=support, n_facets=2)
    check(obs, spec, None, mode, *case, pieces=3)
