"""The degridding kernels against the oracle's adjoint where their shapes break: every compiled AA
width and the wavefront kernel beyond them (and where the kernel table is too large for LDS),
w-kernels from one tap to 63 x 63, sample counts around a wavefront, mostly flagged samples.  Bars
as in test_gpu_degrid."""
import numpy as np
import pytest

from common import make_spec, rel_err, round_to, small_obs, wproj_spec
from bullseye_amd.binding import Binding
from bullseye_amd.library_loader import PATH_FP32_KAHAN, PATH_FP64
from oracle import oracle
from test_gpu_degrid import degrid, open_lib, tolerance

pytestmark = pytest.mark.gpu


def check(obs, spec, halves, mode, precision, path):
    ref = Binding("double", obs, spec)
    rng = np.random.default_rng(5)
    model = (rng.normal(size=ref.output.shape) + 1j * rng.normal(size=ref.output.shape))
    model = model.astype(np.complex64).astype(np.complex128)
    want = oracle.degrid(ref, mode, model)
    lib = open_lib(precision, path, halves)
    b = Binding(precision, obs, spec)
    try:
        assert lib.initLibrary(b.byref()) == 0, lib.bullseye_last_error()
        got = degrid(lib, b, mode, model)
    finally:
        lib.releaseLibrary()
        lib.bullseye_set_wplane_support(None, 0)
    rms, peak = rel_err(got, want)
    print("rms %.3e peak %.3e" % (rms, peak))
    assert np.abs(want).max() > 0
    tol = tolerance(precision, path)
    assert rms <= tol[0] and peak <= tol[1], (rms, peak)


@pytest.mark.parametrize("precision,path", [("double", PATH_FP64), ("mixed", PATH_FP32_KAHAN)])
@pytest.mark.parametrize("mode", ["facet_single_pol", "facet_duel_pol",
                                  "facet_4_cor_corrections"])
@pytest.mark.parametrize("support,oversample", [(1, 63), (2, 63), (3, 63), (4, 63), (5, 63),
                                                (6, 63), (10, 7), (3, 1200)])
def test_aa_widths(support, oversample, mode, precision, path):
    print("case degrid width", support, oversample, mode, precision, flush=True)
    obs = round_to(small_obs(mode, seed=3, n_ant=6, n_time=5, n_chan=7, flag_fraction=0.3),
                   precision)
    spec = make_spec(obs, mode, precision=precision, npix=97, support=support,
                     oversample=oversample, n_facets=2)
    check(obs, spec, None, mode, precision, path)


@pytest.mark.parametrize("precision,path", [("double", PATH_FP64), ("mixed", PATH_FP32_KAHAN)])
@pytest.mark.parametrize("mode", ["grid_single_pol", "facet_4_cor_corrections"])
@pytest.mark.parametrize("halves,n_time,n_chan,flags", [
    ([0] * 4, 1, 1, 0.0), ([1, 3, 4, 7], 3, 21, 0.8), ([31] * 3, 2, 32, 0.05),
    ([0, 10, 20, 31], 13, 5, 0.5)])
def test_wproj_shapes(halves, n_time, n_chan, flags, mode, precision, path):
    print("case degrid w", halves, n_time, n_chan, flags, mode, precision, flush=True)
    obs = round_to(small_obs(mode, seed=4, n_ant=7, n_time=n_time, n_chan=n_chan,
                             flag_fraction=flags), precision)
    spec, halves = wproj_spec(obs, mode, precision, S=max(1, max(halves)), OS=4,
                              planes=len(halves), halves=halves, npix=150)
    check(obs, spec, halves, mode, precision, path)
