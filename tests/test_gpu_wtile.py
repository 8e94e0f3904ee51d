"""The tiled w-projection gridder (csrc/wtile.hip) against the oracle
(cpu_algorithm/convolution_policies.h:231-289), where its bins, work items and passes break: every
width 1..63 at once, grids that end inside a tile, bins of more than one work item, cube slices,
passes of few records over facets and rows, and the class kernels on the same call.

Bars as in test_gpu_wproj: FP64 sums of FP64 products round at 2^-53 per term; FP32 products at
2^-24 each, added in FP64, against the peak of the grid."""
import ctypes

import numpy as np
import pytest

from common import MODES_PSF, rel_err, round_to, set_options, small_obs, wproj_spec
from bullseye_amd.binding import Binding
from bullseye_amd.library_loader import PATH_FP32_KAHAN, PATH_FP64, load_library
from oracle import oracle

pytestmark = pytest.mark.gpu

CASES = [("double", PATH_FP64), ("mixed", PATH_FP32_KAHAN), ("single", PATH_FP32_KAHAN)]
EVERY = list(range(32))


def reserved(flags=0, records=0):
    return (ctypes.c_uint32 * 9)(flags, records)


def grid(precision, path, mode, halves, S, npix, res, cell=None, cube=1, seed=5):
    obs = round_to(small_obs(mode, seed=seed), precision)
    spec, halves = wproj_spec(obs, mode, precision, S=S, OS=2, planes=len(halves),
                              halves=halves, npix=npix)
    if cell:
        spec.cell = cell
    if cube > 1:
        spec.cube = cube
        spec.channel_grid_index = np.arange(obs.n_chan, dtype=np.uint64) % cube
    psf = mode in MODES_PSF
    ref = Binding("double", obs, spec, with_psf=psf)
    want_norm = oracle.run(ref, mode)
    want = ref.psf if psf else ref.output
    lib = load_library("GPU", precision)
    set_options(lib, compute_path=path, reserved=res)
    arr = (ctypes.c_uint32 * len(halves))(*halves)
    assert lib.bullseye_set_wplane_support(arr, len(halves)) == 0
    b = Binding(precision, obs, spec, with_psf=psf)
    try:
        assert lib.initLibrary(b.byref()) == 0, lib.bullseye_last_error()
        assert getattr(lib, mode)(b.byref()) == 0, lib.bullseye_last_error()
        norm = np.ctypeslib.as_array(
            ctypes.cast(b.params.normalization_terms, ctypes.POINTER(ctypes.c_double)),
            (len(want_norm),)).copy()
        if not psf:
            assert lib.normalize(b.byref()) == 0
    finally:
        lib.releaseLibrary()
        lib.bullseye_set_wplane_support(None, 0)
    return rel_err(b.psf if psf else b.output, want), norm, want_norm, want


def check(precision, path, mode, halves, S, npix, res, **kw):
    (rms, peak), norm, want_norm, want = grid(precision, path, mode, halves, S, npix, res, **kw)
    print("rms %.3e peak %.3e" % (rms, peak))
    assert np.abs(want).max() > 0
    tol = (1e-11, 1e-9) if path == PATH_FP64 else (1e-6, 2e-5)
    assert rms <= tol[0] and peak <= tol[1], (rms, peak)
    if mode not in MODES_PSF:
        np.testing.assert_allclose(norm, want_norm, rtol=1e-9)


@pytest.mark.parametrize("flags,records", [(0, 0), (0, 700), (2, 0)])
@pytest.mark.parametrize("precision,path", CASES)
@pytest.mark.parametrize("mode", ["grid_single_pol", "facet_duel_pol", "facet_4_cor_corrections",
                                  "facet_sampling_function"])
def test_every_width(mode, precision, path, flags, records):
    print("case wtile widths", mode, precision, path, flags, records, flush=True)
    check(precision, path, mode, EVERY, 31, 231, reserved(flags, records))


# footprint origins at the first and last cells of a tile: grids of one tile, one cell more, and
# 3 tiles less one cell; compact tracks put more samples into a bin than a work item holds
@pytest.mark.parametrize("npix", [33, 34, 98])
@pytest.mark.parametrize("cell", [4.0, 30.0])
@pytest.mark.parametrize("halves", [[0] * 4, [1, 2, 3, 4], [7, 8, 11, 12]])
def test_tile_edges(npix, cell, halves):
    if 2 * max(halves) + 3 >= npix:
        pytest.skip("support does not fit the grid")
    print("case wtile edges", npix, cell, halves, flush=True)
    check("mixed", PATH_FP32_KAHAN, "grid_single_pol", halves, max(max(halves), 1), npix,
          reserved(), cell=cell)


@pytest.mark.parametrize("records", [0, 300])
def test_cube_slices(records):
    print("case wtile cube", records, flush=True)
    check("double", PATH_FP64, "facet_duel_pol", [1, 2, 3, 5, 8], 8, 100, reserved(0, records),
          cube=3)
