"""A w coordinate on the boundary between two w-planes: w / wavelength rounds to the boundary, w
times the rounded reciprocal of the wavelength just above it.  The classification of the streams
and the gridders must put such a sample on the same plane, or an unchanged plan reports its own
data as wider than planned.  The tiled single-facet call, which classifies nothing, is the
reference; the bars are summation order's (test_gpu_batch, FP64)."""
import ctypes

import numpy as np
import pytest

from common import rel_err, set_options, tiny_obs, wproj_spec
from bullseye_amd.batch import BatchFacet, FacetBatch
from bullseye_amd.binding import Binding
from bullseye_amd.library_loader import (BATCH_PER_FACET, BATCH_PERSISTENT, PATH_FP64,
                                         load_library)

pytestmark = pytest.mark.gpu

HALVES = [1, 2, 3, 6, 6]


def boundary_wavelength():
    """A wavelength l for which (2.5 l) / l == 2.5 < (2.5 l) * (1 / l)."""
    for l in np.random.default_rng(1).uniform(0.19, 0.23, 1000).astype(np.float32):
        l = float(l)
        if 2.5 * l / l == 2.5 and 2.5 * l * (1.0 / l) > 2.5:
            return l
    raise AssertionError("no such wavelength")


@pytest.fixture
def session():
    l = boundary_wavelength()
    rng = np.random.default_rng(2)
    rows = 40
    uvw = np.stack([rng.uniform(-9, 9, rows) * l, rng.uniform(-9, 9, rows) * l,
                    np.full(rows, 2.5 * l)], 1)
    obs = tiny_obs(uvw, rng.normal(size=rows) + 1j * rng.normal(size=rows), wavelength=l)
    spec, halves = wproj_spec(obs, "facet_single_pol", "double", S=6, OS=2, planes=len(HALVES),
                              halves=HALVES, npix=64)
    spec.wmax, spec.cell = 4.0, 3000.0
    spec.facet_centres = np.array([obs.phase_centre], np.float64)
    lib = load_library("GPU", "double")
    arr = (ctypes.c_uint32 * len(halves))(*halves)

    def single(flags):
        set_options(lib, compute_path=PATH_FP64, reserved=(ctypes.c_uint32 * 9)(flags))
        b = Binding("double", obs, spec)
        assert lib.initLibrary(b.byref()) == 0, lib.bullseye_last_error()
        assert lib.facet_single_pol(b.byref()) == 0, lib.bullseye_last_error()
        lib.releaseLibrary()
        return b.output[0]

    assert lib.bullseye_set_wplane_support(arr, len(halves)) == 0
    yield lib, obs, spec, halves, single
    lib.releaseLibrary()
    lib.bullseye_set_wplane_support(None, 0)
    set_options(lib)


def close(got, want):
    assert np.abs(want).max() > 0
    rms, peak = rel_err(got, want)
    assert rms <= 1e-11 and peak <= 1e-9, (rms, peak)


def test_class_kernels(session):
    print("case plane boundary, class kernels", flush=True)
    _, _, _, _, single = session
    close(single(2), single(0))


@pytest.mark.parametrize("schedule", [BATCH_PERSISTENT, BATCH_PER_FACET])
def test_batch(session, schedule):
    print("case plane boundary, batch", schedule, flush=True)
    lib, obs, spec, halves, single = session
    want = single(0)
    set_options(lib, compute_path=PATH_FP64)
    b = Binding("double", obs, spec)
    assert lib.initLibrary(b.byref()) == 0, lib.bullseye_last_error()
    batch = FacetBatch(lib, b)
    batch.kernel_set(0, spec.conv, spec.support, spec.oversample, halves, spec.wmax)
    batch.plan([BatchFacet(64, spec.cell, obs.phase_centre, 0)], schedule)
    grids, _ = batch.execute()
    close(grids[0], want)
