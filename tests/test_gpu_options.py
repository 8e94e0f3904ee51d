"""The kernel choices of bullseye_options::reserved[0]: the generic AA kernel, the w-projection
class kernels.

One stream (a baseline's rows, all channels together) adds into every grid cell in one order, so a
kernel's grid is the same bits every time and tells which kernel ran."""
import ctypes

import numpy as np
import pytest

from common import make_spec, round_to, set_options, tiny_obs
from bullseye_amd.batch import BatchFacet, FacetBatch
from bullseye_amd.binding import Binding
from bullseye_amd.library_loader import PATH_FP32, PATH_FP64, load_library
from test_gpu_batch import facet_list, kernel_specs, observation, open_session
from test_gpu_workspace import FIXED, MB, Context, close, free_bytes

pytestmark = pytest.mark.gpu


def test_any_nonzero_value_forces_the_generic_aa_kernel():
    print("case options generic", flush=True)
    rng = np.random.default_rng(4)
    rows = 600
    obs = tiny_obs(rng.uniform(-40, 40, (rows, 3)), rng.normal(size=rows) + 1j, wavelength=0.2,
                   ant=(np.zeros(rows), np.ones(rows)))
    obs = round_to(obs, "mixed")
    lib = load_library("GPU", "mixed")
    grids = {}
    for flags in (0, 1, 2, 4, 0x80000000):
        set_options(lib, compute_path=PATH_FP32, rows_per_stream=rows,
                    reserved=(ctypes.c_uint32 * 9)(flags))
        b = Binding("mixed", obs, make_spec(obs, "grid_single_pol", precision="mixed", npix=64,
                                            cell=300.0))
        assert lib.initLibrary(b.byref()) == 0, lib.bullseye_last_error()
        assert lib.grid_single_pol(b.byref()) == 0, lib.bullseye_last_error()
        lib.releaseLibrary()
        grids[flags] = b.output.copy()
    set_options(lib)
    assert np.abs(grids[1]).max() > 0
    assert not np.array_equal(grids[0], grids[1])   # the two kernels round differently
    for flags in (2, 4, 0x80000000):
        np.testing.assert_array_equal(grids[flags], grids[1])


def test_batch_on_the_class_kernels():
    """At default tiles: the tiled plan holds its counters (test_gpu_workspace), the class plan does
    not, and their grids agree."""
    print("case options batch classes", flush=True)
    c = Context()
    try:
        batch = FacetBatch(c.lib, c.b)
        got, held = [], []
        for flags in (2, 0):
            batch.kernel_set(0, c.spec.conv, 31, 1, c.halves, c.spec.wmax)
            set_options(c.lib, compute_path=PATH_FP64, reserved=(ctypes.c_uint32 * 9)(flags))
            batch.plan([BatchFacet(4096, c.spec.cell, c.obs.phase_centre, 0)])
            grids, _ = batch.execute()
            got.append(grids[0].copy())
            before = free_bytes()
            batch.release()
            held.append(free_bytes() - before)
        assert held[1] - held[0] >= FIXED - 32 * MB
        close(got[0], got[1])
    finally:
        c.close()


def test_autotune_of_the_class_kernels():
    """Forced, the autotuner compares class kernels only, and its baseline is theirs: the best
    launches of every class are no slower than the default ones."""
    print("case options autotune", flush=True)
    obs = observation("double", seed=15)
    kspecs = kernel_specs(obs, "double")
    lib, s = open_session("double", PATH_FP64, obs, kspecs)
    try:
        set_options(lib, device_resident=1, compute_path=PATH_FP64,
                    reserved=(ctypes.c_uint32 * 9)(2))
        t = s.batch.autotune(facet_list(obs, "double", seed=10))
        s.batch.set_tuning()
    finally:
        s.close()
    assert t["tuned"] == 1 and 0 < t["tuned_ms"] <= t["default_ms"] * 1.5 + 0.05
    assert any(t["shape"].values())   # a tiled choice has none
