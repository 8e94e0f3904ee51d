"""The kernel choices of bullseye_options::reserved[0].

One stream (a baseline's rows, all channels together) adds into every grid cell in one order, so a
kernel's grid is the same bits every time and tells which kernel ran."""
import ctypes

import numpy as np
import pytest

from common import make_spec, round_to, set_options, tiny_obs
from bullseye_amd.binding import Binding
from bullseye_amd.library_loader import PATH_FP32, load_library

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
