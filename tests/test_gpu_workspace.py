"""Device memory of the tiled w-projection gridder: a call or a batch plan that the allowed (or
available) workspace cannot hold runs on the class kernels, and what the context keeps between
calls is given back when another allocation needs it.

A 4096^2 grid of 32 widths takes 15625 tiles x 32 x 16 counters of 4 bytes, and as many first places:
64 MB whatever the records.  Bars between the two kernels as in test_gpu_wproj for FP64."""
import ctypes

import numpy as np
import pytest
import torch

from common import rel_err, round_to, set_options, small_obs, wproj_spec
from bullseye_amd.batch import BatchFacet, FacetBatch
from bullseye_amd.binding import Binding
from bullseye_amd.library_loader import PATH_FP64, load_library

pytestmark = pytest.mark.gpu

MB = 1 << 20
FIXED = 2 * 15625 * 32 * 16 * 4   # bytes of counters and first places


def free_bytes():
    torch.cuda.synchronize()
    return torch.cuda.mem_get_info()[0]


class Context:
    def __init__(self):
        self.obs = round_to(small_obs("facet_single_pol", seed=3), "double")
        self.spec, self.halves = wproj_spec(self.obs, "facet_single_pol", "double", S=31, OS=1,
                                            planes=32, halves=list(range(32)), npix=4096)
        self.spec.facet_centres = np.array([self.obs.phase_centre], np.float64)
        self.lib = load_library("GPU", "double")
        self.options()
        arr = (ctypes.c_uint32 * 32)(*self.halves)
        assert self.lib.bullseye_set_wplane_support(arr, 32) == 0
        self.b = Binding("double", self.obs, self.spec)
        assert self.lib.initLibrary(self.b.byref()) == 0, self.lib.bullseye_last_error()

    def options(self, mib=0):
        set_options(self.lib, compute_path=PATH_FP64, reserved=(ctypes.c_uint32 * 9)(0, 0, mib))

    def grid(self, mib=0):
        self.options(mib)
        assert self.lib.bullseye_reset_grids() == 0
        assert self.lib.facet_single_pol(self.b.byref()) == 0, self.lib.bullseye_last_error()
        return self.b.output[0].copy()

    def close(self):
        self.lib.releaseLibrary()
        self.lib.bullseye_set_wplane_support(None, 0)
        set_options(self.lib)


@pytest.fixture
def context():
    c = Context()
    yield c
    c.close()


def close(got, want):
    assert np.abs(want).max() > 0
    rms, peak = rel_err(got, want)
    assert rms <= 1e-11 and peak <= 1e-9, (rms, peak)


def test_call_beyond_the_workspace(context):
    print("case workspace call", flush=True)
    short = context.grid(mib=16)    # the first call stages its arrays as well
    held = free_bytes()
    tiled = context.grid()
    assert held - free_bytes() >= FIXED
    close(short, tiled)
    context.grid(mib=16)            # a bound below what is held gives it back
    assert held - free_bytes() <= 8 * MB


def test_batch_beyond_the_workspace(context):
    print("case workspace batch", flush=True)
    facets = [BatchFacet(4096, context.spec.cell, context.obs.phase_centre, 0)]
    batch = FacetBatch(context.lib, context.b)
    batch.kernel_set(0, context.spec.conv, 31, 1, context.halves, context.spec.wmax)
    got, held = [], []
    for mib in (16, 0):
        context.options(mib)
        batch.plan(facets)
        grids, _ = batch.execute()
        got.append(grids[0].copy())
        before = free_bytes()
        batch.release()
        held.append(free_bytes() - before)
        batch.kernel_set(0, context.spec.conv, 31, 1, context.halves, context.spec.wmax)
    assert held[1] - held[0] >= FIXED - 32 * MB   # the class kernels' lists take some too
    close(got[0], got[1])


def test_kept_memory_is_given_back(context):
    print("case workspace given back", flush=True)
    context.grid(mib=16)
    held = free_bytes()
    want = context.grid()
    assert held - free_bytes() >= FIXED
    # a plan whose grids exceed any GPU (20 of 45000^2 cells of 16 bytes: 648 GB) is refused, and
    # asking for them has taken what the calls keep
    batch = FacetBatch(context.lib, context.b)
    batch.kernel_set(0, context.spec.conv, 31, 1, context.halves, context.spec.wmax)
    table = [BatchFacet(45000, context.spec.cell, context.obs.phase_centre, 0)] * 20
    refuse(batch, table)
    batch.release()
    assert held - free_bytes() <= 8 * MB
    close(context.grid(), want)


def refuse(batch, facets):
    """bullseye_batch_plan without the facets' outputs."""
    from bullseye_amd.batch import GRID_MODES
    from bullseye_amd.library_loader import bullseye_batch_facet
    table = (bullseye_batch_facet * len(facets))()
    for e, f in zip(table, facets):
        e.nx = e.ny = f.npix
        e.kernel_set, e.cell_x, e.cell_y = f.kernel_set, f.cell, f.cell
        e.ra, e.dec = f.centre
    assert batch.lib.bullseye_batch_plan(batch.binding.byref(), GRID_MODES[batch.mode], table,
                                         len(facets), 0) != 0
    assert b"memory" in batch.lib.bullseye_last_error(), batch.lib.bullseye_last_error()
