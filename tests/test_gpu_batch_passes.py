"""Batches whose records do not fit one pass of the tiled gridder (csrc/batch.hip, plan_tiles), with
the records per pass bounded by the options: several groups of facets, one facet's rows in several
ranges with a shorter last one, the passes taking turns in one workspace inside the captured graph,
visibilities and sampling functions, cube slices.  Each facet against its single-facet call; bars
as in test_gpu_batch."""
import ctypes

import numpy as np
import pytest

from common import round_to, set_options, small_obs
from bullseye_amd.library_loader import (BATCH_PERSISTENT, BATCH_PERSISTENT_GRAPH,
                                         PATH_FP32_KAHAN, PATH_FP64, load_library)
from test_gpu_batch import (FACETS, check_close, facet_list, kernel_specs, open_session,
                            single_facet, to_np)

pytestmark = pytest.mark.gpu

ROWS, CHANNELS = 12 * 11 // 2 * 30, 8   # 1980 rows of 8 channels: 15840 records a facet


# records a pass: two facets of all rows; one; 5 ranges of 500 rows, the last of 480; 28 of 71, the
# last of 63; one row
@pytest.mark.parametrize("records", [2 * ROWS * CHANNELS + 5, ROWS * CHANNELS, 500 * CHANNELS + 3,
                                     71 * CHANNELS, 1])
@pytest.mark.parametrize("mode,cube,precision,path", [
    ("facet_single_pol", 1, "double", PATH_FP64), ("facet_duel_pol", 3, "mixed", PATH_FP32_KAHAN)])
def test_passes_match_single_facet_calls(records, mode, cube, precision, path):
    print("case batch passes", records, mode, cube, precision, flush=True)
    facets_used = FACETS if records > 1 else FACETS[:3:2]   # a launch set per row: two facets
    obs = round_to(small_obs("facet_4_cor", seed=33, n_ant=12, n_time=30, n_chan=CHANNELS),
                   precision)
    assert obs.rows == ROWS
    kspecs = kernel_specs(obs, precision)
    facets = facet_list(obs, precision, facets=facets_used, seed=28)
    lib = load_library("GPU", precision)
    set_options(lib, compute_path=path)
    want = [single_facet(lib, precision, obs, *kspecs[f.kernel_set], f, mode, cube)
            for f in facets]
    lib, s = open_session(precision, path, obs, kspecs, mode=mode, cube=cube)
    try:
        set_options(lib, device_resident=1, compute_path=path,
                    reserved=(ctypes.c_uint32 * 9)(0, records))
        eager = s.run(facets, BATCH_PERSISTENT)
        runs = [eager]
        if records > 1:
            runs += s.run(facets, BATCH_PERSISTENT_GRAPH, repeats=2)
    finally:
        s.close()
    for grids, norms, taps in runs:
        assert taps == sum(w[2] for w in want)
        for i, f in enumerate(facets):
            check_close(to_np(grids[i]), want[i][0], path)
            if not f.sampling_function:
                np.testing.assert_allclose(norms[i].reshape(-1), want[i][1], rtol=1e-9)
