"""Footprint origins on both sides of a tile's edge (csrc/wtile.hip: tiles of 33 x 33 origins).  An
origin reaches at most npix - S - half - 4, so the grids are sized for a largest origin of 32 (the
last of the first tile) and 33 (the first of the next); the tracks reach it, which is checked on
the host.  Bars as in test_gpu_wtile."""
import numpy as np
import pytest

from common import round_to, small_obs, u_scale
from bullseye_amd.library_loader import PATH_FP32_KAHAN
from test_gpu_wtile import check, reserved

pytestmark = pytest.mark.gpu

TILE = 33


@pytest.mark.parametrize("past", [0, 1])
@pytest.mark.parametrize("half,S", [(0, 1), (1, 1), (3, 3), (2, 5)])
def test_last_origin(half, S, past):
    print("case wtile last origin", half, S, past, flush=True)
    npix = TILE - 1 + past + S + half + 4
    cell = 60.0
    obs = round_to(small_obs("grid_single_pol", seed=5), "mixed")
    # origins of the call's samples, as convolution_policies.h:231-289 places them
    seen = set()
    for comp, sign in ((0, 1.0), (1, -1.0)):
        u = obs.uvw[:, comp:comp + 1] / obs.wavelengths[0][None, :] * u_scale(npix, cell) * sign
        u = np.where(obs.uvw[:, 2:3] < 0, -u, u)
        d = np.rint(u + (npix // 2 - S)).astype(int)
        x0 = d[(d >= 0) & (d < npix - 2 * S - 3)] + S - half
        assert x0.max() == TILE - 1 + past, x0.max()
        seen |= set(np.unique(x0 // TILE))
    assert seen == ({0, 1} if past else {0})
    check("mixed", PATH_FP32_KAHAN, "grid_single_pol", [half] * 3, S, npix, reserved(), cell=cell)
