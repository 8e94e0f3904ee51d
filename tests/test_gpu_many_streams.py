"""AA gridding calls of more streams than one launch of the gridding kernels holds (fewer than
2^32 work items, one wavefront a stream for four correlations at W = 7): many baselines and
facets, few of them with samples, against the oracle.  Bars as in test_gpu_parity for the
compensated FP32 path."""
import numpy as np
import pytest

from common import make_spec, rel_err, round_to, run_library, set_options, small_obs
from bullseye_amd.binding import Binding
from bullseye_amd.library_loader import PATH_FP32_KAHAN, load_library
from oracle import oracle

pytestmark = pytest.mark.gpu

ANTENNAS = 2000   # 2.0 M baselines


@pytest.mark.parametrize("mode,facets,support", [
    ("facet_4_cor", 40, 3), ("facet_duel_pol", 150, 3),
    ("facet_single_pol", 80, 7)])   # W = 15: the generic kernel
def test_many_streams(mode, facets, support):
    print("case many streams", mode, facets, support, flush=True)
    obs = round_to(small_obs(mode, n_ant=6, n_time=4, n_chan=3), "mixed")
    # the tracks of the last six antennas: the last streams hold samples too
    obs.ant1 = obs.ant1 + np.uint32(ANTENNAS - 6)
    obs.ant2 = obs.ant2 + np.uint32(ANTENNAS - 6)
    obs.ant1[::3] -= np.uint32(ANTENNAS - 6)
    obs.ant2[::3] -= np.uint32(ANTENNAS - 6)
    obs.n_ant = ANTENNAS
    spec = make_spec(obs, mode, precision="mixed", npix=64, n_facets=facets, support=support)
    ref = Binding("double", obs, spec)
    oracle.run(ref, mode)
    lib = load_library("GPU", "mixed")
    set_options(lib, compute_path=PATH_FP32_KAHAN)
    b = Binding("mixed", obs, spec)
    run_library(lib, b, mode)
    rms, peak = rel_err(b.output, ref.output)
    print("rms %.3e peak %.3e" % (rms, peak))
    assert np.abs(ref.output).max() > 0
    assert rms <= 1e-6 and peak <= 2e-5, (rms, peak)
