"""Forests whose weights or deltas are not level: with signed r_par and with cuts their tasks take
the pair loop, the others of one call the run walk, and every bin is within 1e-12 of 80-bit sums
(bars and inputs of test_host_walk_precision, which runs the same lane program on the CPU)."""
import numpy as np
import pytest

from picca_amd import _native, batch
from picca_amd.engine import params_from_globals
from test_host_walk_precision import extended, survey

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("option", ["cross", "plate"])
@pytest.mark.parametrize("what,walked", [("none", "all"), ("weights", "none"),
                                         ("deltas", "none"), ("half", "half")])
def test_unlevel_forests(option, what, walked):
    case = survey(option)
    s, g = case.store, case.g
    for k in range(s.num_forests):
        if what == "weights" or (what == "half" and k % 2):
            s.weights[s.offsets[k] + 40] = 1.25e8
        elif what == "deltas":
            s.delta[s.offsets[k] + 40] = 1e8
    res = batch.run_xi(s, case.pairs, params_from_globals(g),
                       schedule=_native.XI_SCHEDULE_RUNS)
    rep = res.report
    share = rep["walk_tasks"] / (rep["tasks"] - rep["empty_tasks"])
    assert {"all": share > 0.9, "none": share == 0, "half": 0.2 < share < 0.8}[walked], share
    ref, width = extended(case)
    out = [res.weights, res.xi, res.r_par, res.r_trans, res.z]
    mask = ref[0] > 0
    scale = [ref[0], ref[5], ref[0] * width + np.abs(ref[2]), ref[3], ref[4]]
    for k in range(5):
        assert np.max(np.abs(out[k][0] - ref[k])[mask] / scale[k][mask]) < 1e-12, k
