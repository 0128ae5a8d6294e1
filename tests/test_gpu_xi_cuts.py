"""The specialised pair kernel for the cross-correlation and the cuts on the GPU: run walk and
pair loop against the FP64 oracle (num_pairs bit-exact, edge and overflow counts equal, sums
within 1e-9 relative, 1e-8 on the random geometries, whose xi sums cancel)."""
import pytest

import walk_cases as W
import walk_cut_cases as K
from picca_amd import _native, batch
from picca_amd.engine import params_from_globals

pytestmark = pytest.mark.gpu

SCHEDULES = (_native.XI_SCHEDULE_RUNS, _native.XI_SCHEDULE_PAIRS, _native.XI_SCHEDULE_AUTO)


def check(case, rtol):
    ref, ost = W.oracle(case)
    reports = []
    for schedule in SCHEDULES:
        res = batch.run_xi(case.store, case.pairs, params_from_globals(case.g),
                           schedule=schedule)
        out = [res.weights, res.xi, res.r_par, res.r_trans, res.z, res.num_pairs]
        rep = res.report
        W.assert_matches(out, rep["edge_pairs"], rep["overflow_pairs"], ref, ost, rtol)
        assert rep["accepted_pairs"] == ost[0]
        reports.append(rep)
    assert reports[1]["walk_tasks"] == 0
    return reports


@pytest.mark.parametrize("option", ["cross", "plate", "z", "err", "cross+z", "cross+plate",
                                    "plate+z+err", "cross+plate+z+err"])
@pytest.mark.parametrize("layout,seed", [("lattice", 0), ("irregular", 1)]
                         + [("random", s) for s in range(4)])
def test_against_oracle(layout, option, seed):
    case, _ = K.cut_case(layout, option, seed)
    check(case, 1e-8 if layout == "random" else 1e-9)


@pytest.mark.parametrize("np_par,nt,launches", [(65, 50, 1), (66, 50, 2), (120, 50, 2),
                                                (193, 50, 4), (40, 120, 2), (40, 1500, None)])
def test_row_windows(np_par, nt, launches):
    """Sizes around the number of r_par rows that LDS holds (66 of 51 columns), and one whose
    rows do not fit three to a launch (the general kernel)."""
    case, _ = K.cut_case("lattice", "cross")
    case.g.num_bins_r_par, case.g.num_bins_r_trans = np_par, nt
    runs = check(case, 1e-9)[0]
    if launches is None:
        assert runs["walk_tasks"] == 0
    else:
        assert runs["launches"] == launches and runs["walk_tasks"] > 0
