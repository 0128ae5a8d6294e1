"""The run walk for the cross-correlation (signed r_par, several launches of r_par rows) and
for the pair-redshift and same-half-plate cuts, on the CPU against the FP64 oracle: the
kernel's lane program under bounds checks, bars as in test_host_walk.py (xi sums cancel, so
the random geometries' bound is 1e-8 as there)."""
import pytest

import walk_cases as W
import walk_cut_cases as K
import walk_harness as H
from picca_amd.engine import params_from_globals


def run(case, share, rtol):
    p = case.pairs
    out, st = H.xi_walk_cuts(params_from_globals(case.g), case.store, p.pair_a, p.pair_b,
                             p.pair_ang, p.pair_flags, p.pair_row, p.num_rows, share)
    ref, ost = W.oracle(case)
    assert st["oob"] == 0
    W.assert_matches(out, st["edge"], st["overflow"], ref, ost, rtol)
    return st, ost


@pytest.mark.parametrize("option", ["cross", "plate", "z", "cross+z", "cross+plate", "plate+z"])
@pytest.mark.parametrize("layout,seed", [("lattice", 0), ("irregular", 1)]
                         + [("random", s) for s in range(8)])
def test_against_oracle(layout, option, seed):
    case, share = K.cut_case(layout, option, seed)
    st, ost = run(case, share, 1e-8 if layout == "random" else 1e-9)
    if layout == "lattice":
        assert ost[1] > 1000 and st["walk_tasks"] > 0


def test_row_shares():
    """One launch where the whole histogram fits, else equal shares within the rows that fit."""
    case, _ = K.cut_case("lattice", "cross")
    whole, _ = run(case, case.g.num_bins_r_par, 1e-9)
    parts, _ = run(case, 1, 1e-9)
    assert whole["runs"] < parts["runs"]
