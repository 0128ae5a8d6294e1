"""Forests with negative dist_m (whose r_trans bins lie below 0): the correlation leaves those
pairs out and counts them as overflow pairs, as the oracle does, and the distortion matrix refuses
them with IndexError, as picca's own array access does, whichever kernels the other pairs take."""
import numpy as np
import pytest

import walk_cases as W
import walk_cut_cases as K
from oracle import cf_oracle as O
from picca_amd import _native, batch
from picca_amd.engine import get_engine, params_from_globals
from test_gpu_dmat_band import dmat_store

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("option", ["", "cross", "plate", "z", "cross+z"])
def test_correlation_counts_them(option):
    case, _ = K.cut_case("random", option, seed=3)
    case.g.num_bins_r_par, case.g.num_bins_r_trans = (6 if "cross" in option else 3), 4
    case.g.r_trans_max = 10.0
    case.pairs.pair_ang[:] = np.linspace(0.001, 0.003, case.pairs.num_pairs)
    for k in (0, 2):   # one forest wholly, one in part so far below 0 that no bin is left
        o, e = case.store.offsets[k:k + 2]
        case.store.dist_m[o:e if k == 0 else (o + e) // 2] -= 1e6
    ref, ost = W.oracle(case)
    assert ost[2] > 0 and ost[0] > 0
    for schedule in (_native.XI_SCHEDULE_RUNS, _native.XI_SCHEDULE_PAIRS):
        res = batch.run_xi(case.store, case.pairs, params_from_globals(case.g),
                           schedule=schedule)
        out = [res.weights, res.xi, res.r_par, res.r_trans, res.z, res.num_pairs]
        # (xi sums cancel: the bound of the random geometries in test_gpu_xi_cuts)
        W.assert_matches(out, res.report["edge_pairs"], res.report["overflow_pairs"], ref, ost,
                         1e-8)


@pytest.mark.parametrize("quasar", [False, True])
@pytest.mark.parametrize("shift", ["whole", "part"])
def test_distortion_matrix_refuses_them(quasar, shift):
    case = W.random_case(3)
    g, p = case.g, case.pairs
    g.num_bins_r_par = g.num_bins_r_trans = 12
    # two model bins to a data bin: a pair in the second one of r_par row 0 has a model bin and
    # no data bin
    g.num_model_bins_r_par, g.num_model_bins_r_trans = 24, 12
    g.r_par_max = g.r_trans_max = 120.0
    store = dmat_store(case.store, 0, (1,))
    if quasar:   # a quasar behind every forest's first pixels, which lie in r_par row 0
        g.x_correlation, g.r_par_min = True, -120.0
        n = store.num_forests
        last = store.offsets[1:] - 1
        both = {k: np.concatenate([getattr(store, k), getattr(store, k)[last]])
                for k in ("r_comov", "dist_m", "z", "weights", "delta", "log_lambda")}
        both.update({k: np.concatenate([getattr(store, k)] * 2)
                     for k in ("z_qso", "ra", "dec", "thingid")})
        both["offsets"] = np.concatenate([store.offsets, store.offsets[-1] + np.arange(1, n + 1)])
        both["order"] = np.concatenate([store.order, np.full(n, -1)]).astype(np.int32)
        both["weights"][store.offsets[-1]:] = 1.0
        both["r_comov"][store.offsets[-1]:] = store.r_comov[store.offsets[:-1]] + 104.0
        store = type(store)(**both)
        b = n + p.pair_a
        flags = np.full(len(b), _native.PICCA_PAIR_XCF_COUNT, np.uint8)
    else:
        b, flags = p.pair_a, np.zeros(len(p.pair_a), np.uint8)
    ang = np.full(len(b), 0.01)
    eng = get_engine(0)
    eng.set_forests(store)
    params = params_from_globals(g)
    assert eng.dmat(params, p.pair_a, b, ang, flags)[6][0] > 0
    store.dist_m = store.dist_m.copy()
    o, e = store.offsets[:2]
    mine = slice(o, e) if shift == "whole" else slice(o, o + 2)
    store.dist_m[mine] = -store.dist_m[mine][::-1] - 6000.0
    if not quasar:
        with pytest.raises(IndexError):
            O.dmat_rows(O.params_from_module(g), store, p.pair_a, b, ang, flags)
    eng.set_forests(store)
    with pytest.raises(IndexError):
        eng.dmat(params, p.pair_a, b, ang, flags)
