"""Device memory of the distortion matrix from prefix sums: what a call holds follows its own pair
list and not the store, a workspace that is too small is used in several batches, and pairs whose
prefix sums do not fit take the general kernels, with one result (FP64 sums in another order:
1e-9, or 1e-12 of the largest entry)."""
import numpy as np
import pytest
import torch

import walk_cases as W
from picca_amd import _native, batch, synth
from picca_amd.constants import Cosmo
from picca_amd.engine import Engine, get_engine, params_from_globals
from picca_amd.utils import compute_ang_max
from test_gpu_dmat import assert_outputs_close, make_globals
from test_gpu_dmat_band import dmat_store, quasar_store, with_model

pytestmark = pytest.mark.gpu


def test_memory_follows_the_pair_list():
    s = synth.make_survey("survey_100k", seed=0, scale=0.02)   # 2000 forests, 1.3e6 pixels
    store = s.store
    ang_max = compute_ang_max(Cosmo(0.315, verbose=False), 60.0, s.z_min)
    p = batch.xi_pairs(store, s.healpix, ang_max)
    few = slice(0, 8)
    args = (p.pair_a[few], p.pair_b[few], p.pair_ang[few], p.pair_flags[few])
    eng = Engine()
    try:
        eng.set_forests(store)
        params = params_from_globals(make_globals())
        free = torch.cuda.mem_get_info(0)[0]
        eng.dmat(params, *args)
        held = free - torch.cuda.mem_get_info(0)[0]
        assert eng.dmat_routes()["sums"] > 0
    finally:
        eng.close()
    # a redshift-evolution factor per pixel of the store, and a few MB (2 MB to an allocation);
    # prefix sums and tables of the whole store would be 72 bytes a pixel, 90 MB
    assert held < 8 * len(store.z) + (48 << 20), held


@pytest.fixture
def engine_with_limits():
    eng = get_engine(0)
    yield eng
    eng.set_dmat_workspace()


def inputs(kind):
    case = W.random_case(3)
    g = case.g
    g.num_bins_r_par, g.num_bins_r_trans = 24, 20
    g.r_par_max = g.r_trans_max = 150.0
    case.pairs.pair_ang[:] = np.linspace(0.004, 0.03, case.pairs.num_pairs)
    with_model(case, 2, 1)
    if kind == "quasars":
        store, args = quasar_store(case, 0, (0, 1))
        g.x_correlation, g.r_par_min = True, -150.0
        return g, store, args
    if kind == "roles":
        g.alpha2 = 1.5
    p = case.pairs
    return g, dmat_store(case.store, 0, (0, 1)), (p.pair_a, p.pair_b, p.pair_ang,
                                                  np.zeros(p.num_pairs, np.uint8))


@pytest.mark.parametrize("kind", ["forests", "roles", "quasars"])
def test_batches_and_the_general_kernels_agree(engine_with_limits, kind):
    eng = engine_with_limits
    g, store, args = inputs(kind)
    params = params_from_globals(g)
    eng.set_forests(store)
    whole = eng.dmat(params, *args)
    routes = eng.dmat_routes()
    assert whole[6][0] > 0 and routes["sums"] > 4
    assert eng.dmat_report()["batches"] == 1
    general = None
    for batch_bytes, prefix_bytes in ((1 << 17, 2 ** 63 - 1), (0, 2 ** 63 - 1),
                                      (_native.DMAT_BATCH_BYTES, 64 * 100)):
        eng.set_dmat_workspace(batch_bytes, prefix_bytes)
        out = eng.dmat(params, *args)
        assert np.array_equal(out[6], whole[6])
        assert_outputs_close(out[:6], whole[:6])
        if prefix_bytes == 64 * 100:
            general = eng.dmat_routes()
        else:
            assert eng.dmat_routes() == routes
            if batch_bytes == 0:   # a pair at a time
                assert eng.dmat_report()["batches"] >= routes["sums"]
            elif kind != "quasars":   # (a few kB a pair)
                assert eng.dmat_report()["batches"] > 1
    assert general == dict(sums=0, handed_back=0, general=len(args[0]), outside=0)
