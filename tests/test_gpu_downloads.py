"""Results of more than one chunk of the pinned download ring: matrices of 13.5 MB (one thread) and
20 MB (several) added to what the caller's array holds, the six interleaved results of 300 000
continuum fits, sizes around a chunk, and two contexts' downloads at once."""
import ctypes
from concurrent.futures import ThreadPoolExecutor

import numpy as np
import pytest

import walk_cases as W
from picca_amd import continuum
from picca_amd._native import check
from picca_amd.engine import Engine, as_f64, as_i32, get_engine, params_from_globals, ptr
from test_gpu_continuum_lengths import make_inputs
from test_gpu_dmat_band import dmat_store, with_model

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_par", [46, 56])
def test_matrix_is_added(n_par):
    case = with_model(W.random_case(3), 2, 1)
    g, p = case.g, case.pairs
    g.num_bins_r_par, g.num_bins_r_trans = n_par, 20
    with_model(case, 2, 1)
    store = dmat_store(case.store, 0, (1,))
    eng = get_engine(0)
    eng.set_forests(store)
    params = params_from_globals(g)
    a, b, ang = as_i32(p.pair_a), as_i32(p.pair_b), as_f64(p.pair_ang)
    flags, stats = np.zeros(len(a), np.uint8), np.zeros(4, np.int64)
    nb = g.num_bins_r_par * g.num_bins_r_trans
    nm = g.num_model_bins_r_par * g.num_model_bins_r_trans
    shapes = [nb, nb * nm, nm, nm, nm, nm]
    assert (8 * nb * nm > 2 ** 24) == (n_par > 46) and 8 * nb * nm > 1.5 * 2 ** 23
    rng = np.random.default_rng(1)
    start = [rng.integers(1, 9, n).astype(float) for n in shapes]
    out = [x.copy() for x in start]
    check(eng._lib.picca_dmat_run(eng._ctx, ctypes.byref(params), len(a), ptr(a), ptr(b), ptr(ang),
                                  ptr(flags), *[ptr(x) for x in out], ptr(stats)), "dmat")
    ref = eng.dmat(params, a, b, ang, flags)
    assert stats[0] > 0
    for mine, x, r in zip(out, start, ref[:6]):
        # one rounding of the sum, and the order of the kernels' atomics
        np.testing.assert_allclose(mine, x + r.ravel(), rtol=1e-12, atol=1e-12 * abs(r).max())


def test_many_continuum_fits():
    inputs, _ = make_inputs(5)
    n, copies = 65, 300_000   # the forest of 65 pixels, the first `keep` of them masked
    o = inputs["offsets"][3]
    few = {k: np.tile(v[o:o + n], (5, 1)) for k, v in inputs.items() if k != "offsets"}
    for keep in range(5):
        few["ivar"][keep, :keep] = 0.0
    many = {k: np.tile(v, (copies // 5, 1)).ravel() for k, v in few.items()}
    res = [continuum.fit_arrays({**{k: v.ravel() for k, v in x.items()},
                                 "offsets": np.arange(0, m * n + 1, n)}, order=1)
           for x, m in ((few, 5), (many, copies))]
    for key in ("a", "b", "chi2", "ndata", "status"):
        assert np.array_equal(np.tile(res[0][key], copies // 5), res[1][key]), key


def test_two_contexts_at_once():
    """Two contexts on two host threads, each with downloads of several chunks."""
    rng = np.random.default_rng(3)
    inputs = [(rng.normal(size=(30, bins)), rng.uniform(0.5, 2, (30, bins)))
              for bins in (1500, 1460)]
    engines = [Engine(0), Engine(0)]
    try:
        alone = [eng.cov_subsample(*x)[0] for eng, x in zip(engines, inputs)]
        assert all(c.nbytes > 2 ** 24 for c in alone)
        with ThreadPoolExecutor(2) as pool:
            together = [pool.submit(lambda e=eng, v=x: [e.cov_subsample(*v)[0]
                                                        for _ in range(20)])
                        for eng, x in zip(engines, inputs)]
            for first, results in zip(alone, together):
                assert all(np.array_equal(first, c) for c in results.result())
    finally:
        for eng in engines:
            eng.close()


def test_sizes_around_a_chunk():
    """Results around the smallest block (64 KB), one and two chunks of 1 MB, and 16 MB, where the
    chunks grow and other threads take part, one after the other in one context."""
    rng = np.random.default_rng(4)
    eng = Engine(0)
    try:
        for bins in (3, 90, 91, 362, 363, 512, 513, 1448, 1449, 1774, 100):
            xi, w = rng.normal(size=(20, bins)), rng.uniform(0.5, 2, (20, bins))
            cov = eng.cov_subsample(xi, w)[0]
            mean = (xi * w).sum(0) / w.sum(0)
            x = w * (xi - mean)
            ref = x.T @ x / np.outer(w.sum(0), w.sum(0))
            np.testing.assert_allclose(cov, ref, rtol=1e-9, atol=1e-12 * np.abs(ref).max())
    finally:
        eng.close()
