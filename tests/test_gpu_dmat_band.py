"""The distortion matrix of forest pairs without cuts (prefix sums over runs) on the GPU against
the FP64 oracle: exact bin edges, zero weights, short and non-monotone forests, random
geometries, model bins that split the data bins in 1, 2, 4 (taken) or 3 (general kernels) parts,
more r_par bins than one chunk of the fill and more r_trans rows than one band of the pass.
Every test says which kernels its pairs took.  Counts equal; sums within 1e-9 relative or 1e-12 of
the largest entry, as in test_gpu_dmat."""
import numpy as np
import pytest

import walk_cases as W
from oracle import cf_oracle as O
from picca_amd import _native
from picca_amd.engine import get_engine, params_from_globals
from picca_amd.store import ForestStore
from test_gpu_dmat import assert_outputs_close

pytestmark = pytest.mark.gpu


def lattice_case(angle):
    """walk_cases.lattice_case at an angle where r_trans moves from pixel to pixel (at its own
    2e-8 it does not, and every pair takes the general kernels): pixel pairs lie within a rounding
    or two of the edges of 10 Mpc/h bins in r_par and, every 700 pixels, in r_trans."""
    case = W.lattice_case()
    case.g.num_bins_r_par = case.g.num_bins_r_trans = 20
    if angle is not None:
        r = case.store.r_comov.copy()
        case.store.r_comov[:] = r / np.cos(angle / 2)
        case.store.dist_m[:] = r * (10 / np.sin(angle / 2) / 700)
        case.pairs.pair_ang[:] = angle
    return case


def dmat_store(store, seed, orders):
    rng = np.random.default_rng(seed)
    n = len(store.offsets) - 1
    return ForestStore(store.offsets, store.z, store.r_comov, store.dist_m, store.weights,
                       store.delta, store.z_qso, store.ra, store.dec, store.thingid,
                       log_lambda=np.log10(1215.67 * (1 + store.z)),
                       order=rng.choice(orders, n).astype(np.int32))


def check(case, orders=(1,), flags=None, seed=0, sums=None, general=None):
    """sums, general: whether some pairs take the prefix sums and the general kernels."""
    g, p = case.g, case.pairs
    store = dmat_store(case.store, seed, orders)
    # a forest without two weighted pixels has no projection
    used = np.array([(store.weights[o:e] != 0).sum() for o, e in zip(store.offsets[:-1],
                                                                    store.offsets[1:])])
    keep = (used[p.pair_a] > 1) & (used[p.pair_b] > 1)
    a, b, ang = p.pair_a[keep], p.pair_b[keep], p.pair_ang[keep]
    flags = np.zeros(len(a), np.uint8) if flags is None else flags(len(a))
    eng = get_engine(0)
    eng.set_forests(store)
    mine = eng.dmat(params_from_globals(g), a, b, ang, flags)
    ref, stats = O.dmat_rows(O.params_from_module(g), store, a, b, ang, flags)
    assert list(mine[6]) == list(stats) and stats[0] > 0
    assert_outputs_close(mine[:6], ref)
    assert_routes(eng, len(a), sums, general)
    # no pair of an auto-correlation rounds past a range's end (test_host_dmat_band)
    assert eng.dmat_routes()["handed_back"] == 0


def assert_routes(eng, pairs, sums, general):
    r = eng.dmat_routes()
    assert r["sums"] + r["outside"] + r["general"] - r["handed_back"] == pairs
    assert sums is None or (r["sums"] > 0) == sums, r
    assert general is None or (r["general"] > 0) == general, r


def with_model(case, kp, kt):
    case.g.num_model_bins_r_par = kp * case.g.num_bins_r_par
    case.g.num_model_bins_r_trans = kt * case.g.num_bins_r_trans
    return case


@pytest.mark.parametrize("angle", [None, 0.004, 0.03])
@pytest.mark.parametrize("kp,kt", [(1, 1), (2, 1), (2, 2), (4, 1), (3, 1)])
def test_exact_bin_edges(kp, kt, angle):
    taken = angle is not None and kp != 3
    check(with_model(lattice_case(angle), kp, kt), sums=taken, general=not taken)


@pytest.mark.parametrize("orders", [(1,), (0, 1)])
def test_irregular_forests(orders):
    case = W.irregular_case()
    case.g.num_bins_r_par = case.g.num_bins_r_trans = 25
    check(with_model(case, 2, 1), orders, sums=True, general=True)


@pytest.mark.parametrize("orders", [(1,), (0, 1)])
@pytest.mark.parametrize("layout", ["irregular", "random"])
def test_roles_with_their_own_evolution(layout, orders):
    """alpha2 != alpha: delta1 and delta2 have prefix sums of their own."""
    case = W.irregular_case() if layout == "irregular" else W.random_case(3)
    case.g.num_bins_r_par = case.g.num_bins_r_trans = 25
    case.g.r_par_max = case.g.r_trans_max = 120.0
    case.g.alpha, case.g.alpha2 = 2.9, -1.1
    check(with_model(case, 2, 1), orders, sums=True)


def test_heavy_pixels_take_the_general_kernels():
    """One pixel a forest 1e4 times heavier (beyond that the matrix itself, the identity less the
    projections, cancels in any order of its sums)."""
    case = W.random_case(3)
    case.g.num_bins_r_par = case.g.num_bins_r_trans = 25
    case.g.r_par_max = case.g.r_trans_max = 120.0
    w, off = case.store.weights, case.store.offsets
    w[:] = np.where(w != 0, 1.0 + w / 100, 0.0)
    check(with_model(case, 2, 1), sums=True)
    for o, e in zip(off[:-1], off[1:]):
        w[o + np.flatnonzero(w[o:e])[3]] = 1.5e4
    check(with_model(case, 2, 1), sums=False, general=True)


@pytest.mark.parametrize("seed", [0, 1, 2, 3, 4, 5, 6, 7, 9])   # (8: no pair in range)
def test_random_geometries(seed):
    case = W.random_case(seed)
    case.g.num_bins_r_par = 1 + case.g.num_bins_r_par % 30
    case.g.num_bins_r_trans = 1 + case.g.num_bins_r_trans % 30
    check(with_model(case, (1, 2)[seed % 2], 1), (0, 1), seed=seed, sums=True)


@pytest.mark.parametrize("n_par,n_trans", [(64, 12), (65, 12), (16, 40), (1, 1)])
def test_chunks_and_bands(n_par, n_trans):
    """64 data and 112 model r_par bins make a chunk of the fill; a wide pair reaches more
    r_trans rows than a band of the pass holds."""
    case = W.random_case(3)
    case.g.num_bins_r_par, case.g.num_bins_r_trans = n_par, n_trans
    case.g.r_par_max, case.g.r_trans_max = 120.0, 400.0
    case.pairs.pair_ang[:] = np.linspace(0.001, 0.09, case.pairs.num_pairs)
    check(with_model(case, 2, 1), sums=True)


def test_cut_pairs_take_the_general_kernels():
    case = with_model(W.irregular_case(), 1, 1)
    case.g.num_bins_r_par = case.g.num_bins_r_trans = 15
    with_model(case, 1, 1)
    case.g.remove_same_half_plate_close_pairs = True
    check(case, flags=lambda n: (np.arange(n) % 3 == 0).astype(np.uint8)
          * _native.PICCA_PAIR_SAME_HALF_PLATE, sums=True, general=True)


def quasar_store(case, seed, orders):
    """Every pair's second forest replaced by a quasar at one of its pixels, or between them."""
    p, store = case.pairs, case.store
    rng = np.random.default_rng(seed)
    used = np.array([(store.weights[o:e] != 0).sum() for o, e in zip(store.offsets[:-1],
                                                                    store.offsets[1:])])
    keep = used[p.pair_a] > 1
    a, b, ang = p.pair_a[keep], p.pair_b[keep], p.pair_ang[keep]
    m = len(a)
    first, length = store.offsets[b], store.offsets[b + 1] - store.offsets[b]
    pixel = first + rng.integers(0, 1 << 30, m) % length
    away = rng.choice([0.0, 0.37, -21.0], m)
    both = dict(offsets=np.concatenate([store.offsets, store.offsets[-1] + np.arange(1, m + 1)]),
                r_comov=np.concatenate([store.r_comov, store.r_comov[pixel] + away]),
                dist_m=np.concatenate([store.dist_m, store.dist_m[pixel] + away]),
                z=np.concatenate([store.z, store.z[pixel]]),
                weights=np.concatenate([store.weights,
                                        rng.uniform(0.5, 2, m) * (rng.random(m) < 0.9)]),
                delta=np.concatenate([store.delta, np.zeros(m)]),
                log_lambda=np.concatenate([np.log10(1215.67 * (1 + store.z)), np.zeros(m)]),
                order=np.concatenate([rng.choice(orders, store.num_forests),
                                      np.full(m, -1)]).astype(np.int32))
    for name in ("z_qso", "ra", "dec"):
        both[name] = np.concatenate([getattr(store, name), getattr(store, name)[b]])
    both["thingid"] = np.arange(store.num_forests + m)
    flags = np.full(m, _native.PICCA_PAIR_XCF_COUNT, np.uint8)
    return ForestStore(**both), (a, store.num_forests + np.arange(m), ang, flags)


def check_quasars(case, kp, kt, seed=0, orders=(0, 1), sums=None):
    new, args = quasar_store(case, seed, orders)
    case.g.r_par_min = -case.g.r_par_max if seed % 2 == 0 else -0.6 * case.g.r_par_max
    return check_quasar_pairs(case, new, args, kp, kt, sums)


def check_quasar_pairs(case, new, args, kp, kt, sums=None, copies=1):
    """copies: times that the pair list repeats, each of which adds the same to the result."""
    g = case.g
    g.x_correlation = True
    with_model(case, kp, kt)
    eng = get_engine(0)
    eng.set_forests(new)
    mine = eng.dmat(params_from_globals(g), *args)
    params = O.params_from_module(g)
    nm = g.num_model_bins_r_par * g.num_model_bins_r_trans
    nb = g.num_bins_r_par * g.num_bins_r_trans
    ref = [np.zeros(nb), np.zeros(nb * nm)] + [np.zeros(nm) for _ in range(4)]
    stats = np.zeros(4, dtype=np.int64)
    for x, y, angle in zip(*(v[:len(v) // copies] for v in args[:3])):
        i, j = (slice(new.offsets[k], new.offsets[k + 1]) for k in (x, y))
        O.xdmat_forest(params, new.log_lambda[i], new.r_comov[i], new.dist_m[i], new.z[i],
                       new.weights[i], new.r_comov[j], new.dist_m[j], new.z[j], new.weights[j],
                       [angle], ref, new.order[x], stats)
    ref[1] = ref[1].reshape(nb, nm)
    assert list(mine[6]) == list(copies * stats) and stats[0] > 0
    assert_outputs_close(mine[:6], [copies * x for x in ref])
    assert_routes(eng, len(args[0]), sums, None)
    return eng.dmat_routes()


@pytest.mark.parametrize("angle", [None, 0.004, 0.03])
@pytest.mark.parametrize("kp,kt", [(1, 1), (2, 1), (2, 2), (3, 1)])
def test_quasars_on_exact_bin_edges(kp, kt, angle):
    taken = angle is not None and kp != 3
    check_quasars(lattice_case(angle), kp, kt, sums=taken)


@pytest.mark.parametrize("limit,copies", [("r_par_min", 1), ("r_par_max", 1),
                                          ("r_par_max", 300)])
def test_quasar_pairs_handed_back(limit, copies):
    """A pixel at r_par == r_par_min, which xcf's count pass leaves out, and one just below
    r_par_max whose distance from r_par_min rounds to the whole range: its pair goes back to the
    general kernels, the others stay; also with the whole list several times over."""
    angle = 0.02
    case = W.random_case(3)
    g = case.g
    g.num_bins_r_par, g.num_bins_r_trans = 20, 10
    g.r_par_min, g.r_par_max, g.r_trans_max = -100.0, 100.0, 120.0
    case.pairs.pair_ang[:] = angle
    new, args = quasar_store(case, 0, (0, 1))
    r_par = [(new.r_comov[new.offsets[a]:new.offsets[a + 1]] - new.r_comov[new.offsets[b]])
             * np.cos(angle / 2) for a, b in zip(*args[:2])]
    found = 0
    for v in np.concatenate(r_par):
        if limit == "r_par_min" and -110 < v < -90:
            g.r_par_min, found = float(v), 1
        if limit == "r_par_max" and 90 < v < 110:
            top = np.nextafter(v, np.inf)
            if np.floor((v + 100.0) / (top + 100.0) * 20) == 20:
                g.r_par_max, found = float(top), 1
        if found:
            break
    assert found
    routes = check_quasar_pairs(case, new, tuple(np.tile(x, copies) for x in args), 2, 1,
                                copies=copies)
    assert copies <= routes["handed_back"] < routes["sums"]


@pytest.mark.parametrize("angle", [0.004, 0.03])
def test_quasars_with_irregular_forests(angle):
    case = W.irregular_case()
    case.pairs.pair_ang[:] = angle
    case.g.num_bins_r_par = case.g.num_bins_r_trans = 25
    check_quasars(case, 2, 1, sums=True)


@pytest.mark.parametrize("seed", [0, 1, 2, 3, 5, 6, 7])   # (4: no pair in range)
def test_quasars_in_random_geometries(seed):
    case = W.random_case(seed)
    case.g.num_bins_r_par = 1 + case.g.num_bins_r_par % 30
    case.g.num_bins_r_trans = 1 + case.g.num_bins_r_trans % 30
    case.g.r_par_max = max(case.g.r_par_max, 120.0)
    case.g.r_trans_max = max(case.g.r_trans_max, 120.0)
    case.pairs.pair_ang[:] *= 0.3
    check_quasars(case, (1, 2)[seed % 2], (1, 1, 4)[seed % 3], seed=seed)


@pytest.mark.parametrize("n_par,n_trans", [(64, 12), (65, 12), (130, 40), (1, 1)])
def test_quasar_chunks(n_par, n_trans):
    case = W.random_case(3)
    case.g.num_bins_r_par, case.g.num_bins_r_trans = n_par, n_trans
    case.g.r_par_max, case.g.r_trans_max = 120.0, 400.0
    case.pairs.pair_ang[:] = np.linspace(0.001, 0.09, case.pairs.num_pairs)
    check_quasars(case, 2, 1)
