"""Single bins of the correlation with signed r_par and with cuts, whose runs are differences of a
forest's prefix sums, against 80-bit sums: forests with one pixel far heavier than the others
(their pairs take the pair loop) or with a far larger delta, uniform and log-uniform weights.  And
the rule itself (level_values of picca_amd/csrc/xi_walk.h) at its two bounds.

Bars per bin: 1e-12 of the weight, r_trans and z sums, of the r_par sum plus weight times bin
width (the sum cancels near 0, away from it each pair adds |r_par| times its weight), and of
sum |delta delta w w| for xi.  A bin adds up to 1e4 pairs:
in-order sums stay below 1e4 2^-53 = 1.1e-12 at the worst, 6e-14 as measured; a level forest's
prefix sums below 8192 2^-53 = 9e-13 a pixel, and less where a bin adds many."""
import ctypes

import numpy as np
import pytest

import walk_cases as W
import walk_harness as H
from picca_amd.engine import params_from_globals

LEVEL_W, LEVEL_DW = 8, 16


def level_flags(w, dw):
    n = max(len(w), len(dw))   # the shorter one ends in zeros
    w, dw = (np.concatenate([x, np.zeros(n - len(x))]).astype(np.float64) for x in (w, dw))
    return H.lib().xi_level_flags(ctypes.c_int(len(w)), H._p(w), H._p(dw))


def survey(option, seed=0):
    """Six forests of the 0.8 A grid and all their pairs."""
    rng = np.random.default_rng(seed)
    forests = []
    for n in (350, 420, 300, 260, 330, 380):
        r = 3700.0 + float(rng.uniform(0, 150)) + 0.55 * np.arange(n) + rng.uniform(0, 0.05, n)
        forests.append({"r": r, "d": r - 2.0, "z": 2.0 + r / 1e4, "w": rng.uniform(0.5, 2, n),
                        "delta": rng.normal(0, 0.3, n)})
    pa, pb, _, prow = W._all_pairs(len(forests), 0.0)
    g = W.Globals(num_bins_r_par=25, num_bins_r_trans=12, r_par_max=100.0, r_trans_max=60.0)
    case = W.Case(g, W._store(forests), pa, pb, rng.uniform(0.001, 0.0075, len(pa)), 0 * prow, 1)
    if option == "cross":
        g.x_correlation, g.num_bins_r_par, g.r_par_min = True, 50, -100.0
    else:
        g.remove_same_half_plate_close_pairs = True
        case.pairs.pair_flags[:] = rng.random(case.pairs.num_pairs) < 0.5
    return case


def extended(case):
    """The sums and sum |delta delta w w| per bin in 80 bits."""
    g, p, s = case.g, case.pairs, case.store
    nb = g.num_bins_r_par * g.num_bins_r_trans
    width = (g.r_par_max - g.r_par_min) / g.num_bins_r_par
    bins, terms = [], []
    for a, b, ang, flag in zip(p.pair_a, p.pair_b, p.pair_ang, p.pair_flags):
        i, j = (slice(s.offsets[k], s.offsets[k + 1]) for k in (a, b))
        r_par = (s.r_comov[i][:, None] - s.r_comov[j][None]) * np.cos(ang / 2)
        if not g.x_correlation:
            r_par = np.abs(r_par)
        r_trans = (s.dist_m[i][:, None] + s.dist_m[j][None]) * np.sin(ang / 2)
        keep = ((r_par < g.r_par_max) & (r_par >= g.r_par_min) & (r_trans < g.r_trans_max)
                & (s.weights[i][:, None] * s.weights[j][None] != 0))
        if g.remove_same_half_plate_close_pairs and flag:
            keep &= np.abs(r_par) >= width
        k = (np.floor(r_trans / g.r_trans_max * g.num_bins_r_trans) + g.num_bins_r_trans
             * np.floor((r_par - g.r_par_min) / (g.r_par_max - g.r_par_min) * g.num_bins_r_par))
        long = np.longdouble
        w12 = s.weights[i][:, None].astype(long) * s.weights[j][None]
        x12 = ((s.delta[i] * s.weights[i])[:, None].astype(long)
               * (s.delta[j] * s.weights[j])[None])
        z = (s.z[i][:, None] + s.z[j][None]) / 2
        bins.append(k[keep].astype(np.int64))
        terms.append(np.stack([t[keep] for t in (w12, x12, r_par * w12, r_trans * w12, z * w12,
                                                 np.abs(x12))]))
    bins, terms = np.concatenate(bins), np.concatenate(terms, axis=1)
    order = np.argsort(bins, kind="stable")
    first = np.flatnonzero(np.diff(bins[order], prepend=-1))
    out = np.zeros((6, nb), dtype=np.longdouble)
    out[:, bins[order][first]] = np.add.reduceat(terms[:, order], first, axis=1)
    return out, width


def check(case):
    p, g = case.pairs, case.g
    out, st = H.xi_walk_cuts(params_from_globals(g), case.store, p.pair_a, p.pair_b, p.pair_ang,
                             p.pair_flags, p.pair_row, 1, max(1, g.num_bins_r_par // 2))
    ref, width = extended(case)
    mask = ref[0] > 0
    assert mask.sum() > 100 and st["oob"] == 0
    scale = [ref[0], ref[5], ref[0] * width + np.abs(ref[2]), ref[3], ref[4]]
    for k in range(5):
        assert np.max(np.abs(out[k][0] - ref[k])[mask] / scale[k][mask]) < 1e-12, k
    return st


@pytest.mark.parametrize("option", ["cross", "plate"])
@pytest.mark.parametrize("heavier", [1.0, 100.0, 1e3, 1e4, 1e8])
def test_one_heavy_pixel(option, heavier):
    case = survey(option)
    s, rng = case.store, np.random.default_rng(5)
    for k in range(s.num_forests):
        s.weights[rng.integers(s.offsets[k], s.offsets[k + 1])] = 1.25 * heavier   # (mean 1.25)
    st = check(case)
    assert (st["walk_tasks"] > 0) == (heavier <= 1e3)


@pytest.mark.parametrize("option", ["cross", "plate"])
def test_one_large_delta(option):
    case = survey(option)
    s = case.store
    s.delta[s.offsets[:-1] + 100] = 1e8
    assert check(case)["walk_tasks"] == 0


@pytest.mark.parametrize("option", ["cross", "plate"])
def test_log_uniform_weights(option):
    """Weights over 1e-3..1e2, as the heavy-tailed survey's, are level and walk."""
    case = survey(option)
    rng = np.random.default_rng(2)
    case.store.weights[:] = np.exp(rng.uniform(np.log(1e-3), np.log(1e2),
                                               len(case.store.weights)))
    assert check(case)["pair_tasks"] == 0


def test_level_values():
    ones = np.ones(600)
    both = LEVEL_W | LEVEL_DW
    one_heavy = lambda h: np.concatenate([ones, [h]])
    assert level_flags(ones, 0 * ones) == both
    assert level_flags(-ones, ones) == both
    # the sum is 8192 mean values, 600 + h = 8192; 16384 for delta * weight
    assert level_flags(one_heavy(7592.0), ones) == both
    assert level_flags(one_heavy(7593.0), ones) == LEVEL_DW
    assert level_flags(ones, one_heavy(15784.0)) == both
    assert level_flags(ones, one_heavy(15785.0)) == LEVEL_W
    # one weight below 2^-25 of the sum; a delta may be as small
    light = 600 / (2.0 ** 25 - 1)
    assert level_flags(one_heavy(light * (1 + 1e-9)), ones) == both
    assert level_flags(one_heavy(light * (1 - 1e-9)), ones) == LEVEL_DW
    assert level_flags(ones, one_heavy(1e-300)) == both
    # zeros are no values; one value, or none, is exact
    assert level_flags(np.concatenate([ones, np.zeros(5000)]), ones) == both
    assert level_flags([0.0, 1e200, -0.0], [0.0, 0.0, 1e-300]) == both
    assert level_flags([], []) == both
    assert level_flags([1.0, 1e8], [0.5, 0.5]) == LEVEL_DW
    # more than an eighth heavy: the floor of the weights
    assert level_flags(np.where(np.arange(600) % 5 == 0, 1e8, 1.0), ones) == LEVEL_DW
    # the largest eighth is left out whether one pass settles it or not
    spread = np.exp(np.linspace(np.log(1e-3), np.log(1e2), 600))
    assert level_flags(spread, spread) == both
    # beyond 8192 pixels no weights are level; sums that overflow are not
    assert level_flags(np.ones(8192), ones) == both
    assert level_flags(np.ones(8193), ones) == LEVEL_DW
    assert level_flags(1e308 * ones, ones) == LEVEL_DW
