"""The work that a user of picca_amd has it do, as cases to time and to compare.

Every case goes through the package's public entry points (``picca_amd.engine.Engine`` with a
resident forest store, as the drivers hold it, and ``picca_amd.cf`` for the one-pair call).
Sizes and distributions are those of the benchmark's synthetic surveys (``picca_amd.synth``)
at the same sky density: log10-lambda and 0.8 A grids, forests of 50 to 1500 pixels, 50 x 50
bins to 200 Mpc/h, 15 x 15 to 60 Mpc/h for the smaller binning of picca's own tests.

Kinds:

* ``pair``       one forest pair added to the caller's arrays (the smallest call: one upload,
                 one launch and one download);
* ``xi``         the correlation function over all neighbour pairs of a survey, resident in
                 device memory, one output row per healpix; options: removal of close pairs of
                 one half plate, cuts on the pair redshift, a second catalogue with signed
                 r_par (``--unfold-cf``);
* ``xcf``        the forest x quasar correlation of a survey with its own quasars;
* ``dmat``       the distortion matrix of the pairs kept by the rejection draw;
* ``xdmat``      the forest x quasar distortion matrix;
* ``metal``      a metal distortion matrix (LYA x SiIII(1207)), both absorber passes;
* ``wick``       the Wick covariance terms T1-T3 of a few forest pairs;
* ``cov``        the subsampling covariance of the correlation rows;
* ``continuum``  one iteration of the continuum fit: interpolation of the mean continuum, the
                 fit of every forest, the weighted stack.
"""
import types

import numpy as np
import torch

from picca_amd import _native, batch, cf, metal, synth
from picca_amd.constants import ABSORBER_IGM, Cosmo
from picca_amd.engine import Engine, params_from_globals
from picca_amd.neighbours import find_neighbours
from picca_amd.utils import compute_ang_max

Z_REF = 2.25
ALPHA = 2.9
OMEGA_M = 0.315


# -- cases ----------------------------------------------------------------------------------

def listed():
    return [
        # one call of the per-pair entry point of picca.cf, at the test data's binning
        dict(name="pair", kind="pair", n1=210, n2=190, bins=15, r_max=60.0),
        # a small eBOSS-like field: log10-lambda grid, about two pixels per r_par bin
        dict(name="xi_log", kind="xi", workload="survey_small", forests=1000, bins=50,
             r_max=200.0, cross=False, half_plate=False, z_cut=False),
        # the headline run at its density: 0.8 A grid, forests of 50 to 1500 pixels
        dict(name="xi_linear", kind="xi", workload="survey_100k", forests=3000, bins=50,
             r_max=200.0, cross=False, half_plate=False, z_cut=False),
        # the same with --remove-same-half-plate-close-pairs, the usual eBOSS setting
        dict(name="xi_half_plate", kind="xi", workload="survey_100k", forests=500, bins=50,
             r_max=200.0, cross=False, half_plate=True, z_cut=False),
        # two delta fields with signed r_par: 100 x 50 bins over [-200, 200) Mpc/h
        dict(name="xi_cross", kind="xi", workload="survey_100k", forests=400, bins=50,
             r_max=200.0, cross=True, half_plate=False, z_cut=False),
        # forest x quasar correlation, 100 x 50 bins
        dict(name="xcf", kind="xcf", workload="survey_100k", forests=3000, bins=50,
             r_max=200.0),
        # distortion matrix, 50 x 50 data bins and 100 x 50 model bins
        dict(name="dmat", kind="dmat", workload="survey_100k", forests=2500, bins=50,
             model=2, r_max=200.0, reject=0.99),
        dict(name="xdmat", kind="xdmat", workload="survey_100k", forests=3000, bins=50,
             model=1, r_max=200.0, reject=0.95),
        dict(name="metal", kind="metal", workload="survey_100k", forests=2500, bins=50,
             r_max=200.0, reject=0.95),
        # Wick terms at picca's own binning; the work grows as the square of a pair's pixels
        dict(name="wick", kind="wick", workload="survey_100k", forests=1000, bins=15,
             r_max=60.0, pairs=24),
        # picca_export's covariance: a survey's healpix rows, 50 x 50 bins
        dict(name="cov", kind="cov", samples=1196, bins=2500),
        dict(name="continuum", kind="continuum", forests=20000, tol=1e-12),
    ]


def _log_int(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    kind = rng.choice(["pair", "xi", "xi", "xi", "xcf", "dmat", "xdmat", "metal", "wick",
                       "cov", "continuum"])
    if kind == "pair":
        return dict(kind=kind, n1=_log_int(rng, 1, 1500), n2=_log_int(rng, 1, 1500),
                    bins=rng.choice([15, 30, 50]), r_max=rng.choice([60.0, 120.0, 200.0]))
    if kind == "cov":
        return dict(kind=kind, samples=_log_int(rng, 14, 1500), bins=_log_int(rng, 225, 2500))
    if kind == "continuum":
        return dict(kind=kind, forests=_log_int(rng, 100, 20000),
                    tol=rng.choice([1e-12, 1e-8]))
    workload = rng.choice(["survey_small", "survey_100k", "survey_300k", "survey_100k_heavy"])
    bins, r_max = rng.choice([(50, 200.0), (50, 200.0), (15, 60.0), (37, 150.0)])
    case = dict(kind=kind, workload=workload, bins=bins, r_max=r_max)
    if kind == "xi":
        case["cross"] = rng.random() < 0.3
        case["half_plate"] = rng.random() < 0.3
        case["z_cut"] = rng.random() < 0.2
        slow = case["cross"] or case["half_plate"] or case["z_cut"]
        case["forests"] = _log_int(rng, 20, 400 if slow else 2500)
    elif kind == "xcf":
        case["forests"] = _log_int(rng, 40, 3000)
    elif kind == "wick":
        case.update(bins=15, r_max=60.0, forests=_log_int(rng, 200, 1000),
                    pairs=_log_int(rng, 2, 24))
    else:
        case["forests"] = _log_int(rng, 60, 2500)
        case["reject"] = rng.choice([0.9, 0.99]) if case["forests"] < 700 else 0.99
        if kind != "metal":
            case["model"] = rng.choice([1, 2]) if kind == "dmat" else 1
    return case


# -- inputs ---------------------------------------------------------------------------------

class Globals:
    """The module globals of a run, as the drivers set them."""

    def __init__(self, case):
        bins = case["bins"]
        signed = case["kind"] in ("xcf", "xdmat") or case.get("cross", False)
        self.num_bins_r_par = 2 * bins if signed else bins
        self.num_bins_r_trans = bins
        self.num_model_bins_r_par = self.num_bins_r_par * case.get("model", 1)
        self.num_model_bins_r_trans = bins
        self.r_par_max = case["r_max"]
        self.r_par_min = -case["r_max"] if signed else 0.0
        self.r_trans_max = case["r_max"]
        self.z_min_pairs = 2.3 if case.get("z_cut") else None
        self.z_max_pairs = 2.9 if case.get("z_cut") else None
        self.zerr_cut_deg = None
        self.zerr_cut_kms = None
        self.z_ref = Z_REF
        self.alpha = ALPHA
        self.alpha2 = 1.44 if case["kind"] == "xdmat" else ALPHA
        self.x_correlation = signed
        self.rmu_binning = False
        self.ang_correlation = False
        self.remove_same_half_plate_close_pairs = bool(case.get("half_plate", False))
        self.redshift_evolution_in_distortion_matrix = True


def _survey(case, seed, forests):
    spec = synth.WORKLOADS[case["workload"]]
    survey = synth.make_survey(case["workload"], seed=seed, scale=forests / spec["n"],
                               z_ref=Z_REF, alpha=ALPHA, om=OMEGA_M)
    # spectroscopic plates of 1.5 degrees, fibres 1 to 1000
    rng = np.random.default_rng(seed + 1)
    store = survey.store
    store.plate = (np.floor(store.ra / np.radians(1.5)) * 1000
                   + np.floor(store.dec / np.radians(1.5))).astype(np.int64)
    store.fiberid = rng.integers(1, 1001, store.num_forests)
    return survey


def _rows(case):
    """Output rows of a case: shares of about 84 forests in healpix order, the forests of one
    healpix of the 100k-forest survey (a fixed number, so that the outputs' shape does not
    depend on where the seed puts the forests)."""
    return max(1, round(case["forests"] / 84))


def _row_of(case, healpix, source):
    """The row of each source forest."""
    rank = np.empty(len(healpix), dtype=np.int64)
    rank[np.argsort(healpix, kind="stable")] = np.arange(len(healpix))
    return (rank[source] * _rows(case) // len(healpix)).astype(np.int32)


def _xi_inputs(case, seed):
    g = Globals(case)
    n = case["forests"]
    survey = _survey(case, seed, 2 * n if case["cross"] else n)
    store = survey.store
    ang_max = compute_ang_max(Cosmo(OMEGA_M, verbose=False), g.r_trans_max, survey.z_min)
    if case["cross"]:
        pairs = batch.xi_pairs(store, survey.healpix[:n], ang_max,
                               target_store_index=np.arange(n, store.num_forests),
                               target_healpix=survey.healpix[n:], auto=False,
                               remove_same_half_plate_close_pairs=case["half_plate"])
    else:
        pairs = batch.xi_pairs(store, survey.healpix, ang_max,
                               remove_same_half_plate_close_pairs=case["half_plate"])
    n = n if case["cross"] else store.num_forests
    return g, store, pairs, _row_of(case, survey.healpix[:n], pairs.pair_a)


def _kept_pairs(case, seed):
    """The neighbour pairs that the rejection draw keeps."""
    g = Globals(case)
    survey = _survey(case, seed, case["forests"])
    ang_max = compute_ang_max(Cosmo(OMEGA_M, verbose=False), g.r_trans_max, survey.z_min)
    pairs = batch.xi_pairs(survey.store, survey.healpix, ang_max)
    keep = np.random.RandomState(seed).rand(pairs.num_pairs) > case["reject"]
    return (g, survey.store, pairs.pair_a[keep], pairs.pair_b[keep], pairs.pair_ang[keep],
            pairs.pair_flags[keep])


def _xcf_inputs(case, seed):
    """A survey and its own quasars: (globals, store, quasars, pairs' forest, quasar, angle and
    row, number of rows)."""
    g = Globals(case)
    survey = _survey(case, seed, case["forests"])
    store = survey.store
    cosmo = Cosmo(OMEGA_M, verbose=False)
    qso = types.SimpleNamespace(
        x_cart=store.x_cart, y_cart=store.y_cart, z_cart=store.z_cart, ra=store.ra,
        dec=store.dec, cos_dec=store.cos_dec, thingid=store.thingid, z_qso=store.z_qso,
        r_comov=np.asarray(cosmo.get_r_comov(store.z_qso), dtype=np.float64),
        dist_m=np.asarray(cosmo.get_dist_m(store.z_qso), dtype=np.float64),
        weights=((1 + store.z_qso) / (1 + Z_REF)) ** (1.44 - 1))
    ang_max = compute_ang_max(cosmo, g.r_trans_max, survey.z_min, float(store.z_qso.min()))
    order = np.argsort(survey.healpix, kind="stable")
    nl = find_neighbours(store, order, order, ang_max, auto=False, target_store=qso)
    source = nl.source_index()
    forest, quasar, angle = order[source], order[nl.target], nl.angle
    first = store.r_comov[store.offsets[:-1]]
    last = store.r_comov[store.offsets[1:] - 1]
    c = np.cos(angle / 2.0)
    keep = (((first[forest] - qso.r_comov[quasar]) * c < g.r_par_max)
            & ((last[forest] - qso.r_comov[quasar]) * c > g.r_par_min))
    forest = forest[keep]
    return (g, store, qso, forest, quasar[keep], angle[keep],
            _row_of(case, survey.healpix, forest), _rows(case))


def _xdmat_inputs(case, seed):
    """The deltas followed by one one-pixel forest of order -1 per quasar, and the kept
    (delta, quasar) pairs."""
    g, store, qso, forest, quasar, angle, _, _ = _xcf_inputs(case, seed)
    nf = store.num_forests
    keep = np.random.RandomState(seed).rand(len(forest)) > case["reject"]
    both = dict(offsets=np.concatenate([store.offsets,
                                        store.offsets[-1] + np.arange(1, nf + 1)]),
                log_lambda=np.concatenate([store.log_lambda, np.zeros(nf)]),
                delta=np.concatenate([store.delta, np.zeros(nf)]),
                order=np.concatenate([store.order, np.full(nf, -1, dtype=np.int32)]))
    for name in ("r_comov", "dist_m", "weights"):
        both[name] = np.concatenate([getattr(store, name), getattr(qso, name)])
    both["z"] = np.concatenate([store.z, qso.z_qso])
    for name in ("z_qso", "ra", "dec", "thingid"):
        both[name] = np.concatenate([getattr(store, name), getattr(qso, name)])
    a, b = forest[keep], nf + quasar[keep]
    return (g, type(store)(**both), a, b, angle[keep],
            np.full(len(a), _native.PICCA_PAIR_XCF_COUNT, dtype=np.uint8))


def _metal_inputs(case, seed):
    g, store, a, b, angle, flags = _kept_pairs(case, seed)
    cosmo = Cosmo(OMEGA_M, verbose=False)
    tables = [metal.absorber_table(store, ABSORBER_IGM["LYA"], ALPHA, cosmo),
              metal.absorber_table(store, ABSORBER_IGM["SiIII(1207)"], 1.0, cosmo)]
    return g, store, a, b, angle, flags, tables, (1 + Z_REF) ** (ALPHA + 1.0 - 2)


def _wick_inputs(case, seed):
    """The first neighbour pairs of a random subset of the forests, with a smooth weighted 1-D
    correlation per forest."""
    g = Globals(case)
    survey = _survey(case, seed, case["forests"])
    store = survey.store
    ang_max = compute_ang_max(Cosmo(OMEGA_M, verbose=False), g.r_trans_max, survey.z_min)
    pairs = batch.xi_pairs(store, survey.healpix, ang_max)
    pick = np.random.RandomState(seed).permutation(pairs.num_pairs)[:case["pairs"]]
    pick.sort()
    a, b, angle = pairs.pair_a[pick], pairs.pair_b[pick], pairs.pair_ang[pick]
    wx_off = np.full(store.num_forests, -1, dtype=np.int64)
    mats, used = [], 0
    for f in np.unique(np.concatenate([a, b])):
        w = store.weights[store.offsets[f]:store.offsets[f + 1]]
        k = np.arange(len(w))
        profile = 0.01 * np.exp(-k / 7.0)
        mats.append((np.outer(w, w) * profile[np.abs(k[:, None] - k[None, :])]).ravel())
        wx_off[f] = used
        used += len(w) ** 2
    wx = np.concatenate(mats) if mats else np.zeros(0)
    zev = ((1 + store.z) / (1 + Z_REF)) ** (ALPHA - 1)
    return g, store, a, b, angle, zev, wx_off, wx


def _cov_inputs(case, seed):
    rng = np.random.default_rng(seed)
    shape = (case["samples"], case["bins"])
    weights = np.exp(rng.normal(8.0, 0.5, (shape[0], 1)) + rng.normal(0.0, 0.2, shape))
    xi = rng.normal(-1e-4, 1e-3, shape) + 1e-3 / np.sqrt(1.0 + np.arange(shape[1]))
    weights[rng.random(shape) < 0.01] = 0.0   # rows at the edge of the footprint
    return xi, weights


def _continuum_inputs(case, seed):
    """Forests of 1040-1200 A rest on the log10-lambda grid of step 1e-4 from 3600 A, with a
    linear continuum, absorption and noise, and smooth variance functions."""
    rng = np.random.default_rng(seed)
    n = case["forests"]
    z_qso = rng.uniform(2.1, 3.5, n)
    shift = np.log10(1 + z_qso)
    ll0, step = np.log10(3600.0), 1e-4
    lo = np.maximum(np.ceil((np.log10(1040.0) + shift - ll0) / step), 0).astype(np.int64)
    hi = np.floor((np.log10(1200.0) + shift - ll0) / step).astype(np.int64)
    lengths = hi - lo + 1
    offsets = np.zeros(n + 1, dtype=np.int64)
    np.cumsum(lengths, out=offsets[1:])
    npix = int(offsets[-1])
    seg = np.repeat(np.arange(n), lengths)
    ll = ll0 + step * (np.repeat(lo - offsets[:-1], lengths) + np.arange(npix))
    ll_rest = ll - shift[seg]
    ll_min = np.log10(1040.0)
    x = (ll_rest - ll_min) / (np.log10(1200.0) - ll_min)
    amp = np.exp(rng.uniform(np.log(0.5), np.log(5.0), n))
    slope = amp * rng.normal(0.0, 0.3, n)
    snr = rng.uniform(1.0, 10.0, n)
    shape = 1.0 + 0.1 * np.sin(9.0 * x)
    cont = (amp[seg] + slope[seg] * (x - 0.5)) * shape
    z = 10 ** ll / 1215.67 - 1
    trans = np.exp(-0.0023 * (1 + z) ** 3.64 * np.exp(rng.normal(0.0, 0.8, npix) - 0.32))
    sigma = np.abs(cont) / snr[seg] + 1e-3
    grid = np.arange(ll_min, np.log10(1200.0) + 0.5e-3, 1e-3)
    bins = np.clip(((ll_rest - grid[0]) / 1e-3 + 0.5).astype(np.int64), 0, len(grid) - 1)
    flux = cont * trans + sigma * rng.normal(size=npix)
    ivar = 1.0 / sigma ** 2
    ivar[rng.random(npix) < 0.01] = 0.0   # masked pixels
    a0 = np.bincount(seg, weights=flux * ivar, minlength=n) / np.bincount(
        seg, weights=ivar, minlength=n)
    return dict(offsets=offsets, flux=flux, ivar=ivar, x=x, eta=1.0 + 0.1 * np.cos(z),
                var_lss=0.05 + 0.02 * z, fudge=np.full(npix, 1e-3), ll_rest=ll_rest,
                trans=np.ones(npix), bins=bins, grid=grid,
                nodes=1.0 + 0.05 * np.sin(40.0 * (grid - grid[0])), a0=a0, b0=np.zeros(n))


def _one_pair(case, seed):
    """Two forests of the 0.8 A grid, a few arcminutes apart."""
    rng = np.random.default_rng(seed)
    cosmo = Cosmo(OMEGA_M, verbose=False)
    forests = []
    for n in (case["n1"], case["n2"]):
        start = int(rng.integers(600, 900))
        z = (3600.0 + 0.8 * (start + np.arange(n))) / 1215.67 - 1.0
        w = ((1 + z) / (1 + Z_REF)) ** (ALPHA - 1) / (rng.uniform(0.1, 1.0, n) ** 2 + 0.05)
        forests.append((z, np.asarray(cosmo.get_r_comov(z)), np.asarray(cosmo.get_dist_m(z)),
                        w, rng.normal(0.0, 0.3, n), float(z[-1] + 0.1)))
    return Globals(case), forests[0], forests[1], float(rng.uniform(1e-4, 0.8)
                                                        * case["r_max"] / 4000.0)


# -- passes ---------------------------------------------------------------------------------

def prepare(case, seed):
    kind = case["kind"]
    state = types.SimpleNamespace(kind=kind)
    if kind == "pair":
        g, one, two, angle = _one_pair(case, seed)
        state.globals, state.args = vars(g), (*one, *two, angle, False)
        state.bins = g.num_bins_r_par * g.num_bins_r_trans
        return state
    state.engine = eng = Engine()
    if kind == "cov":
        state.args = _cov_inputs(case, seed)
    elif kind == "continuum":
        c = state.inputs = _continuum_inputs(case, seed)
        ones = np.ones(len(c["flux"]))
        eng.cont_set_forests(c["offsets"], c["flux"], c["ivar"], ones, c["x"], c["eta"],
                             c["var_lss"], c["fudge"],
                             np.ones(case["forests"], dtype=np.int32))
        eng.cont_set_rest_frame(c["ll_rest"], c["trans"], c["bins"], len(c["grid"]))
        state.tol = case["tol"]
    elif kind == "xi":
        g, store, pairs, row = _xi_inputs(case, seed)
        eng.set_forests(store)
        eng.set_xi_pairs(pairs.pair_a, pairs.pair_b, pairs.pair_ang, pairs.pair_flags, row,
                         _rows(case))
        state.params = params_from_globals(g)
    elif kind == "xcf":
        g, store, qso, forest, quasar, angle, row, rows = _xcf_inputs(case, seed)
        eng.set_forests(store)
        eng.xcf_set_pairs(forest, qso.r_comov[quasar], qso.dist_m[quasar], qso.z_qso[quasar],
                          qso.weights[quasar], angle, row, rows)
        state.params = params_from_globals(g)
    elif kind in ("dmat", "xdmat"):
        g, store, *state.pairs = (_kept_pairs if kind == "dmat" else _xdmat_inputs)(case, seed)
        eng.set_forests(store)
        state.params = params_from_globals(g)
    elif kind == "metal":
        g, store, *rest = _metal_inputs(case, seed)
        state.pairs, tables, state.den = rest[:4], rest[4], rest[5]
        eng.set_forests(store)
        for slot, table in enumerate(tables):
            eng.metal_set_absorber(slot, *table)
        state.params = params_from_globals(g)
        state.sizes = (g.num_bins_r_par * g.num_bins_r_trans,
                       g.num_model_bins_r_par * g.num_model_bins_r_trans)
    elif kind == "wick":
        g, store, a, b, angle, zev, wx_off, wx = _wick_inputs(case, seed)
        eng.set_forests(store)
        state.params = params_from_globals(g)
        state.args = (a, b, angle, zev, zev, wx_off, wx)
    return state


def run(state):
    kind = state.kind
    if kind == "pair":
        for name, value in state.globals.items():
            setattr(cf, name, value)
        out = [np.zeros(state.bins) for _ in range(5)] + [np.zeros(state.bins, dtype=np.int64)]
        cf.compute_xi_forest_pairs_fast(*state.args, *out)
        return out
    eng = state.engine
    if kind in ("xi", "xcf"):
        r = eng.xi(state.params) if kind == "xi" else eng.xcf(state.params)
        return [r.weights, r.xi, r.r_par, r.r_trans, r.z, r.num_pairs]
    if kind in ("dmat", "xdmat"):
        return list(eng.dmat(state.params, *state.pairs))
    if kind == "metal":
        out = metal.outputs(*state.sizes)
        counts = []
        for slots in ((0, 1), (1, 0)):
            r = eng.metal_pass(state.params, _native.PICCA_METAL_AUTO, *slots, state.den,
                               *state.pairs, out)
            counts.append([r["data_pairs"], r["model_pairs"]])
        return out + [np.array(counts)]
    if kind == "wick":
        return list(eng.wick_t123(state.params, *state.args)[:5])
    if kind == "cov":
        return [eng.cov_subsample(*state.args)[0]]
    c = state.inputs
    eng.cont_set_mean_cont(c["grid"], c["nodes"])
    fit = eng.cont_fit(c["a0"], c["b0"], tol=state.tol)
    total, weight, _ = eng.cont_stack(len(c["grid"]))
    return [fit["a"], fit["b"], fit["chi2"], fit["ndata"], fit["status"], total, weight]


# -- work and tolerance ---------------------------------------------------------------------

def _typical(case):
    """(mean pixels of a forest, expected neighbour pairs) of a case's survey."""
    spec = synth.WORKLOADS[case["workload"]]
    pixels = {"rest": 207, "uniform": 640, "loguniform": 390}[spec["length"]]
    n = case["forests"]
    density = spec["n"] / spec["side_deg"] ** 2
    disc = np.pi * (case["r_max"] / 68.0) ** 2      # square degrees within r_trans_max
    near = min(0.75 * n, density * disc)
    return pixels, 0.5 * n * near


def work(case):
    """Bytes: the inputs read once and the outputs written once.  Operations: of the sums that
    the definition asks for over the accepted pixel pairs (five products and sums per pair for
    a correlation, the pair's terms for a matrix)."""
    kind = case["kind"]
    if kind == "pair":
        n1, n2 = case["n1"], case["n2"]
        return {"bytes": 40.0 * (n1 + n2) + 48.0 * case["bins"] ** 2, "flops": 10.0 * n1 * n2}
    if kind == "cov":
        s, b = case["samples"], case["bins"]
        return {"bytes": 16.0 * s * b + 8.0 * b * b, "flops": 1.0 * s * b * b}
    if kind == "continuum":
        pixels = 600.0 * case["forests"]
        return {"bytes": 76.0 * pixels, "flops": 4 * 60.0 * pixels}
    pixels, pairs = _typical(case)
    g = Globals(case)
    nb = g.num_bins_r_par * g.num_bins_r_trans
    nm = g.num_model_bins_r_par * g.num_model_bins_r_trans
    store = 40.0 * pixels * case["forests"]
    reach = 0.28 * min(1.0, case["r_max"] / 200.0)   # accepted share of the pixel pairs
    if kind == "xi":
        fields = 2 if case["cross"] else 1
        pairs *= 2 if case["cross"] else 1
        rows = _rows(case)
        return {"bytes": fields * store + 25.0 * pairs + 48.0 * rows * nb,
                "flops": 10.0 * reach * pairs * pixels ** 2}
    if kind == "xcf":
        rows = _rows(case)
        return {"bytes": store + 48.0 * 2 * pairs + 48.0 * rows * nb,
                "flops": 10.0 * 0.4 * 2 * pairs * pixels}
    if kind == "wick":
        n = case["pairs"]
        return {"bytes": 16.0 * n * pixels ** 2 + 24.0 * nb * nb,
                "flops": 4.0 * n * (0.1 * pixels ** 2) ** 2 / 7}
    kept = pairs * (1 - case["reject"])
    if kind == "dmat":
        return {"bytes": store + 25.0 * kept + 8.0 * nb * nm,
                "flops": 60.0 * reach * kept * pixels ** 2}
    if kind == "xdmat":
        return {"bytes": store + 25.0 * 2 * kept + 8.0 * nb * nm,
                "flops": 40.0 * 0.4 * 2 * kept * pixels}
    return {"bytes": 2.6 * store + 25.0 * kept + 8.0 * nb * nm,
            "flops": 2 * 20.0 * reach * kept * pixels ** 2}


def tolerance(case):
    """FP64 sums in another order (measured against 64-bit torch: up to 1.5e-14 relative, 6e-14
    for a single value); the counts are whole numbers and equal.  The continuum's (a, b) are
    those of a minimiser that stops at a Newton decrement of tol |chi2|, so they are known to
    about the square root of it (measured at 1e-12: 1.7e-6 relative, 2.8e-5 for one forest)."""
    if case["kind"] == "continuum":
        wide = (case["tol"] / 1e-12) ** 0.5
        return {"rel": 7e-6 * wide, "max": 1.2e-4 * wide}
    return {"rel": 1e-13, "max": 1e-12}


# -- the same in plain torch, 64 bits ---------------------------------------------------------

EXACT_PIXEL_PAIRS = 6.0e8     # of a case whose sums over pixel pairs are done here


def _dev(x):
    return torch.as_tensor(np.ascontiguousarray(x), device="cuda" if torch.cuda.is_available()
                           else "cpu")


def _blocks(off, a, b, budget=1 << 24):
    """Index ranges of the pair list whose padded pixel blocks hold at most `budget` pairs."""
    n1, n2 = np.diff(off)[a], np.diff(off)[b]
    start = 0
    while start < len(a):
        end, m1, m2 = start, 0, 0
        while end < len(a):
            k1, k2 = max(m1, n1[end]), max(m2, n2[end])
            if end > start and (end + 1 - start) * k1 * k2 > budget:
                break
            m1, m2, end = k1, k2, end + 1
        yield start, end, int(m1), int(m2)
        start = end


def _gather(off, which, length, arrays):
    """Padded [pairs, length] views of per-pixel arrays, and which entries are pixels."""
    start, n = off[which], off[which + 1] - off[which]
    k = torch.arange(length, device=off.device)
    inside = k[None, :] < n[:, None]
    index = torch.where(inside, start[:, None] + k[None, :], 0)
    return inside, [x[index] for x in arrays]


def _separations(g, one, two, angle):
    """(r_par, r_trans, in range) of padded blocks of (r_comov, dist_m)."""
    c, s = torch.cos(angle / 2)[:, None, None], torch.sin(angle / 2)[:, None, None]
    r_par = (one[0][:, :, None] - two[0][:, None, :]) * c
    if not g.x_correlation:
        r_par = r_par.abs()
    r_trans = (one[1][:, :, None] + two[1][:, None, :]) * s
    ok = (r_par < g.r_par_max) & (r_trans < g.r_trans_max) & (r_par >= g.r_par_min)
    return r_par, r_trans, ok


def _flat_bin(g, r_par, r_trans, n_par, n_trans):
    span = g.r_par_max - g.r_par_min
    bp = torch.floor((r_par - g.r_par_min) / span * n_par)
    bt = torch.floor(r_trans / g.r_trans_max * n_trans)
    return (bt + n_trans * bp).long()


def _exact_xi(g, store, a, b, angle, flags, row, rows):
    if float(np.dot(np.diff(store.offsets)[a].astype(float),
                    np.diff(store.offsets)[b])) > EXACT_PIXEL_PAIRS:
        return None
    nb = g.num_bins_r_par * g.num_bins_r_trans
    off = _dev(store.offsets)
    pix = [_dev(x) for x in (store.r_comov, store.dist_m, store.z, store.weights,
                             store.delta * store.weights)]
    out = torch.zeros(5, rows * nb, dtype=torch.float64, device=off.device)
    count = torch.zeros(rows * nb, dtype=torch.int64, device=off.device)
    ta, tb, tang, trow = _dev(a).long(), _dev(b).long(), _dev(angle), _dev(row).long()
    tflag = _dev(flags).bool()
    width = (g.r_par_max - g.r_par_min) / g.num_bins_r_par
    for lo, hi, m1, m2 in _blocks(store.offsets, a, b):
        in1, one = _gather(off, ta[lo:hi], m1, pix)
        in2, two = _gather(off, tb[lo:hi], m2, pix)
        r_par, r_trans, ok = _separations(g, one, two, tang[lo:hi])
        ok &= (in1 & (one[3] != 0))[:, :, None] & (in2 & (two[3] != 0))[:, None, :]
        z = (one[2][:, :, None] + two[2][:, None, :]) / 2
        if g.z_min_pairs is not None:
            ok &= (z >= g.z_min_pairs) & (z <= g.z_max_pairs)
        if g.remove_same_half_plate_close_pairs:
            ok &= ~(tflag[lo:hi, None, None] & (r_par.abs() < width))
        w = (one[3][:, :, None] * two[3][:, None, :])[ok]
        wx = (one[4][:, :, None] * two[4][:, None, :])[ok]
        r_par, r_trans, z = r_par[ok], r_trans[ok], z[ok]
        flat = _flat_bin(g, r_par, r_trans, g.num_bins_r_par, g.num_bins_r_trans)
        flat += trow[lo:hi, None, None].expand_as(ok)[ok] * nb
        for k, v in enumerate((w, wx, r_par * w, r_trans * w, z * w)):
            out[k].index_add_(0, flat, v)
        count.index_add_(0, flat, torch.ones_like(flat))
    shape = (rows, nb) if rows > 0 else (nb,)
    return [x.reshape(shape).cpu().numpy() for x in out] + [
        count.reshape(shape).cpu().numpy()]


def _exact_xcf(case, seed):
    g, store, qso, forest, quasar, angle, row, rows = _xcf_inputs(case, seed)
    if np.diff(store.offsets)[forest].sum() > EXACT_PIXEL_PAIRS:
        return None
    n, nf = len(forest), store.num_forests
    # one one-pixel forest per quasar after the deltas; z, w and delta w of a quasar
    both = types.SimpleNamespace(
        offsets=np.concatenate([store.offsets, store.offsets[-1] + np.arange(1, nf + 1)]),
        r_comov=np.concatenate([store.r_comov, qso.r_comov]),
        dist_m=np.concatenate([store.dist_m, qso.dist_m]),
        z=np.concatenate([store.z, qso.z_qso]),
        weights=np.concatenate([store.weights, qso.weights]),
        delta=np.concatenate([store.delta, np.ones(nf)]))
    return _exact_xi(g, both, forest, nf + quasar, angle, np.zeros(n, np.uint8), row, rows)


def _exact_metal(case, seed):
    g, store, a, b, angle, _, tables, den = _metal_inputs(case, seed)
    if 2 * float(np.dot(np.diff(store.offsets)[a].astype(float),
                        np.diff(store.offsets)[b])) > EXACT_PIXEL_PAIRS:
        return None
    nb, nm = g.num_bins_r_par * g.num_bins_r_trans, (g.num_model_bins_r_par
                                                     * g.num_model_bins_r_trans)
    off = _dev(store.offsets)
    lya = [_dev(store.r_comov), _dev(store.dist_m)]
    dev = [[_dev(x) for x in t] for t in tables]
    wd = torch.zeros(nb, dtype=torch.float64, device=off.device)
    dm = torch.zeros(nb * nm, dtype=torch.float64, device=off.device)
    eff = torch.zeros(4, nm, dtype=torch.float64, device=off.device)
    counts = []
    ta, tb, tang = _dev(a).long(), _dev(b).long(), _dev(angle)
    for first, second in ((0, 1), (1, 0)):
        n_data = n_model = 0
        for lo, hi, m1, m2 in _blocks(store.offsets, a, b):
            in1, one = _gather(off, ta[lo:hi], m1, lya + dev[first])
            in2, two = _gather(off, tb[lo:hi], m2, lya + dev[second])
            r_par, r_trans, ok = _separations(g, one[:2], two[:2], tang[lo:hi])
            ok &= (in1 & (one[5] != 0))[:, :, None] & (in2 & (two[5] != 0))[:, None, :]
            m_par, m_trans, m_ok = _separations(g, one[3:5], two[3:5], tang[lo:hi])
            w = (one[5][:, :, None] * two[5][:, None, :])[ok]
            wz = w * (one[6][:, :, None] * two[6][:, None, :])[ok] / den
            z = ((one[2][:, :, None] + two[2][:, None, :]) / 2)[ok]
            flat = _flat_bin(g, r_par[ok], r_trans[ok], g.num_bins_r_par, g.num_bins_r_trans)
            wd.index_add_(0, flat, w)
            m_ok, m_par, m_trans = m_ok[ok], m_par[ok], m_trans[ok]
            n_data += flat.numel()
            flat, wz, z, m_par, m_trans = (x[m_ok] for x in (flat, wz, z, m_par, m_trans))
            n_model += flat.numel()
            model = _flat_bin(g, m_par, m_trans, g.num_model_bins_r_par,
                              g.num_model_bins_r_trans)
            dm.index_add_(0, flat * nm + model, wz)
            for k, v in enumerate((m_par * wz, m_trans * wz, z * wz, wz)):
                eff[k].index_add_(0, model, v)
        counts.append([n_data, n_model])
    return [wd.cpu().numpy(), dm.cpu().numpy()] + [x.cpu().numpy() for x in eff] + [
        np.array(counts)]


def _exact_dmat(case, seed):
    """The matrix of py/picca/cf.py:520-887 (forest x quasar: py/picca/xcf.py:427-658) pair by
    pair, with the continuum-fit terms as dense products; eta is the weighted sum over the
    pixels of the other forest in each model bin."""
    quasars = case["kind"] == "xdmat"
    g, store, a, b, angle, _ = (_xdmat_inputs if quasars else _kept_pairs)(case, seed)
    nb, nm = g.num_bins_r_par * g.num_bins_r_trans, (g.num_model_bins_r_par
                                                     * g.num_model_bins_r_trans)
    lengths = np.diff(store.offsets).astype(float)
    dense = 4.0 * nb * nm * float(np.sum(lengths[a] + (0 if quasars else lengths[b])))
    if dense > 1.0e14 or len(a) > 4000:
        return None
    off = store.offsets
    r, d, z, w, ll = (_dev(x) for x in (store.r_comov, store.dist_m, store.z, store.weights,
                                        store.log_lambda))
    zfa = ((1 + z) / (1 + g.z_ref)) ** (g.alpha - 1)
    zfb = ((1 + z) / (1 + g.z_ref)) ** (g.alpha2 - 1)
    f8 = dict(dtype=torch.float64, device=r.device)
    wd, dm, eff = torch.zeros(nb, **f8), torch.zeros(nb, nm, **f8), torch.zeros(4, nm, **f8)
    stats = [0, 0, 0, 0]
    for fa, fb, ang in zip(a, b, angle):
        sa, sb = slice(off[fa], off[fa + 1]), slice(off[fb], off[fb + 1])
        g_ang = torch.tensor([ang], **f8)
        r_par, r_trans, ok = (x[0] for x in _separations(
            g, (r[None, sa], d[None, sa]), (r[None, sb], d[None, sb]), g_ang))
        ok = ok & (w[sa] != 0)[:, None] & (w[sb] != 0)[None, :]
        i, j = torch.nonzero(ok, as_tuple=True)
        if quasars and not bool((r_par[ok] > g.r_par_min).any()):
            continue
        if i.numel() == 0:
            continue
        stats[0] += i.numel()
        stats[1] += i.numel()
        r_par, r_trans = r_par[ok], r_trans[ok]
        A = _flat_bin(g, r_par, r_trans, g.num_bins_r_par, g.num_bins_r_trans)
        M = _flat_bin(g, r_par, r_trans, g.num_model_bins_r_par, g.num_model_bins_r_trans)
        w1, w2 = w[sa], w[sb]
        w12 = w1[i] * w2[j]
        zf = zfa[sa][i] * zfb[sb][j]
        l1 = ll[sa] - (w1 * ll[sa]).sum() / w1.sum()
        l2 = ll[sb] - (w2 * ll[sb]).sum() / w2.sum()
        wd.index_add_(0, A, w12)
        for k, v in enumerate((r_par, r_trans, (z[sa][i] + z[sb][j]) / 2, torch.ones_like(w12))):
            eff[k].index_add_(0, M, v * w12)
        dm.view(-1).index_add_(0, A * nm + M, w12 * zf)

        def fold(size, index, bins, width, value):
            t = torch.zeros(size * width, **f8)
            return t.index_add_(0, index * width + bins, value).view(size, width)

        def project(index, n, inner):
            """- sum over the pixels of one forest of P (x) eta, order-0 and order-1 terms;
            `inner`: weight / norm of the other forest's pixel, for each order, and dll."""
            for weight, dll in inner:
                e = fold(n, index, M, nm, zf * weight)
                p = fold(n, index, A, nb, w12 * dll)
                dm.sub_(p.T @ e)

        one = torch.ones_like(w12)
        a_terms = [(w1[i] / w1.sum(), one), ((w1 * l1)[i] / (w1 * l1 ** 2).sum(), l1[i])]
        project(j, len(w2), a_terms)
        if quasars:
            continue
        b_terms = [(w2[j] / w2.sum(), one), ((w2 * l2)[j] / (w2 * l2 ** 2).sum(), l2[j])]
        project(i, len(w1), b_terms)
        for weight1, dll1 in a_terms:
            for weight2, dll2 in b_terms:
                e = torch.zeros(nm, **f8).index_add_(0, M, zf * weight1 * weight2)
                s = torch.zeros(nb, **f8).index_add_(0, A, w12 * dll1 * dll2)
                dm.add_(s[:, None] * e[None, :])
    return [wd.cpu().numpy(), dm.cpu().numpy()] + [x.cpu().numpy() for x in eff] + [
        np.array(stats)]


def _exact_wick(case, seed):
    """T[P, Q] as the sum of Wx1 E_P Wx2 over the pixel pairs of Q, with E_P the indicator of
    bin P; the products with a shared pixel replace one factor by w zev."""
    g, store, a, b, angle, zev, wx_off, wx = _wick_inputs(case, seed)
    nb = g.num_bins_r_par * g.num_bins_r_trans
    r, w, zv = _dev(store.r_comov), _dev(store.weights), _dev(zev)
    f8 = dict(dtype=torch.float64, device=r.device)
    weights, count = torch.zeros(nb, **f8), torch.zeros(nb, dtype=torch.int64, device=r.device)
    t1, t2, t3 = (torch.zeros(nb, nb, **f8) for _ in range(3))
    if len(a) * nb * float(np.mean(np.diff(store.offsets))) ** 3 > 3e13:
        return None
    for fa, fb, ang in zip(a, b, angle):
        sa = slice(store.offsets[fa], store.offsets[fa + 1])
        sb = slice(store.offsets[fb], store.offsets[fb + 1])
        x1, x2 = (_dev(wx[wx_off[f]:wx_off[f] + n * n].reshape(n, n)) for f, n in
                  ((fa, sa.stop - sa.start), (fb, sb.stop - sb.start)))
        r_par, r_trans, ok = (x[0] for x in _separations(
            g, (r[None, sa], r[None, sa]), (r[None, sb], r[None, sb]),
            torch.tensor([ang], **f8)))
        i, j = torch.nonzero(ok, as_tuple=True)
        p = _flat_bin(g, r_par[ok], r_trans[ok], g.num_bins_r_par, g.num_bins_r_trans)
        w12 = w[sa][i] * w[sb][j]
        weights.index_add_(0, p, w12)
        count.index_add_(0, p, torch.ones_like(p))
        v1, v2 = w[sa] * zv[sa], w[sb] * zv[sb]
        t1.view(-1).index_add_(0, p * nb + p, w12 * zv[sa][i] * zv[sb][j])
        o1, o2 = (x - torch.diag(torch.diagonal(x)) for x in (x1, x2))
        for k in torch.unique(p).tolist():
            e = torch.zeros(len(v1), len(v2), **f8)
            e[i[p == k], j[p == k]] = 1.0
            t2[k].index_add_(0, p, ((v1[:, None] * (e @ o2)) + (o1 @ e) * v2[None, :])[i, j])
            t3[k].index_add_(0, p, (o1 @ e @ o2)[i, j])
    return [weights.cpu().numpy(), count.cpu().numpy()] + [x.cpu().numpy()
                                                            for x in (t1, t2, t3)]


def _exact_cov(case, seed):
    xi, w = (_dev(x) for x in _cov_inputs(case, seed))
    total = w.sum(0)
    mean = (xi * w).sum(0)
    mean = torch.where(total > 0, mean / total, mean)
    y = w * (xi - mean)
    cov = y.T @ y
    norm = total[:, None] * total[None, :]
    return [torch.where(norm > 0, cov / norm, cov).cpu().numpy()]


def _exact_continuum(case, seed):
    """Damped Newton on chi2 + log terms for all forests at once, until no step lowers chi2."""
    c = _continuum_inputs(case, seed)
    n = case["forests"]
    seg = _dev(np.repeat(np.arange(n), np.diff(c["offsets"])))
    f, iv, x, eta, lss, fud = (_dev(c[k]) for k in ("flux", "ivar", "x", "eta", "var_lss",
                                                    "fudge"))
    m = _dev(np.interp(c["ll_rest"], c["grid"], c["nodes"]) * c["trans"])
    # the nodes' end intervals extend beyond them
    last = c["grid"][-1]
    beyond = c["ll_rest"] > last
    slope = (c["nodes"][-1] - c["nodes"][-2]) / (last - c["grid"][-2])
    m[_dev(beyond)] = _dev(c["nodes"][-1] + slope * (c["ll_rest"][beyond] - last))
    good = iv > 0
    seg_g, f_g, iv_g, x_g, m_g, eta_g, lss_g, fud_g = (
        v[good] for v in (seg, f, iv, x, m, eta, lss, fud))

    def sums(v):
        return torch.zeros(n, dtype=torch.float64, device=v.device).index_add_(0, seg_g, v)

    def chi2(a, b, derivatives):
        C = (a[seg_g] + b[seg_g] * x_g) * m_g
        D = eta_g / iv_g + lss_g * C ** 2 + fud_g * iv_g * C ** 4
        res = f_g - C
        value = sums(res ** 2 / D + torch.log(D))
        if not derivatives:
            return value
        D1 = 2 * lss_g * C + 4 * fud_g * iv_g * C ** 3
        D2 = 2 * lss_g + 12 * fud_g * iv_g * C ** 2
        t1 = -2 * res / D - res ** 2 * D1 / D ** 2 + D1 / D
        t2 = (2 / D + 4 * res * D1 / D ** 2 + 2 * res ** 2 * D1 ** 2 / D ** 3
              - res ** 2 * D2 / D ** 2 + D2 / D - D1 ** 2 / D ** 2)
        mx = m_g * x_g
        return (value, sums(t1 * m_g), sums(t1 * mx), sums(t2 * m_g ** 2), sums(t2 * m_g * mx),
                sums(t2 * mx ** 2))

    a, b = _dev(c["a0"]), _dev(c["b0"])
    lam = torch.zeros(n, dtype=torch.float64, device=f.device)
    for _ in range(25):
        value, ga, gb, haa, hab, hbb = chi2(a, b, True)
        haa, hbb = haa * (1 + lam), hbb * (1 + lam)
        det = haa * hbb - hab * hab
        fine = (haa > 0) & (det > 0)
        det = torch.where(fine, det, 1.0)
        da = torch.where(fine, -(hbb * ga - hab * gb) / det, 0.0)
        db = torch.where(fine, -(haa * gb - hab * ga) / det, 0.0)
        if not bool((-0.5 * (ga * da + gb * db) > 1e-16 * value.abs()).any()):
            break
        took = fine & (chi2(a + da, b + db, False) < value)
        a, b = torch.where(took, a + da, a), torch.where(took, b + db, b)
        lam = torch.where(took, lam * 0.1, torch.where(lam == 0, 1e-3, lam * 10.0))
        lam = torch.where(lam < 1e-9, 0.0, torch.clamp(lam, max=1e12))
    value = chi2(a, b, False)
    C = (b[seg] * x + a[seg]) * m
    negative = torch.zeros(n, dtype=torch.int64, device=f.device).index_add_(
        0, seg, (C < 0).long()) > 0
    status = torch.where(negative, 2, 0)
    keep = good & ~negative[seg]
    Ck, var = C[keep], 1.0 / iv[keep] / C[keep] ** 2
    wk = 1.0 / (eta[keep] * var + lss[keep] + fud[keep] / var)
    bins = _dev(c["bins"])[keep]
    stack = torch.zeros(2, len(c["grid"]), dtype=torch.float64, device=f.device)
    stack[0].index_add_(0, bins, f[keep] / (Ck + 1e-16) * wk)
    stack[1].index_add_(0, bins, wk)
    ndata = torch.zeros(n, dtype=torch.int64, device=f.device).index_add_(0, seg, good.long())
    return [a.cpu().numpy(), b.cpu().numpy(), value.cpu().numpy(),
            ndata.int().cpu().numpy(), status.int().cpu().numpy(), stack[0].cpu().numpy(),
            stack[1].cpu().numpy()]


def exact(case, seed):
    kind = case["kind"]
    if kind == "pair":
        g, one, two, angle = _one_pair(case, seed)
        store = types.SimpleNamespace(
            offsets=np.array([0, case["n1"], case["n1"] + case["n2"]]),
            **{name: np.concatenate([one[k], two[k]]) for k, name in
               enumerate(("z", "r_comov", "dist_m", "weights", "delta"))})
        out = _exact_xi(g, store, np.array([0]), np.array([1]), np.array([angle]),
                        np.zeros(1, np.uint8), np.zeros(1, np.int64), 1)
        return [x.reshape(-1) for x in out]
    if kind == "xi":
        g, store, pairs, row = _xi_inputs(case, seed)
        return _exact_xi(g, store, pairs.pair_a, pairs.pair_b, pairs.pair_ang,
                         pairs.pair_flags, row, _rows(case))
    return {"xcf": _exact_xcf, "dmat": _exact_dmat, "xdmat": _exact_dmat,
            "metal": _exact_metal, "wick": _exact_wick, "cov": _exact_cov,
            "continuum": _exact_continuum}[kind](case, seed)
