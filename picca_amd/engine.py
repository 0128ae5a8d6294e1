"""Python handle on one device context of the HIP engine.

``Engine`` owns a ``picca_ctx`` (device buffers + stream).  It keeps one forest store and
one xi pair list resident in HBM, so repeated executions (benchmarks, several parameter
sets on the same pairs) do not re-upload them.
"""
import ctypes
import math

import numpy as np

from . import _native
from ._native import as_f64, as_i32, as_i64, as_u8, check, ptr

DEFAULT_EDGE_TOL = 1e-9  # Mpc/h (r_par, r_trans) distance that makes a pair an edge pair


def params_from_globals(module, edge_tol=DEFAULT_EDGE_TOL):
    """Fill picca_cf_params from an object carrying the cf module globals."""
    p = _native.CfParams()

    def get(name, default=None):
        return getattr(module, name, default)

    p.num_bins_r_par = int(get("num_bins_r_par"))
    p.num_bins_r_trans = int(get("num_bins_r_trans"))
    p.num_model_bins_r_par = int(get("num_model_bins_r_par") or 0)
    p.num_model_bins_r_trans = int(get("num_model_bins_r_trans") or 0)
    p.r_par_min = float(get("r_par_min"))
    p.r_par_max = float(get("r_par_max"))
    p.r_trans_max = float(get("r_trans_max"))
    z_min_pairs = get("z_min_pairs")
    z_max_pairs = get("z_max_pairs")
    p.has_z_min_pairs = int(z_min_pairs is not None)
    p.has_z_max_pairs = int(z_max_pairs is not None)
    p.z_min_pairs = float(z_min_pairs) if z_min_pairs is not None else math.nan
    p.z_max_pairs = float(z_max_pairs) if z_max_pairs is not None else math.nan
    zerr_deg = get("zerr_cut_deg")
    zerr_kms = get("zerr_cut_kms")
    p.has_zerr_cut = int(zerr_deg is not None)
    p.zerr_cut_deg = float(zerr_deg) if zerr_deg is not None else math.nan
    p.zerr_cut_kms = float(zerr_kms) if zerr_kms is not None else math.nan
    for name in ("z_ref", "alpha", "alpha2"):
        value = get(name)
        setattr(p, name, float(value) if value is not None else math.nan)
    p.edge_tol = float(edge_tol)
    p.x_correlation = int(bool(get("x_correlation", False)))
    p.rmu_binning = int(bool(get("rmu_binning", False)))
    p.ang_correlation = int(bool(get("ang_correlation", False)))
    p.remove_same_half_plate_close_pairs = int(bool(get("remove_same_half_plate_close_pairs",
                                                        False)))
    p.redshift_evolution = int(bool(get("redshift_evolution_in_distortion_matrix", True)))
    return p


class XiResult:
    """Un-normalised per-row sums of one xi execution, arrays of shape [num_rows, nb]."""

    def __init__(self, weights, xi, r_par, r_trans, z, num_pairs, report):
        self.weights = weights
        self.xi = xi
        self.r_par = r_par
        self.r_trans = r_trans
        self.z = z
        self.num_pairs = num_pairs
        self.report = report

    def normalised(self):
        """Per-row (weights, xi, r_par, r_trans, z, num_pairs), divided like
        ``py/picca/cf.py:242-246``."""
        we = self.weights.copy()
        out = []
        for arr in (self.xi, self.r_par, self.r_trans, self.z):
            arr = arr.copy()
            mask = we > 0
            arr[mask] /= we[mask]
            out.append(arr)
        return (we, out[0], out[1], out[2], out[3], self.num_pairs.copy())


class Engine:
    """One HIP device context."""

    def __init__(self, device=0):
        self._lib = _native.load()
        handle = ctypes.c_void_p()
        check(self._lib.picca_create(int(device), ctypes.byref(handle)), "picca_create")
        self._ctx = handle
        self.device = device
        self._store_key = None
        self._pairs_key = None
        self.num_rows = 0
        self.num_pairs = 0

    def close(self):
        if self._ctx:
            self._lib.picca_destroy(self._ctx)
            self._ctx = None

    def __del__(self):
        try:
            self.close()
        except Exception:
            pass

    # -- forest store ---------------------------------------------------------
    def set_forests(self, store, key=None):
        """Upload a ForestStore (skipped when ``key`` matches the resident store)."""
        if key is not None and key == self._store_key:
            return
        ll = store.log_lambda
        self._hold_store = (as_i64(store.offsets), as_f64(store.z), as_f64(store.r_comov),
                            as_f64(store.dist_m), as_f64(store.weights),
                            as_f64(store.delta), None if ll is None else as_f64(ll),
                            as_f64(store.z_qso), as_i32(store.order))
        off, z, r, d, w, delta, ll, zq, order = self._hold_store
        status = self._lib.picca_set_forests(
            self._ctx, store.num_forests, ptr(off), ptr(z), ptr(r), ptr(d), ptr(w),
            ptr(delta), ptr(ll), ptr(zq), ptr(order))
        check(status, "picca_set_forests")
        self._hold_store = None
        self._store_key = key
        self._pairs_key = None

    # -- xi -------------------------------------------------------------------
    def set_xi_pairs(self, pair_a, pair_b, pair_ang, pair_flags, pair_row, num_rows, key=None):
        if key is not None and key == self._pairs_key:
            return
        a = as_i32(pair_a)
        b = as_i32(pair_b)
        ang = as_f64(pair_ang)
        flags = as_u8(pair_flags)
        row = as_i32(pair_row)
        status = self._lib.picca_xi_set_pairs(self._ctx, len(a), ptr(a), ptr(b), ptr(ang),
                                              ptr(flags), ptr(row), int(num_rows))
        check(status, "picca_xi_set_pairs")
        self.num_rows = int(num_rows)
        self.num_pairs = len(a)
        self._pairs_key = key

    def xcf_set_pairs(self, pair_forest, obj_r, obj_d, obj_z, obj_w, pair_ang, pair_row,
                      num_rows, angular=False):
        f = as_i32(pair_forest)
        arrays = [as_f64(a) for a in (obj_r, obj_d, obj_z, obj_w, pair_ang)]
        row = as_i32(pair_row)
        check(self._lib.picca_xcf_set_pairs(self._ctx, len(f), ptr(f), *(ptr(a) for a in arrays),
                                            ptr(row), int(num_rows), int(bool(angular))),
              "picca_xcf_set_pairs")
        self.num_rows = int(num_rows)

    def xcf(self, params):
        report = _native.XiReport()
        check(self._lib.picca_xcf_execute(self._ctx, ctypes.byref(params), ctypes.byref(report)),
              "picca_xcf_execute")
        (we, xi, rp, rt, z), nb = self.xi_download(params)
        return XiResult(we, xi, rp, rt, z, nb, report.as_dict())

    def use_xi_graph(self, on):
        """Launch xi through its captured HIP graph (default) or directly."""
        check(self._lib.picca_xi_use_graph(self._ctx, int(bool(on))), "picca_xi_use_graph")

    def set_xi_schedule(self, schedule):
        """Schedule of the specialised pair kernel: _native.XI_SCHEDULE_AUTO, _PAIRS or
        _RUNS (picca_xi_set_schedule)."""
        check(self._lib.picca_xi_set_schedule(self._ctx, int(schedule)),
              "picca_xi_set_schedule")

    def xi_execute(self, params):
        report = _native.XiReport()
        check(self._lib.picca_xi_execute(self._ctx, ctypes.byref(params), ctypes.byref(report)),
              "picca_xi_execute")
        return report

    def xi_download(self, params):
        nb = params.num_bins_r_par * params.num_bins_r_trans
        shape = (self.num_rows, nb)
        out = [np.zeros(shape) for _ in range(5)]
        num_pairs = np.zeros(shape, dtype=np.int64)
        check(self._lib.picca_xi_download(self._ctx, *(ptr(a) for a in out), ptr(num_pairs)),
              "picca_xi_download")
        return out, num_pairs

    def xi(self, params):
        report = self.xi_execute(params)
        (we, xi, rp, rt, z), nb = self.xi_download(params)
        return XiResult(we, xi, rp, rt, z, nb, report.as_dict())

    # -- continuum fit --------------------------------------------------------
    def cont_set_forests(self, offsets, flux, ivar, mean_cont, x, eta, var_lss, fudge, order):
        offsets = as_i64(offsets)
        arrays = [as_f64(a) for a in (flux, ivar, mean_cont, x, eta, var_lss, fudge)]
        order = as_i32(order)
        check(self._lib.picca_cont_set_forests(self._ctx, len(offsets) - 1, ptr(offsets),
                                               *(ptr(a) for a in arrays), ptr(order)),
              "picca_cont_set_forests")
        self._cont_forests = len(offsets) - 1

    def cont_fit(self, a0, b0, max_iter=100, tol=1e-12, use_constant_weight=False, tol_abs=0.0):
        """Fit every resident forest from (a0, b0).  Returns a dict of arrays a, b, chi2,
        ndata, status, evaluations and the kernel time kernel_ms."""
        n = self._cont_forests
        a0 = as_f64(a0)
        b0 = as_f64(b0)
        if len(a0) != n or len(b0) != n:
            raise ValueError("one start value per forest is needed")
        params = _native.ContParams(int(max_iter), int(bool(use_constant_weight)), float(tol),
                                    float(tol_abs))
        out = {"a": np.zeros(n), "b": np.zeros(n), "chi2": np.zeros(n),
               "ndata": np.zeros(n, np.int32), "status": np.zeros(n, np.int32),
               "evaluations": np.zeros(n, np.int32)}
        ms = ctypes.c_double()
        check(self._lib.picca_cont_fit(self._ctx, ctypes.byref(params), ptr(a0), ptr(b0),
                                       ptr(out["a"]), ptr(out["b"]), ptr(out["chi2"]),
                                       ptr(out["ndata"]), ptr(out["status"]),
                                       ptr(out["evaluations"]), ctypes.byref(ms)),
              "picca_cont_fit")
        out["kernel_ms"] = ms.value
        return out

    def cont_set_rest_frame(self, log_lambda_rest, transmission, bins, num_bins):
        """Per-pixel rest-frame log lambda, transmission correction and rest-frame bin of
        the resident continuum forests."""
        llr = as_f64(log_lambda_rest)
        trans = as_f64(transmission)
        bins = np.ascontiguousarray(bins, dtype=np.int32)
        check(self._lib.picca_cont_set_rest_frame(self._ctx, ptr(llr), ptr(trans), ptr(bins),
                                                  int(num_bins)), "picca_cont_set_rest_frame")
        self._cont_nbins = int(num_bins)

    def cont_stack(self, num_bins):
        """Weighted F / C stack of the last fit: (sum_ratio, sum_weight, kernel_ms)."""
        total = np.zeros(num_bins)
        weight = np.zeros(num_bins)
        ms = ctypes.c_double()
        check(self._lib.picca_cont_stack(self._ctx, ptr(total), ptr(weight), ctypes.byref(ms)),
              "picca_cont_stack")
        return total, weight, ms.value

    def cont_set_mean_cont(self, x, y):
        """Interpolate the mean continuum nodes to every pixel; returns the kernel ms."""
        x = as_f64(x)
        y = as_f64(y)
        ms = ctypes.c_double()
        check(self._lib.picca_cont_set_mean_cont(self._ctx, len(x), ptr(x), ptr(y),
                                                 ctypes.byref(ms)), "picca_cont_set_mean_cont")
        return ms.value

    def diag_copy(self, nbytes):
        """Plain device copy of nbytes (multiple of 16); returns the kernel time in ms."""
        ms = ctypes.c_double()
        check(self._lib.picca_diag_copy(self._ctx, int(nbytes), ctypes.byref(ms)),
              "picca_diag_copy")
        return ms.value

    # -- dmat -----------------------------------------------------------------
    def dmat(self, params, pair_a, pair_b, pair_ang, pair_flags):
        nb = params.num_bins_r_par * params.num_bins_r_trans
        nm = params.num_model_bins_r_par * params.num_model_bins_r_trans
        weights_dmat = np.zeros(nb)
        dmat = np.zeros(nb * nm)
        r_par_eff = np.zeros(nm)
        r_trans_eff = np.zeros(nm)
        z_eff = np.zeros(nm)
        weight_eff = np.zeros(nm)
        stats = np.zeros(4, dtype=np.int64)
        a = as_i32(pair_a)
        b = as_i32(pair_b)
        ang = as_f64(pair_ang)
        flags = as_u8(pair_flags)
        status = self._lib.picca_dmat_run(
            self._ctx, ctypes.byref(params), len(a), ptr(a), ptr(b), ptr(ang), ptr(flags),
            ptr(weights_dmat), ptr(dmat), ptr(r_par_eff), ptr(r_trans_eff), ptr(z_eff),
            ptr(weight_eff), ptr(stats))
        check(status, "picca_dmat_run")
        return (weights_dmat, dmat.reshape(nb, nm), r_par_eff, r_trans_eff, z_eff, weight_eff,
                stats)

    def dmat_report(self):
        """Kernel times and matrix-core work of the last dmat() call (a dict)."""
        rep = _native.DmatReport()
        check(self._lib.picca_dmat_last_report(self._ctx, ctypes.byref(rep)),
              "picca_dmat_last_report")
        return rep.as_dict()

    def dmat_routes(self):
        """Pairs of the last dmat() call by the kernels they took (picca_dmat_last_routes)."""
        routes = np.zeros(len(_native.DMAT_ROUTES), dtype=np.int64)
        check(self._lib.picca_dmat_last_routes(self._ctx, ptr(routes)), "picca_dmat_last_routes")
        return dict(zip(_native.DMAT_ROUTES, (int(n) for n in routes)))

    def set_dmat_workspace(self, batch_bytes=_native.DMAT_BATCH_BYTES, prefix_bytes=2 ** 63 - 1):
        """Device memory that dmat() may take (picca_dmat_set_workspace)."""
        check(self._lib.picca_dmat_set_workspace(self._ctx, int(batch_bytes), int(prefix_bytes)),
              "picca_dmat_set_workspace")

    # -- subsampling covariance --------------------------------------------------
    def cov_subsample(self, xi, weights):
        """compute_cov of the rows of xi [num_samples, num_bins]; returns
        (covariance [num_bins, num_bins], total kernel ms, matrix-product kernel ms)."""
        xi = np.ascontiguousarray(xi, dtype=np.float64)
        weights = np.ascontiguousarray(weights, dtype=np.float64)
        if xi.ndim != 2 or xi.shape != weights.shape:
            raise ValueError("xi and weights must be 2-d arrays of one shape")
        ns, nb = xi.shape
        cov = np.zeros((nb, nb))
        ms = np.zeros(2)
        check(self._lib.picca_cov_subsample(self._ctx, ns, nb, ptr(xi), ptr(weights), ptr(cov),
                                            ptr(ms)), "picca_cov_subsample")
        return cov, float(ms[0]), float(ms[1])

    # -- Wick covariance terms ---------------------------------------------------
    def wick_t123(self, params, pair_a, pair_b, pair_ang, zev1, zev2, wx_offsets, wx):
        """T1, T2, T3 of the resident store's pairs; returns (weights_wick, num_pairs_wick,
        t1, t2, t3 [nb, nb], report dict)."""
        nb = params.num_bins_r_par * params.num_bins_r_trans
        a = as_i32(pair_a)
        b = as_i32(pair_b)
        ang = as_f64(pair_ang)
        zev1 = as_f64(zev1)
        zev2 = as_f64(zev2)
        wx_offsets = as_i64(wx_offsets)
        wx = as_f64(wx)
        weights_wick = np.zeros(nb)
        num_pairs_wick = np.zeros(nb, dtype=np.int64)
        t = [np.zeros(nb * nb) for _ in range(3)]
        report = _native.WickReport()
        check(self._lib.picca_wick_t123(self._ctx, ctypes.byref(params), len(a), ptr(a), ptr(b),
                                        ptr(ang), ptr(zev1), ptr(zev2), ptr(wx_offsets),
                                        len(wx), ptr(wx), ptr(weights_wick),
                                        ptr(num_pairs_wick), *(ptr(x) for x in t),
                                        ctypes.byref(report)), "picca_wick_t123")
        return (weights_wick, num_pairs_wick, t[0].reshape(nb, nb), t[1].reshape(nb, nb),
                t[2].reshape(nb, nb), report.as_dict())

    # -- metal distortion matrix -------------------------------------------------
    def metal_set_absorber(self, slot, z, r_comov, dist_m, weights, zfac):
        """One absorber's view of every pixel of the resident store (store order)."""
        arrays = [as_f64(a) for a in (z, r_comov, dist_m, weights, zfac)]
        check(self._lib.picca_metal_set_absorber(self._ctx, int(slot),
                                                 *(ptr(a) for a in arrays)),
              "picca_metal_set_absorber")

    def metal_pass(self, params, mode, slot_a, slot_b, zw_den, pair_a, pair_b, pair_ang,
                   pair_flags, out):
        """One absorber pass over the kept pairs, accumulated into
        out = (weights_dmat, dmat (flat), r_par_eff, r_trans_eff, z_eff, weight_eff).
        Returns the pass report as a dict."""
        a = as_i32(pair_a)
        b = as_i32(pair_b)
        ang = as_f64(pair_ang)
        flags = as_u8(pair_flags)
        for arr in out:
            if arr.dtype != np.float64 or not arr.flags["C_CONTIGUOUS"]:
                raise ValueError("metal outputs must be contiguous float64 arrays")
        report = _native.MetalReport()
        check(self._lib.picca_metal_pass(self._ctx, ctypes.byref(params), int(mode),
                                         int(slot_a), int(slot_b), float(zw_den), len(a),
                                         ptr(a), ptr(b), ptr(ang), ptr(flags),
                                         *(ptr(x) for x in out), ctypes.byref(report)),
              "picca_metal_pass")
        return report.as_dict()


_ENGINES = {}


def get_engine(device=0):
    """Process-wide engine of ``device`` (created on first use)."""
    engine = _ENGINES.get(device)
    if engine is None:
        engine = Engine(device)
        _ENGINES[device] = engine
    return engine


def device_info(device=0):
    lib = _native.load()
    name = ctypes.create_string_buffer(256)
    cus = ctypes.c_int32()
    lds = ctypes.c_int64()
    mem = ctypes.c_int64()
    check(lib.picca_device_info(int(device), name, 256, ctypes.byref(cus), ctypes.byref(lds),
                                ctypes.byref(mem)), "picca_device_info")
    return {"name": name.value.decode(), "num_cus": cus.value, "lds_per_cu": lds.value,
            "global_mem": mem.value}
