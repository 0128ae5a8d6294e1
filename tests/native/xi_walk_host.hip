// CPU harness of the pair kernel's run walk (test infrastructure, no product path).
//
// Runs the lane program of picca_amd/csrc/xi_walk.h -- the code the kernel runs -- on the
// host over a list of forest pairs, with the kernel's task split (64-pixel chunks of delta1,
// the pruned window of delta2, the same eligibility test) and every memory access checked
// against the forest's bounds.  Tasks the kernel would not walk are evaluated pair by pair
// with the reference's arithmetic.  The tests compare the result with the oracle, so the
// walk's keys, probes, prefix sums and edge pixels are checked on the CPU.
#include <algorithm>
#include <cmath>
#include <cstdint>
#include <cstring>
#include <vector>

#include "../../picca_amd/csrc/dmat_band.h"
#include "../../picca_amd/csrc/xi_const.h"
#include "../../picca_amd/csrc/xi_walk.h"

using picca::PrefixRecord;
using picca::XiConst;

namespace {

enum { ST_EDGE, ST_OVER, ST_WALK_TASKS, ST_PAIR_TASKS, ST_RUNS, ST_PROBES, ST_OOB, ST_COVER,
       ST_N };

struct Hist {
    std::vector<double> we, xi, rp, rt, z;
    std::vector<int64_t> nb;
    explicit Hist(size_t n) : we(n), xi(n), rp(n), rt(n), z(n), nb(n) {}
};

// Memory of one walk task: delta2's pixels [0, lb) and prefix entries [0, lb]; an access
// outside them is counted and answered with a harmless value.
struct HostMem {
    const double *rp_, *dp_, *wp_, *zp_, *dwp_;
    const picca::PrefixPair *pre_;
    int64_t lb;
    Hist *hist;
    int64_t *stats;

    bool bad(int p, int64_t n) {
        if (p < 0 || p >= n) {
            ++stats[ST_OOB];
            return true;
        }
        return false;
    }
    void rd(int p, double &rv, double &dv) {
        if (bad(p, lb)) {
            rv = dv = 0.0;
            return;
        }
        rv = rp_[p];
        dv = dp_[p];
    }
    PrefixRecord prefix(int p) {
        if (bad(p, lb + 1)) return PrefixRecord{0, 0, 0, 0, 0, 0};
        return picca::prefix_entry(pre_[p], pre_[lb + 1 + p], pre_[2 * (lb + 1) + p]);
    }
    double w(int p) { return bad(p, lb) ? 0.0 : wp_[p]; }
    double z(int p) { return bad(p, lb) ? 0.0 : zp_[p]; }
    double dw(int p) { return bad(p, lb) ? 0.0 : dwp_[p]; }
    void add(int bin, double we, double xi, double rp, double rt, double zz, uint32_t n) {
        if (bin < 0 || (size_t)bin >= hist->we.size()) {
            ++stats[ST_OOB];
            return;
        }
        hist->we[bin] += we;
        hist->xi[bin] += xi;
        hist->rp[bin] += rp;
        hist->rt[bin] += rt;
        hist->z[bin] += zz;
        hist->nb[bin] += n;
    }
    void flush(bool on, const picca::RunSums &r) {
        if (on) add(r.bin, r.we, r.xi, r.rp, r.rt, r.z, r.n);
    }
    bool any(bool v) { return v; }
    const picca::XiConst &consts(const picca::XiConst &C) { return C; }
    void pin(picca::RunSums &) {}
    void count_edge() { ++stats[ST_EDGE]; }
    void count_overflow() { ++stats[ST_OVER]; }
    void count_probe() { ++stats[ST_PROBES]; }
    void count_run(bool closed, uint32_t n) {
        if (!closed) return;
        ++stats[ST_RUNS];
        stats[ST_COVER] += (int64_t)n;
    }
};

bool monotone(const double *x, int64_t n) {
    for (int64_t k = 1; k < n; ++k)
        if (!(x[k] >= x[k - 1])) return false;
    return true;
}

// first index in [0, n) with arr[idx] >= x (strict) or arr[idx] > x, arr non-decreasing
int lower(const double *arr, int n, double x, bool strict) {
    int lo = 0, hi = n;
    while (lo < hi) {
        const int mid = (lo + hi) / 2;
        const bool below = strict ? arr[mid] < x : arr[mid] <= x;
        if (below) lo = mid + 1;
        else hi = mid;
    }
    return lo;
}

// One pixel pair with the reference's arithmetic (py/picca/cf.py:355-387), specialised
// case (XC: cross-correlation, the rows [C.row0, C.row0 + C.rows); shp: close pairs of one
// half plate removed); same edge / overflow conventions as the kernel.
template <bool XC>
void exact_pair(const XiConst &C, double r1, double d1, double zh1, double w1, double dw1,
                double r2, double d2, double z2, double w2, double dw2, double cos_half,
                double sin_half, bool shp, Hist &h, int64_t *stats) {
    const picca::WalkExact e = picca::walk_exact<XC>(C, r1, d1, r2, d2, cos_half, sin_half);
    if (!e.mine) return;
    const bool cut = shp && std::fabs(e.r_par) < C.width_p;
    if (e.edge) ++stats[ST_EDGE];
    if (e.over && !cut) ++stats[ST_OVER];
    const bool out = (e.r_par >= C.rpmax) | (e.r_trans >= C.rtmax) | (XC && e.r_par < C.rpmin);
    if (out || e.over || cut) return;
    int pbin;
    if (e.wrap) {
        pbin = e.pbin;
    } else {
        const int row = !XC && e.m >= 0 ? e.m : -e.m - 1;
        pbin = (row - C.row0) * C.ntp + e.c;
    }
    const double w12 = w1 * w2;
    h.we[pbin] += w12;
    h.xi[pbin] += dw1 * dw2;
    h.rp[pbin] += e.r_par * w12;
    h.rt[pbin] += e.r_trans * w12;
    h.z[pbin] += (zh1 + z2 * 0.5) * w12;
    h.nb[pbin] += 1;
}

// The launch of the kernel over the rows [row0, row0 + rows) of r_par; pflags: the pairs'
// same-half-plate flags (CUTS).
template <bool XC, bool CUTS>
int walk_launch(const picca_cf_params *params, int64_t num_forests, const int64_t *off,
                 const double *z, const double *r, const double *d, const double *w,
                 const double *delta, int64_t num_pairs, const int32_t *pa, const int32_t *pb,
                 const double *pang, const uint8_t *pflags, const int32_t *prow,
                 int32_t num_rows, int32_t schedule, int32_t row0, int32_t rows_n,
                 double *o_we, double *o_xi, double *o_rp, double *o_rt, double *o_z,
                 int64_t *o_nb, int64_t *stats) {
    XiConst C;
    int mode = 0;
    if (picca::fill_xi_const(params, C, mode) || !picca::xi_fast_path(params, mode) ||
        (!XC && !CUTS && !picca::xi_specialised(params, mode)))
        return -1;
    if (rows_n > 0) picca::set_xi_rows(C, row0, std::min(rows_n, C.np - row0));
    const int64_t npix = off[num_forests];
    double max_r = 0, max_d = 0;
    for (int64_t k = 0; k < npix; ++k) {
        max_r = std::fmax(max_r, std::fabs(r[k]));
        max_d = std::fmax(max_d, std::fabs(d[k]));
    }
    if (picca::widen_xi_margins(C, max_r, max_d)) return -1;
    picca::apply_xi_schedule(C, schedule);

    std::vector<double> dw((size_t)npix);
    for (int64_t k = 0; k < npix; ++k) dw[k] = delta[k] * w[k];
    std::vector<picca::PrefixPair> pre(picca::PREFIX_PLANES * (size_t)(npix + num_forests));
    std::vector<double> spc_r((size_t)num_forests), spc_d((size_t)num_forests);
    std::vector<uint8_t> mono((size_t)num_forests);
    std::vector<double> scratch;
    for (int64_t b = 0; b < num_forests; ++b) {
        const int64_t o = off[b], n = off[b + 1] - off[b];
        picca::build_walk_forest(r + o, d + o, z + o, w + o, dw.data() + o, n,
                                 pre.data() + picca::PREFIX_PLANES * (o + b), spc_r[b], spc_d[b]);
        mono[b] = (uint8_t)((monotone(r + o, n) ? 1 : 0) | (monotone(d + o, n) ? 2 : 0) |
                            (monotone(z + o, n) ? 4 : 0) |
                            picca::level_flags(w + o, dw.data() + o, n, scratch));
    }
    const bool z_cut = (C.flags & (picca::XI_HAS_ZMIN | picca::XI_HAS_ZMAX)) != 0;
    const double z_lo = (C.flags & picca::XI_HAS_ZMIN) ? C.zmin : -INFINITY;
    const double z_hi = (C.flags & picca::XI_HAS_ZMAX) ? C.zmax : INFINITY;
    const size_t nbp = (size_t)(C.rows + 1 + (C.row0 + C.rows < C.np ? 1 : 0)) * C.ntp;
    std::vector<Hist> rows;
    rows.reserve((size_t)num_rows);
    for (int32_t k = 0; k < num_rows; ++k) rows.emplace_back(nbp);

    for (int64_t p = 0; p < num_pairs; ++p) {
        const int a = pa[p], b = pb[p];
        const double ang = pang[p];
        const double cos_half = std::cos(ang / 2), sin_half = std::sin(ang / 2);
        Hist &h = rows[(size_t)prow[p]];
        const int64_t oa = off[a], ob = off[b];
        const int la = (int)(off[a + 1] - oa), lb = (int)(off[b + 1] - ob);
        // the kernel's task list: the chunks of delta1 xi_chunk_kernel keeps
        int first = 0, end = (la + 63) >> 6;
        if (cos_half > 0 && (mono[b] & 3) == 3 && (mono[a] & 1) && la > 0 && lb > 0) {
            const double reach = std::fmax(C.rpmax, std::fabs(C.rpmin)) / cos_half;
            const double slack = 8.0 * C.edge_tol / cos_half + 2e-6;
            double lo = r[ob] + (XC ? C.prune_lo / cos_half : -reach);
            double hi = r[ob + lb - 1] + (XC ? C.prune_hi / cos_half : reach);
            lo -= slack + 2e-12 * std::fabs(lo);
            hi += slack + 2e-12 * std::fabs(hi);
            const int i_lo = lower(r + oa, la, lo, true);
            int i_hi = lower(r + oa, la, hi, false);
            if (sin_half > 0 && (mono[a] & 2)) {
                double d_lim = (C.rtmax + 8.0 * C.edge_tol) / sin_half - d[ob];
                d_lim += 2e-6 + 2e-12 * std::fabs(d_lim);
                i_hi = std::min(i_hi, lower(d + oa, la, d_lim, false));
            }
            first = i_lo >= i_hi ? 0 : i_lo >> 6;
            end = i_lo >= i_hi ? 0 : (i_hi + 63) >> 6;
        }
        for (int chunk = first; chunk < end; ++chunk) {
            const int i0 = chunk * 64, i1 = std::min(la, i0 + 64);
            double r_min = INFINITY, r_max = -INFINITY, d_min = INFINITY;
            bool any = false;
            for (int i = i0; i < i1; ++i) {
                if (w[oa + i] == 0) continue;
                any = true;
                r_min = std::fmin(r_min, r[oa + i]);
                r_max = std::fmax(r_max, r[oa + i]);
                d_min = std::fmin(d_min, d[oa + i]);
            }
            if (!any) continue;
            int j_lo = 0, j_hi = lb;
            bool pruned = false;
            if (cos_half > 0 && (mono[b] & 3) == 3) {
                pruned = true;
                const double slack = 4.0 * C.edge_tol / cos_half + 1e-6;
                double lo_r = r_min - (XC ? C.prune_hi : C.rpmax) / cos_half;
                double hi_r = XC ? r_max - C.prune_lo / cos_half : r_max + C.rpmax / cos_half;
                lo_r -= slack + 1e-12 * std::fabs(lo_r);
                hi_r += slack + 1e-12 * std::fabs(hi_r);
                j_lo = lower(r + ob, lb, lo_r, true);
                j_hi = lower(r + ob, lb, hi_r, false);
                if (sin_half > 0) {
                    double d_lim = (C.rtmax + 4.0 * C.edge_tol) / sin_half - d_min;
                    d_lim += 1e-6 + 1e-12 * std::fabs(d_lim);
                    const int j_d = lower(d + ob, lb, d_lim, false);
                    if (j_d < j_hi) j_hi = j_d;
                }
            }
            // an empty window: the kernel returns before choosing a loop
            if (j_lo >= j_hi) continue;
            const double cp = cos_half * C.inv_p, st = sin_half * C.inv_t;
            double q0 = 1.0;
            if (j_hi - j_lo >= 2) {
                const double span = (r[ob + j_hi - 1] - r[ob + j_lo]) * cp;
                if (span > 0) q0 = (double)(j_hi - 1 - j_lo) / span;
            }
            const bool shp = CUTS && (C.flags & picca::XI_REMOVE_SHP) &&
                             (pflags[p] & picca::PAIR_SAME_HALF_PLATE);
            const int level = picca::FOREST_LEVEL_W | picca::FOREST_LEVEL_DW;
            const bool cuts_ok = !(XC && shp) && (!z_cut || (mono[b] & 4)) &&
                                 (!(XC || CUTS) || (mono[b] & level) == level);
            const bool walk = pruned && cuts_ok && picca::walk_task(C, spc_r[b], spc_d[b], cp, st, q0);
            if (walk) {
                ++stats[ST_WALK_TASKS];
                picca::WalkTask T;
                T.cos_half = cos_half;
                T.sin_half = sin_half;
                T.cp = cp;
                T.st = st;
                T.rc = r[ob + (lb >> 1)];
                T.dc = d[ob + (lb >> 1)];
                T.j_lo = j_lo;
                T.j_hi = j_hi;
                T.q0 = q0;
                HostMem mem;
                mem.rp_ = r + ob;
                mem.dp_ = d + ob;
                mem.wp_ = w + ob;
                mem.zp_ = z + ob;
                mem.dwp_ = dw.data() + ob;
                mem.pre_ = pre.data() + picca::PREFIX_PLANES * (ob + b);
                mem.lb = lb;
                mem.hist = &h;
                mem.stats = stats;
                for (int i = i0; i < i1; ++i) {
                    if (w[oa + i] == 0) continue;
                    picca::WalkLane L{r[oa + i], d[oa + i], z[oa + i] * 0.5, w[oa + i],
                                      dw[oa + i]};
                    T.shp = shp;
                    if (CUTS) {
                        // the kernel's binary searches of the pair-redshift cut
                        L.j_lo = j_lo;
                        while (L.j_lo < j_hi && L.zh1 + z[ob + L.j_lo] * 0.5 < z_lo) ++L.j_lo;
                        L.j_hi = L.j_lo;
                        while (L.j_hi < j_hi && !(L.zh1 + z[ob + L.j_hi] * 0.5 > z_hi)) ++L.j_hi;
                        if (L.j_lo >= L.j_hi) continue;
                    }
                    picca::walk_lane<XC, CUTS>(C, T, L, mem, true);
                }
            } else {
                ++stats[ST_PAIR_TASKS];
                for (int i = i0; i < i1; ++i) {
                    if (w[oa + i] == 0) continue;
                    for (int j = j_lo; j < j_hi; ++j) {
                        if (w[ob + j] == 0) continue;
                        const double zp = z[oa + i] * 0.5 + z[ob + j] * 0.5;
                        if (CUTS && (zp < z_lo || zp > z_hi)) continue;
                        exact_pair<XC>(C, r[oa + i], d[oa + i], z[oa + i] * 0.5, w[oa + i],
                                   dw[oa + i], r[ob + j], d[ob + j], z[ob + j], w[ob + j],
                                   dw[ob + j], cos_half, sin_half, shp, h, stats);
                    }
                }
            }
        }
    }
    // padded layout -> flat rows
    for (int32_t row = 0; row < num_rows; ++row) {
        const Hist &h = rows[(size_t)row];
        // (column 0 of the row after the launch's: pairs whose r_trans bin rounds to nt)
        const int bins = C.rows * C.nt + (C.row0 + C.rows < C.np ? 1 : 0);
        for (int k = 0; k < bins; ++k) {
            const int kp = k + k / C.nt;
            const size_t o = (size_t)row * C.nb + C.row0 * C.nt + k;
            o_we[o] += h.we[kp];
            o_xi[o] += h.xi[kp];
            o_rp[o] += h.rp[kp];
            o_rt[o] += h.rt[kp];
            o_z[o] += h.z[kp];
            o_nb[o] += h.nb[kp];
        }
    }
    return 0;
}

}  // namespace

extern "C" {

// The walk's guess reciprocal (walk_rcp_guess), for its unit test.
double xi_walk_rcp_guess(double x) { return picca::walk_rcp_guess(x); }

// A forest's level_flags.
int xi_level_flags(int n, const double *w, const double *dw) {
    std::vector<double> scratch;
    return picca::level_flags(w, dw, n, scratch);
}

// The banded distortion matrix's keys and edges (dmat_band.h) of one pixel along a partner of n
// rising values v (kind: BAND_*; from: r_par_min of BAND_SIGNED).  keys[k]: of pixel k; edges[k]: first pixel
// whose key is at least k_lo + k.  The index table is made as the table kernel makes it.
void dmat_band_host(int kind, double from, int n, const double *v, double self, double scale, double range,
                    int bins, double margin, int *keys, int k_lo, int num, int *edges) {
    const double mul = scale * bins / range;
    const picca::BandAxis A =
        kind == picca::BAND_SIGNED
            ? picca::band_signed_axis(self, mul, scale, from, range, bins, margin)
        : kind == picca::BAND_PAR ? picca::band_par_axis(self, mul, scale, range, bins, margin)
                                  : picca::band_trans_axis(self, mul, scale, range, bins, margin);
    const double h = picca::band_mean_step(v[0], v[n - 1], n);
    std::vector<int32_t> first((size_t)n);
    for (int k = 0; k < n; ++k) first[(size_t)k] = lower(v, n, v[0] + k * h, true);
    const picca::BandTable T{first.data(), v[0], 1.0 / h, n};
    for (int k = 0; k < n; ++k) keys[k] = picca::band_key(A, v[k]);
    for (int k = 0; k < num; ++k)
        edges[k] = picca::band_edge(A, T, [&](int p) { return v[p]; }, k_lo + k);
}

// Correlation of the listed forest pairs (specialised case of the pair kernel only).
// Outputs are [num_rows * np * nt] each, added to; stats = edge, overflow, walked tasks,
// pair-by-pair tasks, runs, probes, out-of-bounds accesses, pixel pairs covered by runs.
// Returns 0, or -1 when the parameters are not the specialised case.
int xi_walk_host(const picca_cf_params *params, int64_t num_forests, const int64_t *off,
                 const double *z, const double *r, const double *d, const double *w,
                 const double *delta, int64_t num_pairs, const int32_t *pa, const int32_t *pb,
                 const double *pang, const int32_t *prow, int32_t num_rows, int32_t schedule,
                 double *o_we, double *o_xi, double *o_rp, double *o_rt, double *o_z,
                 int64_t *o_nb, int64_t *stats) {
    std::memset(stats, 0, sizeof(int64_t) * ST_N);
    return walk_launch<false, false>(params, num_forests, off, z, r, d, w, delta, num_pairs, pa,
                                     pb, pang, nullptr, prow, num_rows, schedule, 0, 0, o_we,
                                     o_xi, o_rp, o_rt, o_z, o_nb, stats);
}

// The same for the cross-correlation and the cuts (no zerr cut), in launches of `share` rows
// of r_par (the cross-correlation) or one launch.
int xi_walk_host_cuts(const picca_cf_params *params, int64_t num_forests, const int64_t *off,
                      const double *z, const double *r, const double *d, const double *w,
                      const double *delta, int64_t num_pairs, const int32_t *pa,
                      const int32_t *pb, const double *pang, const uint8_t *pflags,
                      const int32_t *prow, int32_t num_rows, int32_t share, double *o_we,
                      double *o_xi, double *o_rp, double *o_rt, double *o_z, int64_t *o_nb,
                      int64_t *stats) {
    std::memset(stats, 0, sizeof(int64_t) * ST_N);
    const bool xc = params->x_correlation != 0;
    const int np = params->num_bins_r_par;
    if (params->has_zerr_cut) return -1;
    const int step = xc ? share : np;
    for (int row0 = 0; row0 < np; row0 += step) {
        auto launch = xc ? walk_launch<true, true> : walk_launch<false, true>;
        const int rc = launch(params, num_forests, off, z, r, d, w, delta, num_pairs, pa, pb,
                              pang, pflags, prow, num_rows, PICCA_XI_SCHEDULE_RUNS, row0, step,
                              o_we, o_xi, o_rp, o_rt, o_z, o_nb, stats);
        if (rc) return rc;
    }
    return 0;
}

}  // extern "C"
