// CPU harness of the run walk's smallest memory interface (test infrastructure, no product
// path): prefix sums as records, no constants of the memory's own, closed runs counted one by
// one.  One pixel of delta1 against a whole delta2.
#include <cstdint>
#include <vector>

#include "../../picca_amd/csrc/xi_const.h"
#include "../../picca_amd/csrc/xi_walk.h"

namespace {

struct RecordMem {
    const double *r_, *d_, *w_, *z_, *dw_;
    const picca::PrefixRecord *pre;
    double *out;   // [bins][5]
    int64_t *runs;

    void rd(int p, double &r, double &d) {
        r = r_[p];
        d = d_[p];
    }
    picca::PrefixRecord prefix(int p) { return pre[p]; }
    double w(int p) { return w_[p]; }
    double z(int p) { return z_[p]; }
    double dw(int p) { return dw_[p]; }
    void add(int bin, double we, double xi, double rp, double rt, double z, uint32_t) {
        const double v[5] = {we, xi, rp, rt, z};
        for (int c = 0; c < 5; ++c) out[5 * bin + c] += v[c];
    }
    void flush(bool on, const picca::RunSums &r) {
        if (on) add(r.bin, r.we, r.xi, r.rp, r.rt, r.z, r.n);
    }
    bool any(bool v) { return v; }
    void pin(picca::RunSums &) {}
    void count_edge() {}
    void count_overflow() {}
    void count_probe() {}
    void count_run(uint32_t) { ++*runs; }
};

}  // namespace

extern "C" {

// Sums (weight, xi, r_par, r_trans, z) per padded bin [(np + 1) * (nt + 1)][5] of pixel (r1, d1,
// z1, w1, delta1) with delta2's n pixels; pre: n + 1 records, also returned as [n + 1][6].
// Returns the runs closed, or -1 when the parameters are not the specialised case.
int64_t xi_walk_records(const picca_cf_params *params, double ang, const double *pixel1, int n,
                        const double *r, const double *d, const double *z, const double *w,
                        const double *delta, double *out, double *records) {
    picca::XiConst C;
    int mode = 0;
    if (picca::fill_xi_const(params, C, mode) || !picca::xi_specialised(params, mode) ||
        picca::widen_xi_margins(C, r[n - 1], d[n - 1]))
        return -1;
    picca::apply_xi_schedule(C, PICCA_XI_SCHEDULE_RUNS);
    std::vector<double> dw((size_t)n);
    for (int k = 0; k < n; ++k) dw[k] = delta[k] * w[k];
    std::vector<picca::PrefixRecord> pre((size_t)n + 1);
    double spc_r = 0, spc_d = 0;
    picca::build_walk_forest(r, d, z, w, dw.data(), n, pre.data(), spc_r, spc_d);
    for (int k = 0; k <= n; ++k) {
        const double v[6] = {pre[k].c, pre[k].w, pre[k].x, pre[k].r, pre[k].d, pre[k].z};
        for (int c = 0; c < 6; ++c) records[6 * k + c] = v[c];
    }
    picca::WalkTask T;
    T.cos_half = std::cos(ang / 2);
    T.sin_half = std::sin(ang / 2);
    T.cp = T.cos_half * C.inv_p;
    T.st = T.sin_half * C.inv_t;
    T.rc = r[n / 2];
    T.dc = d[n / 2];
    T.j_lo = 0;
    T.j_hi = n;
    T.q0 = 1.0;
    if (!picca::walk_task(C, spc_r, spc_d, T.cp, T.st, T.q0)) return -1;
    int64_t runs = 0;
    RecordMem mem{r, d, w, z, dw.data(), pre.data(), out, &runs};
    const picca::WalkLane L{pixel1[0], pixel1[1], pixel1[2] * 0.5, pixel1[3],
                            pixel1[4] * pixel1[3]};
    picca::walk_lane(C, T, L, mem, true);
    return runs;
}

// The kernel's planes of the same entries, [3][n + 1][2].
void xi_walk_planes(int n, const double *r, const double *d, const double *z, const double *w,
                    const double *delta, double *planes) {
    std::vector<double> dw((size_t)n);
    for (int k = 0; k < n; ++k) dw[k] = delta[k] * w[k];
    double spc_r = 0, spc_d = 0;
    picca::build_walk_forest(r, d, z, w, dw.data(), n, (picca::PrefixPair *)planes, spc_r, spc_d);
}

}  // extern "C"
