// Pieces of the banded distortion-matrix kernels (dmat_band_kernel.hip) that also run on the
// host: along a monotone partner forest the r_par run index and the r_trans bin of the pairs
// of one pixel are monotone, so a pixel's pairs in one r_trans row are a range of partner
// pixels, and its sums per r_par bin are differences of the partner's prefix sums at the bins'
// edges.
//
// The header is compiled into the kernels and into a CPU harness of the tests; `Mem` supplies
// the memory accesses.
#pragma once

#include <math.h>
#include <stdint.h>

#include "engine.h"
#include "xi_walk.h"

namespace picca {

// Entry k of a forest's prefix sums covers its pixels [0, k): sums of w, w dll, w zf, w zf dll
// (zf: the redshift-evolution factor of the forest's role), pixels with w != 0, and w (r_comov
// - r_c), w (dist_m - d_c), w z as in PrefixRecord.  Forest f of L pixels has L + 1 entries
// starting at offsets[f] + f.
struct alignas(16) DmatPrefix {
    double w, wl, zw, zwl, c, r, d, z;
};
static_assert(sizeof(DmatPrefix) == 64, "DmatPrefix layout");

// Sums of the pair pass over one run of pixels of delta2 with one model bin: S0 = sum w1 w2,
// Sj = sum w1 w2 dll2, Z0 and Zj the same with zf1 zf2, and the effective-coordinate sums.
struct DmatSums {
    int bin;       // model r_trans bin * npm + model r_par bin
    uint32_t n;    // pairs with w2 != 0
    double s0, sj, z0, zj, rp, rt, z;
};

// The walk's sums for the pair pass: L.dw1 holds w1 zf1.
struct DmatAcc {
    using Prefix = DmatPrefix;
    using Sums = DmatSums;
    static constexpr bool RUNS = true;
    PICCA_HD static bool sums(const XiConst &C, const WalkTask &T, const WalkLane &L, int m, int c,
                              const Prefix &ps, const Prefix &pe, Sums &o) {
        const double n = pe.c - ps.c;
        const double dw = pe.w - ps.w;
        const double s_r = (pe.r - ps.r) - (L.r1 - T.rc) * dw;
        const double s_d = (L.d1 + T.dc) * dw + (pe.d - ps.d);
        o.bin = walk_bin(c, C.np, m >= 0 ? m : -m - 1);
        o.s0 = L.w1 * dw;
        o.sj = L.w1 * (pe.wl - ps.wl);
        o.z0 = L.dw1 * (pe.zw - ps.zw);
        o.zj = L.dw1 * (pe.zwl - ps.zwl);
        o.rp = T.cos_half * (L.w1 * (m >= 0 ? s_r : -s_r));
        o.rt = T.sin_half * (L.w1 * s_d);
        o.z = L.w1 * (L.zh1 * dw + 0.5 * (pe.z - ps.z));
        o.n = (uint32_t)fmax(n, 0.0);
        return n > 0;
    }
};

// One coordinate of the pairs of a pixel along its partner forest, in bins: x = v mul + off
// with v the partner's r_comov (the signed r_par run index is floor(x): -row - 1 below the
// pixel, row above it) or dist_m (the r_trans bin).  A coordinate within `margin` of an integer
// is redone with the reference's divide-then-multiply, so every key is the reference's.
struct BandAxis {
    double mul, off, margin;
    double self;       // the pixel's own r_comov or dist_m
    double scale;      // cos(ang/2) or sin(ang/2)
    double range;      // r_par_max - r_par_min or r_trans_max
    double n;          // bins of the range
    int kind;          // BAND_*
    double from;       // BAND_SIGNED: r_par_min
};

// r_trans; |r_par| of the auto-correlation; r_par = (partner - self) cos(ang/2) of a forest
// (the partner) with a quasar, whose bins count from r_par_min
enum : int { BAND_TRANS = 0, BAND_PAR = 1, BAND_SIGNED = 2 };

PICCA_HD inline BandAxis band_par_axis(double r, double mul, double cos_half, double span, int n,
                                       double margin) {
    return BandAxis{mul, -r * mul, margin, r, cos_half, span, (double)n, BAND_PAR, 0.0};
}

PICCA_HD inline BandAxis band_trans_axis(double d, double mul, double sin_half, double rtmax,
                                         int n, double margin) {
    return BandAxis{mul, d * mul, margin, d, sin_half, rtmax, (double)n, BAND_TRANS, 0.0};
}

PICCA_HD inline BandAxis band_signed_axis(double r, double mul, double cos_half, double from,
                                          double span, int n, double margin) {
    return BandAxis{mul, -r * mul - from / span * n, margin, r, cos_half, span, (double)n,
                    BAND_SIGNED, from};
}

// The key with the reference's arithmetic, clamped to [-n - 1, n].
PICCA_HD inline int band_exact_key(const BandAxis &A, double v) {
    if (A.kind == BAND_SIGNED) {
        const double t = ((v - A.self) * A.scale - A.from) / A.range * A.n;
        return (int)fmin(fmax(floor(t), -1.0), A.n);
    }
    if (A.kind == BAND_PAR) {
        const double rps = (A.self - v) * A.scale;
        const double row = fmin(floor(fabs(rps) / A.range * A.n), A.n);
        return (int)(rps > 0 ? -row - 1.0 : row);
    }
    return (int)fmin(floor((A.self + v) * A.scale / A.range * A.n), A.n);
}

PICCA_HD inline int band_key(const BandAxis &A, double v) {
    const double x = fma(v, A.mul, A.off);
    if (fabs(x - rint(x)) < A.margin) return band_exact_key(A, v);
    return (int)fmin(fmax(floor(x), -A.n - 1.0), A.n);
}

// key(v) < K
PICCA_HD inline bool band_below(const BandAxis &A, double v, int K) {
    const double x = fma(v, A.mul, A.off - (double)K);
    if (fabs(x) < A.margin) return band_exact_key(A, v) < K;
    return x < 0;
}

// Index table of a forest's rising values v (r_comov or dist_m): entry k < n holds the first
// pixel with v >= v[0] + k h, h the mean step.  Forest f's table starts at offsets[f].
struct BandTable {
    const int32_t *first;
    double v0, inv_h;
    int n;
};

PICCA_HD inline double band_mean_step(double v0, double v1, int n) {
    return n > 1 ? (v1 - v0) / (double)(n - 1) : 1.0;
}

// First pixel (n: none) of the partner forest whose key is at least K: from the table entry
// below the edge, two pixels at a time.  Keys do not fall along the forest, so the pixels before
// the entry lie below K (its position is taken 1e-3 steps low, far above the rounding).
template <class Val>
PICCA_HD inline int band_edge(const BandAxis &A, const BandTable &T, const Val &v, int K) {
    const double u = (((double)K - A.off) / A.mul - T.v0) * T.inv_h - 1e-3;
    int g = T.first[(int)fmin(fmax(u, 0.0), (double)(T.n - 1))];
    for (;;) {
        const double a = v(g < T.n ? g : T.n - 1), b = v(g + 1 < T.n ? g + 1 : T.n - 1);
        if (g >= T.n || !band_below(A, a, K)) return g;
        if (g + 1 >= T.n || !band_below(A, b, K)) return g + 1;
        g += 2;
    }
}

}  // namespace picca
