// Run walk of the pair kernel: the pixel pairs of one pixel i of delta1 with the pixels j of
// a monotone delta2, taken as runs of consecutive j that share one bin.
//
// Along a forest with strictly increasing r_comov and dist_m, the reference's r_par bin
// (py/picca/cf.py:355-376) of the pair (i, j) falls as j approaches r_comov1[i] and rises
// after it, and its r_trans bin never falls: every FP64 operation on the way is monotone.
// So the pairs of pixel i split into runs of consecutive j with one (side, r_par bin,
// r_trans bin) key, and a run's contribution to compute_xi's five sums and the pair count
// is the difference of two entries of prefix sums over delta2.  The walk finds each run's
// end with a few probes (a guess from the window's pixel density, then steps and
// bisection), so its cost grows with the number of runs, not of pairs.
//
// Exactness: a probe takes the bin coordinates with reciprocal multiplies and redoes the
// pixel with the reference's arithmetic when a coordinate lies within the rounding margin
// of an integer, so every probed key is the reference's.  Keys are monotone, so the pixels
// between two probes with one key share it.  A pixel within the margin of a bin edge or
// range limit is the first or last pixel of its run whenever consecutive pixels of delta2
// are more than four margins apart in both coordinates (the kernel walks only such pairs),
// and those pixels get the reference's edge, overflow and wrap-around treatment one by one.
//
// The cross-correlation (signed r_par, r_par_min any) walks the same way with the run index
// m = -row - 1, which rises with j; the cuts of the auto-correlation that leave whole runs
// (pair redshift, close pairs of one half plate) are a pixel window per lane and a dropped
// run.  Both are template parameters, so that the plain auto-correlation's code is its own.
// They walk only forests with level weights (level_values); the plain auto-correlation, whose
// bins collect the pairs of a whole survey, walks the others too.
//
// The header is compiled into the kernel and into a CPU harness of the tests, which runs
// the same lane program under bounds checks; `Mem` supplies the memory accesses.
#pragma once

#include <math.h>
#include <stdint.h>

#include <algorithm>
#include <cstddef>
#include <vector>

#include "engine.h"

#if defined(__HIPCC__)
#define PICCA_HD __host__ __device__
#else
#define PICCA_HD
#endif

namespace picca {

// Entry k of a forest's prefix sums covers its pixels [0, k): pixels with w != 0, and the
// sums of w, w * delta, w * (r_comov - r_c), w * (dist_m - d_c) and w * z, where r_c and
// d_c are r_comov and dist_m of the forest's pixel L / 2.  A forest of L pixels has L + 1
// entries.
struct PrefixRecord {
    double c, w, x, r, d, z;
};

// The entries in memory: per forest three planes of L + 1 pairs, (c, w), (x, r) and (d, z); the
// forests' blocks follow each other, so forest b's starts at pair 3 (offsets[b] + b).  The
// lanes of a wave read entries a pixel or a few apart: in planes 16 of them lie in two or three
// cache lines, as records of 48 bytes in six, and the walk reads at the L1 cache's line rate.
struct alignas(16) PrefixPair {
    double a, b;
};
constexpr int PREFIX_PLANES = 3;

PICCA_HD inline PrefixRecord prefix_entry(const PrefixPair &cw, const PrefixPair &xr,
                                          const PrefixPair &dz) {
    return PrefixRecord{cw.a, cw.b, xr.a, xr.b, dz.a, dz.b};
}

// Host side: the prefix entries of one forest of n pixels, store(k, entry) for k = 0 .. n, and
// the smallest step of r_comov and of dist_m between consecutive pixels (-1 unless both
// increase strictly; a forest of fewer than two pixels has no step and gets +1e300).  dw =
// delta * w, the same products the pair loops use.
template <class Store>
inline void walk_forest_entries(const double *r, const double *d, const double *z,
                                const double *w, const double *dw, int64_t n,
                                const Store &store, double &spc_r, double &spc_d) {
    const double rc = n > 0 ? r[n / 2] : 0.0;
    const double dc = n > 0 ? d[n / 2] : 0.0;
    PrefixRecord acc = {0, 0, 0, 0, 0, 0};
    store(0, acc);
    spc_r = 1e300;
    spc_d = 1e300;
    for (int64_t k = 0; k < n; ++k) {
        if (w[k] != 0) acc.c += 1.0;
        acc.w += w[k];
        acc.x += dw[k];
        acc.r += w[k] * (r[k] - rc);
        acc.d += w[k] * (d[k] - dc);
        acc.z += w[k] * z[k];
        store(k + 1, acc);
        if (k > 0) {
            const double sr = r[k] - r[k - 1];
            const double sd = d[k] - d[k - 1];
            spc_r = sr < spc_r ? sr : spc_r;
            spc_d = sd < spc_d ? sd : spc_d;
        }
    }
    if (!(spc_r > 0) || !(spc_d > 0)) {
        spc_r = -1.0;
        spc_d = -1.0;
    }
}

// The n + 1 entries as records, and as the kernel's planes.
inline void build_walk_forest(const double *r, const double *d, const double *z,
                              const double *w, const double *dw, int64_t n,
                              PrefixRecord *pre, double &spc_r, double &spc_d) {
    walk_forest_entries(r, d, z, w, dw, n, [&](int64_t k, const PrefixRecord &e) { pre[k] = e; },
                        spc_r, spc_d);
}

inline void build_walk_forest(const double *r, const double *d, const double *z,
                              const double *w, const double *dw, int64_t n,
                              PrefixPair *pre, double &spc_r, double &spc_d) {
    walk_forest_entries(r, d, z, w, dw, n, [&](int64_t k, const PrefixRecord &e) {
        pre[k] = PrefixPair{e.c, e.w};
        pre[n + 1 + k] = PrefixPair{e.x, e.r};
        pre[2 * (n + 1) + k] = PrefixPair{e.d, e.z};
    }, spc_r, spc_d);
}

// Whether sums over pixels of a forest may be differences of its prefix sums v[0] + v[1] + ...:
// a difference carries the rounding of everything before it, 2^-53 of the prefix, however light
// its own pixels are.  Level values: without their largest eighth the sum S of |v| is at most
// `most` mean values (8192 for weights: a typical pixel's share of the error stays below 1e-12;
// twice that for delta * weight), and no value other than 0 is below S / `least` (2^25 for
// weights: 4e-9 of the lightest pixel at worst; deltas may vanish).  The synthetic surveys reach
// 2100 mean weights and 2^13.2 smallest ones, with weights spread log-uniformly over 1e-3..1e2
// 5900 and 2^24, and 9200 mean delta * weight with heavy-tailed deltas too.  One pixel 1e4 times
// heavier than the others of a forest (not level): signed r_par 2.2e-13 in the weights, 5.2e-12
// in the r_par sums near 0 and 5.6e-13 in xi at worst from prefix sums (1e8 times: 1.9e-9,
// 9.6e-8 and 1.3e-8), 4e-14 to 6e-14 pair by pair (40 forests of the 0.8 A grid against 80-bit
// sums).  Up to 1e3 times the prefix sums' 2-norms are the smaller ones, 2e-15 to 4e-15 against
// 1e-14.
inline bool level_values(const double *v, int64_t n, double most, double least,
                         std::vector<double> &scratch) {
    // (eight values at a time, so that the additions do not wait for each other)
    constexpr int LANES = 8;
    double s[LANES] = {}, l[LANES], h[LANES] = {}, c[LANES] = {};   // h: of squares
    for (int q = 0; q < LANES; ++q) l[q] = INFINITY;
    auto take = [&](int q, double a) {
        s[q] += a;
        h[q] += a * a;
        c[q] += a != 0 ? 1.0 : 0.0;
        a = a != 0 ? a : INFINITY;
        l[q] = a < l[q] ? a : l[q];
    };
    int64_t k0 = 0;
    for (; k0 + LANES <= n; k0 += LANES)
        for (int q = 0; q < LANES; ++q) take(q, fabs(v[k0 + q]));
    for (; k0 < n; ++k0) take(0, fabs(v[k0]));
    double sum = 0.0, low = INFINITY, squares = 0.0, number = 0.0;
    for (int q = 0; q < LANES; ++q) {
        sum += s[q];
        low = l[q] < low ? l[q] : low;
        squares += h[q];
        number += c[q];
    }
    const int64_t count = (int64_t)number;
    const int64_t top = (count + 7) / 8, rest = count - top;
    if (rest == 0) return true;   // no value, or one: its prefix sums are exact
    // (a sum that overflows is not level)
    if (!(sum < 1e290) || !(sum <= least * low)) return false;
    // what the largest eighth holds at most (Cauchy-Schwarz): settles most forests in one pass
    if (sum * (double)rest <= most * (sum - sqrt((double)top * squares))) return true;
    scratch.clear();
    for (int64_t k = 0; k < n; ++k)
        if (v[k] != 0) scratch.push_back(fabs(v[k]));
    std::nth_element(scratch.begin(), scratch.begin() + (std::ptrdiff_t)(rest - 1), scratch.end());
    double low_sum = 0.0;
    for (int64_t k = 0; k < rest; ++k) low_sum += scratch[(size_t)k];
    return sum * (double)rest <= most * low_sum;
}

// Flags of a forest for the kernels (ForestView::mono).
enum : int {
    FOREST_RISES_R = 1,        // r_comov non-decreasing
    FOREST_RISES_D = 2,        // dist_m non-decreasing
    FOREST_RISES_Z = 4,        // z non-decreasing
    FOREST_LEVEL_W = 8,        // level weights
    FOREST_LEVEL_DW = 16       // level delta * weights
};

inline int level_flags(const double *w, const double *dw, int64_t n,
                       std::vector<double> &scratch) {
    return (level_values(w, n, 8192.0, 0x1p25, scratch) ? FOREST_LEVEL_W : 0) |
           (level_values(dw, n, 16384.0, INFINITY, scratch) ? FOREST_LEVEL_DW : 0);
}

// Per (forest pair, chunk of delta1): wave-uniform constants of the walk.
struct WalkTask {
    double cos_half, sin_half;
    double cp, st;       // cos(ang/2) * np / span_p and sin(ang/2) * nt / r_trans_max
    double rc, dc;       // r_c and d_c of delta2's prefix sums
    double q0;           // mean delta2 pixels per unit of the r_par coordinate in the window
    int32_t j_lo, j_hi;  // pruned pixel window of delta2
    bool shp = false;    // CUTS: close pairs of one half plate are removed
};

// Pixel i of delta1 (weight != 0).
struct WalkLane {
    double r1, d1, zh1, w1, dw1;  // zh1 = z1 / 2, dw1 = delta1 * w1
    int32_t j_lo = 0, j_hi = 0;   // CUTS: the lane's window, inside [T.j_lo, T.j_hi)
};

// Everything the reference does with one pixel pair (standard binning, auto-correlation,
// r_par_min == 0, no cuts), py/picca/cf.py:355-376, with its key: m is the signed r_par run
// index, m = bin for r_comov2 >= r_comov1 and -bin - 1 below it, clamped to [-np - 1, np]
// (|m| beyond np - 1 is rejected); c is the r_trans bin clamped to nt (nt is rejected, or a
// wrap-around pair).  The cross-correlation (XC): m = -bin - 1 for every pair, clamped to
// [-np - 1, 0] (0: r_par < r_par_min, rejected).
struct WalkExact {
    int32_t m, c;
    bool edge;      // within edge_tol of a bin edge, or outside the range but within
                    // edge_tol of it in both coordinates
    bool over;      // accepted, flat bin index >= np * nt (picca writes out of bounds)
    bool wrap;      // accepted with its r_trans bin rounded to nt: the flat index is
                    // column 0 of the next r_par row, where the pair is added
    int32_t pbin;   // padded histogram bin of a wrap pair
    bool mine;      // XC: the pair's r_par row lies in the launch's rows [row0, row0 + rows),
                    // which count its edge and overflow pairs (rows beyond the range belong
                    // to the first and last launch)
    double r_par, r_trans;
};

PICCA_HD inline double walk_edge_distance(double t, double width) {
    const double frac = t - floor(t);
    const double lo = frac * width;
    const double hi = (1.0 - frac) * width;
    return lo < hi ? lo : hi;
}

template <bool XC = false>
PICCA_HD inline WalkExact walk_exact(const XiConst &C, double r1, double d1, double r2,
                                     double d2, double cos_half, double sin_half) {
    WalkExact e;
    const double rps = (r1 - r2) * cos_half;
    const double r_par = XC ? rps : fabs(rps);
    const double r_trans = (d1 + d2) * sin_half;
    const double t_par = (XC ? r_par - C.rpmin : r_par) / C.span_p * C.np_d;
    const double t_trans = r_trans / C.rtmax * C.nt_d;
    const double f_par = floor(t_par);
    const double f_trans = floor(t_trans);
    // (no fmin: it would quiet the constants once per call, also in passes without a call)
    const double row = f_par < C.np_d ? f_par : C.np_d;
    if (XC) {
        e.m = (int32_t)(-fmax(row, -1.0) - 1.0);
        const double own = fmin(fmax(row, 0.0), C.np_d - 1.0);
        e.mine = own >= (double)C.row0 && own < (double)(C.row0 + C.rows);
    } else {
        e.m = (int32_t)(rps > 0 ? -row - 1.0 : row);
        e.mine = true;
    }
    e.c = (int32_t)(f_trans < C.nt_d ? f_trans : C.nt_d);
    const bool out_p = XC ? (r_par >= C.rpmax) | (r_par < C.rpmin) : r_par >= C.rpmax;
    const bool out_t = r_trans >= C.rtmax;
    const bool out = out_p | out_t;
    // outside the range, but within edge_tol of it in both coordinates
    bool edge_out = (r_par - C.rpmax < C.edge_tol) & (r_trans - C.rtmax < C.edge_tol);
    if (XC) edge_out = edge_out & (C.rpmin - r_par < C.edge_tol);
    const bool edge_in = (r_par != 0 && walk_edge_distance(t_par, C.width_p) < C.edge_tol) ||
                         (r_trans != 0 && walk_edge_distance(t_trans, C.width_t) < C.edge_tol);
    e.edge = out ? edge_out : edge_in;
    const double bin_f = f_trans + C.nt_d * f_par;
    e.over = !out & !(bin_f < C.nb_d);
    e.wrap = !out & !e.over & (f_trans >= C.nt_d);
    // (the cross-correlation's histogram holds the rows from row0 on)
    e.pbin = e.wrap ? (int32_t)(C.ntp_d * (f_par + 1.0)) - (XC ? C.row0 * C.ntp : 0) : 0;
    e.r_par = r_par;
    e.r_trans = r_trans;
    return e;
}

// The reference's treatment of a pixel within the margin of an edge: edge and overflow
// counts, and the wrap-around pair, which no run holds.  Pixels with w == 0 (either sign)
// are skipped before any arithmetic, as in the reference.  With T.shp the walk drops the runs
// of r_par row 0; the reference drops the pairs with r_par < the row's width, which can
// differ from the row by rounding: such a pair is added here, or taken back from its run.
template <bool XC, bool CUTS, class Mem>
PICCA_HD inline void walk_special(const XiConst &C, const WalkTask &T, const WalkLane &L,
                                  Mem &mem, int p) {
    const double w2 = mem.w(p);
    if (w2 == 0) return;
    double r2, d2;
    mem.rd(p, r2, d2);
    const WalkExact e = walk_exact<XC>(C, L.r1, L.d1, r2, d2, T.cos_half, T.sin_half);
    if (XC && !e.mine) return;
    if (e.edge) mem.count_edge();
    bool cut = false;
    double sign = e.wrap ? 1.0 : 0.0;
    int bin = e.pbin;
    if constexpr (CUTS && !XC) {
        cut = T.shp & (fabs(e.r_par) < C.width_p);
        const bool in = !e.over & !e.wrap & (e.r_par < C.rpmax) & (e.r_trans < C.rtmax);
        const int row = e.m >= 0 ? e.m : -e.m - 1;
        if (T.shp & in) {
            sign = row == 0 ? (cut ? 0.0 : 1.0) : (cut ? -1.0 : 0.0);
            bin = row * C.ntp + e.c;
        }
        if (e.wrap & cut) sign = 0.0;
    }
    if (e.over & !cut) mem.count_overflow();
    if (sign != 0.0) {
        const double w12 = L.w1 * w2 * sign;
        const double z = L.zh1 + mem.z(p) * 0.5;
        mem.add(bin, w12, L.dw1 * mem.dw(p) * sign, e.r_par * w12, e.r_trans * w12, z * w12,
                sign > 0 ? 1u : ~0u);   // ~0u: -1 modulo 2^32
    }
}

// row * len + col of a histogram, whose rows and columns are below 2^23
PICCA_HD inline int walk_bin(int row, int len, int col) {
#if defined(__HIP_DEVICE_COMPILE__)
    return __mul24(row, len) + col;   // the full multiply takes four times as long
#else
    return row * len + col;
#endif
}

// Histogram addition of the run [j, jn) of key (m, c): prefix differences times the lane's
// pixel.  False for an empty run.  No branch, and finite for any finite state.
struct RunSums {
    int bin;
    double we, xi, rp, rt, z;
    uint32_t n;
};

template <bool XC>
PICCA_HD inline bool walk_run_sums(const XiConst &C, const WalkTask &T, const WalkLane &L, int m,
                                   int c, const PrefixRecord &ps, const PrefixRecord &pe,
                                   RunSums &o) {
    const double n = pe.c - ps.c;  // pixels of the run with w2 != 0 (>= 0)
    const double dw = pe.w - ps.w;
    const double dx = pe.x - ps.x;
    const double dr = pe.r - ps.r;
    const double dd = pe.d - ps.d;
    const double dz = pe.z - ps.z;
    // sum over the run of w2 (r2 - r1) and w2 (d1 + d2), from the centred sums
    const double s_r = fma(T.rc - L.r1, dw, dr);
    const double s_d = fma(L.d1 + T.dc, dw, dd);
    const bool up = !XC && m >= 0;   // r_par counted as r2 - r1
    o.bin = walk_bin(up ? m : XC ? -m - 1 - C.row0 : -m - 1, C.ntp, c);
    o.we = L.w1 * dw;
    o.xi = L.dw1 * dx;
    o.rp = T.cos_half * (L.w1 * (up ? s_r : -s_r));
    o.rt = T.sin_half * (L.w1 * s_d);
    o.z = L.w1 * fma(L.zh1, dw, 0.5 * dz);
    o.n = (uint32_t)(int32_t)n;
    return n > 0;
}

// What a walk sums over its runs: the prefix records it reads, the sums of a run, and whether
// its memory wants each closed run (mem.closed).  XiAcc: compute_xi's sums.
template <bool XC>
struct XiAcc {
    using Prefix = PrefixRecord;
    using Sums = RunSums;
    static constexpr bool RUNS = false;
    PICCA_HD static bool sums(const XiConst &C, const WalkTask &T, const WalkLane &L, int m, int c,
                              const Prefix &ps, const Prefix &pe, Sums &o) {
        return walk_run_sums<XC>(C, T, L, m, c, ps, pe, o);
    }
};

// What a memory type need not have: constants of its own for the exact arithmetic (the walk's
// are taken), and the count of runs of every lane with each pass (count_run(closed, n)): without
// it the closed runs alone are counted.
template <class Mem>
PICCA_HD inline auto walk_consts(Mem &mem, const XiConst &C, int) -> decltype(mem.consts(C)) {
    return mem.consts(C);
}
template <class Mem>
PICCA_HD inline const XiConst &walk_consts(Mem &, const XiConst &C, long) {
    return C;
}
template <class Mem>
PICCA_HD inline auto walk_count_run(Mem &mem, bool closed, uint32_t n, int)
    -> decltype(mem.count_run(closed, n)) {
    mem.count_run(closed, n);
}
template <class Mem>
PICCA_HD inline void walk_count_run(Mem &mem, bool closed, uint32_t n, long) {
    if (closed) mem.count_run(n);
}

// Reciprocal of x > 0 within 2.5e-4 relative, the same on the host and the device: the
// seed is the bit pattern of 2.0^1023 (0x7FE0...) minus that of x, within 12.5 % of 1 / x
// for a normal x, then two Newton steps y (2 - x y).  For the guess of a run's end only.
PICCA_HD inline double walk_rcp_guess(double x) {
    const uint64_t b = 0x7FE0000000000000ull - __builtin_bit_cast(uint64_t, x);
    double y = __builtin_bit_cast(double, b);
    y = y * fma(-x, y, 2.0);
    y = y * fma(-x, y, 2.0);
    return y;
}

// Key of pixel p from its coordinates relative to the upper edges of the run key (m, c):
// a = (r2 - r1) cp - (m + 1) and b = (d1 + d2) st - (c + 1), so the pixel's r_par run index
// is m + 1 + floor(a) and its r_trans bin c + 1 + floor(b), clamped as in walk_exact.
template <bool XC>
PICCA_HD inline void walk_key_from(const XiConst &C, int m, int c, double a, double b,
                                   int &mp, int &cp) {
    // |a| and |b| stay within a few times the bin counts inside the pruned window
    const int fm = (int)floor(a) + (m + 1);
    const int fc = (int)floor(b) + (c + 1);
    const int top = XC ? 0 : C.np;
    const int below = fm < top ? fm : top;
    mp = below > -C.np - 1 ? below : -C.np - 1;
    cp = fc < C.nt ? fc : C.nt;
}

// Whether a task takes the run walk: delta2 increases strictly with consecutive pixels more
// than four rounding margins apart in both bin coordinates (spc_r, spc_d: its smallest steps
// of r_comov and dist_m), and, under the automatic schedule, the window holds at least
// XI_WALK_MIN_DENSITY pixels per unit of the r_par coordinate (q0).
PICCA_HD inline bool walk_task(const XiConst &C, double spc_r, double spc_d, double cp, double st,
                               double q0) {
    return (C.flags & XI_WALK) && spc_r > 0 && spc_d > 0 && cp * spc_r > 4.0 * (0.5 - C.half_p) &&
           st * spc_d > 4.0 * (0.5 - C.half_t) &&
           (!(C.flags & XI_WALK_AUTO) || q0 >= XI_WALK_MIN_DENSITY);
}

// r_comov2 beyond r_par_max on the far side (XC: r_par below the launch's rows), or r_trans
// beyond r_trans_max: every later pixel is rejected too
template <bool XC>
PICCA_HD inline bool walk_terminal(const XiConst &C, int m, int c) {
    return m >= (XC ? -C.row0 : C.np) || c >= C.nt;
}

// All pairs of lane pixel L with delta2's window [T.j_lo, T.j_hi).
//
// Every lane starts at j_lo and walks its runs in order, so the lanes of a wave (consecutive
// pixels of delta1) probe neighbouring pixels of delta2 at the same time and their loads
// share cache lines.  (Starting each lane at a different point of its r_par range, so that
// the lanes add to different bins, and prefetching two runs ahead were both measured
// slower.)
//
// One loop, one memory round trip per pass: every pass tests pixels pa, pb (their r_comov
// and dist_m) and the prefix entry at pb against the thresholds of the current run key
// (Ka = r1 cp + m + 1, Kb = c + 1 - d1 st: a pixel at or after the run's first pixel keeps
// the key iff r2 cp < Ka and d2 st < Kb):
//   * start of the walk at j (pa = pb = j): the run's key, its prefix entry, the first
//     guess of its end;
//   * test of a candidate end g of the run [j, ...) (pa = g - 1, pb = g): pixel g - 1 with
//     the run's key and pixel g without it close the run at g, and pixel g opens the next
//     run with its own key; otherwise the bracket (lo, hi) of the end shrinks (a step back
//     after the first overshoot, then bisection; galloping forward after an undershoot).
// The next pass's loads are issued before the closed run is added to the histogram; the
// addition is made by all lanes of the wave together (mem.flush), so every lane stays in
// the loop until the wave's last lane is done (`alive` false: a lane without a pixel, or
// one past its last run).  The guess of a run's end is its first pixel plus the distance
// to the run's upper r_par edge times the pixel density where the previous run closed (the
// window's mean for the first run), so a run is usually closed in one pass.
// A coordinate within the rounding margin of an integer is redone with the reference's
// arithmetic (walk_exact); such a pixel is the first or last pixel of its run and gets the
// reference's edge, overflow and wrap-around treatment (walk_special).
// XC: cross-correlation (signed r_par; the launch's rows [C.row0, C.row0 + C.rows)).  CUTS:
// the lane's own window [L.j_lo, L.j_hi) (pair-redshift cuts; empty: `alive` false) and T.shp.
template <bool XC = false, bool CUTS = false, class Acc = XiAcc<XC>, class Mem = void>
PICCA_HD inline void walk_lane(const XiConst &C, const WalkTask &T, const WalkLane &L, Mem &mem,
                               bool alive) {
    const int j_hi = CUTS ? L.j_hi : T.j_hi;
    if (T.j_lo >= T.j_hi) return;  // wave-uniform
    const XiConst &exact = walk_consts(mem, C, 0);
    const int last = T.j_hi - 1;  // pixel reads stay inside the window
    // the run coordinate is (r2 - r1) cp, from r_par_min for the cross-correlation
    const double r1cp = XC ? L.r1 * T.cp - C.rpmin * C.inv_p : L.r1 * T.cp;
    const double d1st = L.d1 * T.st;
    // Before the first run opens the key is (-1, -1), which no pixel has (r_trans >= 0
    // here), so the thresholds give each pixel's own coordinates.
    int m = -1, c = -1;
    double nKa = -r1cp, nKb = d1st;   // -Ka, -Kb
    int j = CUTS ? L.j_lo : T.j_lo;
    bool starting = true;
    typename Acc::Prefix ps = {};
    int lo = j, hi = j_hi, g = j, step = 1;
    bool near_lo = false, missed = false;
    // the pass's probes: pixels pa and pb and the prefix entry at pb, loaded at the end of
    // the previous pass so that the loads overlap that pass's histogram additions
    int pa = j, pb = j;
    double ra, da, rb, db;
    mem.rd(pa, ra, da);
    mem.rd(pb, rb, db);
    typename Acc::Prefix pg = mem.prefix(pb);
    for (;;) {
        // the sums of the run [j, g) of the current key, added by mem.flush with every lane
        // of the wave if the run closes in this pass (`on`); computed by every lane, so that
        // the values the flush moves between lanes are finite
        typename Acc::Sums run;
        const bool nonempty = Acc::sums(C, T, L, m, c, ps, pg, run);
        mem.pin(run);
        bool on = false, close = false;
        if (alive) {
            mem.count_probe();
            const double aA = fma(ra, T.cp, nKa), bA = fma(da, T.st, nKb);
            const double aB = fma(rb, T.cp, nKa), bB = fma(db, T.st, nKb);
            // pixel pb: within the margin of any bin edge; pixel pa: of the run's upper edges
            const bool nearB =
                (fabs(aB - rint(aB)) < C.fast_p) || (fabs(bB - rint(bB)) < C.fast_t);
            const bool nearA = (fabs(aA) < C.fast_p) || (fabs(bA) < C.fast_t);
            int mB, cB;
            walk_key_from<XC>(C, m, c, aB, bB, mB, cB);
            if (nearB) {
                const WalkExact e =
                    walk_exact<XC>(exact, L.r1, L.d1, rb, db, T.cos_half, T.sin_half);
                mB = e.m;
                cB = e.c;
            }
            bool inA = (aA < 0) & (bA < 0);
            if (nearA & !starting) {
                const WalkExact e =
                    walk_exact<XC>(exact, L.r1, L.d1, ra, da, T.cos_half, T.sin_half);
                inA = (e.m == m) && (e.c == c);
            }
            // outcome of the pass
            const bool has1 = g - 1 > lo;    // pa is not yet known to have the run's key
            const bool has2 = g < j_hi;      // pb lies inside the window
            const bool same1 = !has1 | inA;
            const bool same2 = has2 & (mB == m) & (cB == c);
            const bool miss = !starting & !same1;            // the run ends at g - 1 or before
            const bool gallop = !starting & same1 & same2;   // the run goes on past g
            close = !starting & same1 & !same2;              // the run is [j, g)
            const bool open = starting | (close & has2);     // a run starts at pb
            const bool terminal = open & walk_terminal<XC>(C, mB, cB);
            const bool done = (close & !has2) | terminal;
            const bool special_last =
                close & ((has1 & nearA) | (!has1 & near_lo)) & (g - 1 > j);
            const int p_last = g - 1;
            const bool special_first = open & nearB;
            const int p_first = pb;
            // the closing run [j, g): prefix entries ps and pg (the entry at g)
            on = close & nonempty & (m >= (XC ? -(C.row0 + C.rows) : -C.np));
            if constexpr (CUTS && !XC) on = on & !(T.shp & ((m == 0) | (m == -1)));
            if constexpr (Acc::RUNS) mem.closed(on, j, g, c);
            // next state
            const int g_miss = missed ? lo + 1 + ((g - 1 - lo) >> 1) : g - 1;
            const int g_gallop = g + step < hi ? g + step : hi;
            if (miss) {
                hi = g - 1;
                g = g_miss;
                missed = true;
            }
            if (gallop) {
                lo = g;
                near_lo = nearB;
                g = g_gallop;
                step <<= 1;
            }
            if (open && !terminal) {
                // pixels per unit of the r_par coordinate: from the spacing of pixels g - 1
                // and g where a run closed here, else the window's mean
                const double q = starting ? T.q0 : walk_rcp_guess(T.cp * (rb - ra));
                j = pb;
                m = mB;
                c = cB;
                ps = pg;
                starting = false;
                nKa = -r1cp - (double)(m + 1);
                nKb = d1st - (double)(c + 1);
                lo = j;
                hi = j_hi;
                near_lo = nearB;
                missed = false;
                step = 1;
                // pixels to the run's upper r_par edge
                const double ahead = ceil(-fma(rb, T.cp, nKa) * q);
                g = j + (int)fmin(fmax(ahead, 1.0), (double)(j_hi - j));
            }
            if (!done) {
                pa = g - 1;
                pb = g;
            }
            if (special_last) walk_special<XC, CUTS>(exact, T, L, mem, p_last);
            if (special_first) walk_special<XC, CUTS>(exact, T, L, mem, p_first);
            if (done) alive = false;
        }
        walk_count_run(mem, close, run.n, 0);
        // the next pass's probes, issued before the histogram additions (a lane that is done
        // reloads its last probes, which lie inside the window)
        const bool more = mem.any(alive);
        mem.rd(pa, ra, da);
        mem.rd(pb < last ? pb : last, rb, db);
        pg = mem.prefix(pb);
        mem.flush(on, run);
        if (!more) break;
    }
}

}  // namespace picca
