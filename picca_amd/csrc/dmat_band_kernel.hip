// Distortion matrix of forest pairs without cuts on gfx950 (MI355X): the sums of
// dmat_kernel.hip (compute_dmat_forest_pairs_fast, py/picca/cf.py:520-887) taken from prefix
// sums over the forests instead of pixel pair by pixel pair.
//
// It covers the standard auto-correlation binning (r_par_min == 0, |r_par|; forest x quasar
// pairs below), forests whose r_comov and dist_m rise strictly with steps above the rounding
// margins and whose weights are level (xi_walk.h), model bins that split the data bins in 2^k
// parts (so that a model bin lies in one data bin to the last bit) and no pair-redshift, zerr or
// same-half-plate cut on the pair; the host sends the other pairs to dmat_kernel.hip.  Every pair in range is then selected, the model bins U of a pair are all
// that it reaches, and the pair-bin term of (A, M) is the pair's sum of w1 w2 zf in M.
//
// dmat_band_pass_kernel  one workgroup per forest pair, a lane per pixel of delta1: the run walk
//     of xi_walk.h over the model bins, adding each run's sums (S0, Sj, Si, Sij, the same with
//     the redshift factors, and the effective coordinates) to LDS; rows of S and eta5..eta8 to
//     the workspace, the pair-bin term, weights_dmat and the effective sums to HBM, and the
//     pixel ranges of every r_trans row.
// dmat_band_{count,scan,list}_kernel  the list of forest pairs of every (data r_trans row t,
//     model row u) tile, cut into work items.
// dmat_band_fill_kernel  persistent workgroups take items: the np x npm block of a tile in the
//     FP64 matrix cores' accumulators, per forest pair the rank-4 term and, for 16 pixels of a
//     forest at a time, their vectors P, P' and eta (rows t and u) in LDS, then
//     P^T eta + P'^T eta' as K = 4 products.  A wave builds the vectors of four pixels, 16 lanes
//     each: a lane finds the partner pixel at the edge of one r_par bin (an index table of the
//     forest and one or two probes) and takes the difference of the prefix sums there and at
//     its neighbour's edge.
//
// Why this split: pair by pair, the walk of a pixel's partners is repeated for every tile the
// pixel feeds (8.5 tiles a pair on the 0.8 A grid, 8 on the 100k survey), with the four vector
// sums and the bins of every pixel pair (976 vector instructions per pixel and tile, LDS
// atomics whose lanes meet in one bin) and a workgroup barrier every four pixels.  From the
// prefix sums the work is one edge per run of 3.6 to 7.2 pixels, the edges are independent of
// each other (stepping from pixel to pixel or from run to run along the partner is a serial
// chain: 88 ms on 21k pairs of the 0.8 A grid where this takes 61 ms), and the barriers come
// every 16 pixels.  On those pairs (2500 forests, 50 x 50 data and 100 x 50 model bins) the
// call takes 88 ms against 350 ms, the fill 61 ms against 264 ms, the pass 15 ms against 83 ms.
//
// In range means binned here: for r_trans, and for |r_par| from 0, x < end gives x / end <=
// 1 - 2^-53 after rounding, which times n stays below n.  Only a signed r_par can round to the end
// of its range (its distance from r_par_min may); such a quasar's pair, and one with a pixel at
// r_par_min exactly, which xcf counts apart, goes into the redo list for dmat_kernel.hip and adds
// nothing.  The pass does the same with a run outside the rows that the host bounded, which the
// bounds leave no pair.
#include <hip/hip_runtime.h>
#include <limits.h>
#include <stdint.h>

#include "device_util.h"
#include "dmat_band.h"
#include "engine.h"

namespace picca {

namespace {

typedef double double4_t __attribute__((ext_vector_type(4)));

constexpr int PASS_WAVES = DMAT_BAND_PASS_BLOCK / 64;
constexpr int FILL_WAVES = DMAT_BAND_FILL_BLOCK / 64;
constexpr int FILL_CB = DMAT_CHUNK_MRP / 16;   // 16-column blocks of model r_par bins
static_assert(DMAT_CHUNK_RP == 16 * FILL_WAVES, "one 16-row block of data bins per wave");

// vectors of one pixel in the fill's panel (doubles): P, P', eta, eta' and padding, so that
// the four pixels of a K = 4 product start 32 banks apart
constexpr int PX = 16;   // pixels of a panel
constexpr int VP = 0, VP2 = DMAT_CHUNK_RP, VE = 2 * DMAT_CHUNK_RP,
              VE2 = 2 * DMAT_CHUNK_RP + DMAT_CHUNK_MRP;
constexpr int VLEN = 2 * DMAT_CHUNK_RP + 2 * DMAT_CHUNK_MRP + 16;
static_assert((2 * VLEN) % 64 == 32, "pixels of a panel 32 banks apart");
// the rank-4 term's S and eta rows lie in the panel's memory, before the panel is used
static_assert(4 * (DMAT_CHUNK_RP + DMAT_CHUNK_MRP) <= PX * VLEN, "rank-4 rows fit the panel");

__device__ __forceinline__ void lds_add(double *p, double v) {
    __hip_atomic_fetch_add(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

struct BandPair {
    int a, b, la, lb;
    int64_t oa, ob;
    double cos_half, sin_half;
    double inv_w1, inv_w2, inv_s1, inv_s2;
    bool order1, order2;
};

__device__ BandPair load_band_pair(const DmatForests &F, const DmatBandSlots &P, int s) {
    BandPair q;
    q.a = uniform_int(P.slot[s].a);
    q.b = uniform_int(P.slot[s].b);
    q.oa = uniform_i64(F.off[q.a]);
    q.la = (int)(uniform_i64(F.off[q.a + 1]) - q.oa);
    q.ob = uniform_i64(F.off[q.b]);
    q.lb = (int)(uniform_i64(F.off[q.b + 1]) - q.ob);
    q.cos_half = uniform_f64(P.cs[2 * s]);
    q.sin_half = uniform_f64(P.cs[2 * s + 1]);
    q.inv_w1 = 1.0 / uniform_f64(F.sum_w[q.a]);
    q.inv_w2 = 1.0 / uniform_f64(F.sum_w[q.b]);
    q.inv_s1 = 1.0 / uniform_f64(F.sw_dll[q.a]);
    q.inv_s2 = 1.0 / uniform_f64(F.sw_dll[q.b]);
    q.order1 = uniform_int(F.order[q.a]) == 1;
    q.order2 = uniform_int(F.order[q.b]) == 1;
    return q;
}

// Memory of the pass's walk: delta2's pixels and prefix sums in HBM, the LDS rows of the
// pair's model bins and pixel ranges.
struct BandPassMem {
    const double *__restrict__ rp;
    const double *__restrict__ dp;
    const double *__restrict__ wp;
    const double *__restrict__ zp;
    const DmatPrefix *__restrict__ pre;
    double *acc;          // [DMAT_BAND_SUMS][rows][npm] from model row uc0
    int32_t *rng;         // [rows of the pair][4]: first and last i, first and last j
    int *special;
    int stride;           // rows * npm
    int nu;               // model rows of the pair
    int base;             // uc0 * npm
    int u0;               // first model row of the pair
    int i;                // the lane's pixel of delta1
    double l1;            // its dll
    const XiConst *exact;   // LDS copy
    uint64_t n_in;
    int row, r_first, r_last;   // run of runs in one model row

    __device__ void rd(int p, double &r, double &d) const {
        r = rp[p];
        d = dp[p];
    }
    __device__ DmatPrefix prefix(int p) const { return pre[p]; }
    __device__ const XiConst &consts(const XiConst &) const { return *exact; }
    __device__ double w(int p) const { return wp[p]; }
    __device__ double z(int p) const { return zp[p]; }
    __device__ double dw(int) const { return 0.0; }
    __device__ void add(int, double, double, double, double, double, uint32_t) { *special = 1; }
    // Adds the runs that the wave's lanes closed in one pass (every lane calls it).  As in the xi
    // kernel the lanes of a group of four that closed runs of one bin are summed first: eleven
    // FP64 atomics per lane, many of them on one address, bound the pass (21k pairs of the 0.8 A
    // grid: 15.0 ms, one lane at a time 17.6 ms).
    __device__ void flush(bool on, const DmatSums &o) {
        const int k = o.bin - base;
        if (on) n_in += o.n;
        if (on && (unsigned)k >= (unsigned)stride) {   // outside the rows that the host bounded
            *special = 1;
            on = false;
        }
        const int key = on ? k + 1 : 0;
        const int gl = __lane_id() & 3;
        const int head = (key != dpp_int<DPP_ROW_SHR1>(key)) || gl == 0;
        const int head2 = head | dpp_int<DPP_ROW_SHR1>(head);
        const bool write = on && ((key != dpp_int<DPP_ROW_SHL1>(key)) || gl == 3);
        const double take1 = head ? 0.0 : 1.0, take2 = head2 ? 0.0 : 1.0;
        double *b = acc + (on ? k : 0);
        auto add_sum = [&](int c, double v) {
            v = fma(dpp_f64<DPP_ROW_SHR1>(v), take1, v);
            v = fma(dpp_f64<DPP_ROW_SHR2>(v), take2, v);
            if (write) lds_add(b + c * stride, v);
        };
        add_sum(0, o.s0);
        add_sum(1, o.sj);
        add_sum(2, l1 * o.s0);
        add_sum(3, l1 * o.sj);
        add_sum(4, o.z0);
        add_sum(5, o.zj);
        add_sum(6, l1 * o.z0);
        add_sum(7, l1 * o.zj);
        add_sum(8, o.rp);
        add_sum(9, o.rt);
        add_sum(10, o.z);
    }
    __device__ void note() {
        if (row < 0) return;
        int32_t *r = rng + 4 * (row - u0);
        atomicMin(r, i);
        atomicMax(r + 1, i);
        atomicMin(r + 2, r_first);
        atomicMax(r + 3, r_last);
    }
    __device__ void closed(bool on, int j, int g, int c) {
        if (!on) return;
        if ((unsigned)(c - u0) >= (unsigned)nu) {
            *special = 1;
            return;
        }
        if (c != row) {
            note();
            row = c;
            r_first = j;
        }
        r_last = g - 1;
    }
    __device__ bool any(bool v) const { return __builtin_amdgcn_ballot_w64(v) != 0; }
    __device__ static void pin(DmatSums &) {}
    __device__ void count_edge() {}
    __device__ void count_overflow() { *special = 1; }
    __device__ void count_probe() {}
    __device__ void count_run(bool, uint32_t) {}
};

}  // namespace

// Prefix sums of the listed forests for both roles: one wave per forest.  The sums are taken in
// pixel order (so that a pixel without weight leaves them as they are), a lane per field, from
// terms that all lanes make of 64 pixels at a time in LDS, the next 64 pixels already loading; the
// rows leave as they lie in memory.  Bound by the chain of additions where the list is short and
// by the stores where it is long: 100 forests of up to 1500 pixels, both roles, PREFIX_SHORT, 3000
// forests PREFIX_LONG (a thread per forest and field that loads eight pixels ahead: 460 us and
// 540 us).
template <bool BOTH>
__global__ __launch_bounds__(64) void dmat_prefix_kernel(DmatForests F, DmatListed T,
                                                         DmatPrefix *__restrict__ pa,
                                                         DmatPrefix *__restrict__ pb) {
    constexpr int FIELDS = BOTH ? 16 : 8;
    constexpr int ROW = FIELDS + 1;   // odd: the lanes' rows start in different banks
    __shared__ double term[64 * ROW];
    const int lane = threadIdx.x;
    const int64_t f = T.forest[blockIdx.x].forest, at = T.forest[blockIdx.x].at;
    const int64_t o = F.off[f];
    const int n = (int)(F.off[f + 1] - o);
    const double rc = n > 0 ? F.r[o + n / 2] : 0.0, dc = n > 0 ? F.d[o + n / 2] : 0.0;
    // field c of entry k of delta1's sums (c < 8) and of delta2's
    auto out = [&](int c) { return (double *)((BOTH && c >= 8 ? pb : pa) + at) + (c & 7); };
    if (lane < FIELDS) out(lane)[0] = 0.0;
    double acc = 0.0;   // lane c < FIELDS: field c
    double w = 0, l = 0, za = 0, zb = 0, r = 0, d = 0, z = 0;
    auto load = [&](int q) {
        if (q >= n) return;
        w = F.w[o + q];
        l = F.dll[o + q];
        za = F.zfa[o + q];
        if (BOTH) zb = F.zfb[o + q];
        r = F.r[o + q];
        d = F.d[o + q];
        z = F.z[o + q];
    };
    load(lane);
    for (int q0 = 0; q0 < n; q0 += 64) {
        const int count = min(64, n - q0);
        double *t = term + lane * ROW;
        if (lane < count) {
            const double common[8] = {w, w * l, 0, 0, w != 0 ? 1.0 : 0.0, w * (r - rc),
                                      w * (d - dc), w * z};
#pragma unroll
            for (int c = 0; c < FIELDS; ++c) {
                const double zw = w * (c < 8 ? za : zb);
                t[c] = (c & 7) == 2 ? zw : (c & 7) == 3 ? zw * l : common[c & 7];
            }
        }
        __syncthreads();
        load(q0 + 64 + lane);
        if (lane < FIELDS) {
            double *field = term + lane;
            int k = 0;
            for (; k + 8 <= count; k += 8) {
                double v[8];
#pragma unroll
                for (int u = 0; u < 8; ++u) v[u] = field[(k + u) * ROW];
#pragma unroll
                for (int u = 0; u < 8; ++u) {
                    acc += v[u];
                    field[(k + u) * ROW] = acc;
                }
            }
            for (; k < count; ++k) {
                acc += field[k * ROW];
                field[k * ROW] = acc;
            }
        }
        __syncthreads();
        for (int k = lane; k < 8 * count; k += 64) {
            const int64_t to = (int64_t)(q0 + 1 + (k >> 3)) * 8;
            const double *row = term + (k >> 3) * ROW + (k & 7);
            out(k & 7)[to] = row[0];
            if (BOTH) out(8 + (k & 7))[to] = row[8];
        }
        __syncthreads();   // the terms are read
    }
}

// Index tables of r_comov (blockIdx.y 0) and dist_m (1) (BandTable) of the listed forests: one
// workgroup per forest and coordinate, a binary search per entry: 10 us for 100 forests, 49 us for
// 3000 (one wave for both coordinates: 68 us and 150 us).
__global__ __launch_bounds__(256) void dmat_table_kernel(DmatForests F, DmatListed T,
                                                         int32_t *__restrict__ tr,
                                                         int32_t *__restrict__ td) {
    const int64_t f = T.forest[blockIdx.x].forest;
    const int64_t o = F.off[f];
    const int n = (int)(F.off[f + 1] - o);
    if (n <= 0) return;
    const double *__restrict__ v = (blockIdx.y ? F.d : F.r) + o;
    int32_t *__restrict__ first = (blockIdx.y ? td : tr) + T.forest[blockIdx.x].at;
    const double v0 = v[0], h = band_mean_step(v0, v[n - 1], n);
    for (int k = threadIdx.x; k < n; k += 256) {
        const double x = v0 + k * h;
        int lo = 0;
        for (int m = n; m > 0;) {
            const int half = m >> 1;
            if (v[lo + half] < x) { lo += half + 1; m -= half + 1; }
            else m = half;
        }
        first[k] = lo;
    }
}

namespace {

__device__ __forceinline__ BandTable load_table(const int32_t *first, const double *v, int n) {
    const double v0 = uniform_f64(v[0]);
    return BandTable{first, v0, 1.0 / band_mean_step(v0, uniform_f64(v[n - 1]), n), n};
}

}  // namespace

__global__ __launch_bounds__(DMAT_BAND_PASS_BLOCK) void dmat_band_pass_kernel(
    XiConst M, DmatConst C, DmatForests F, DmatBandSlots P, DmatBandWork W, DmatOut O,
    int band_rows) {
    extern __shared__ __align__(16) unsigned char smem[];
    __shared__ unsigned long long s_in;
    __shared__ int s_special;
    __shared__ XiConst s_const;
    const int s = blockIdx.x;
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = tid >> 6;
    const BandPair q = load_band_pair(F, P, s);
    const int u0 = uniform_int(P.slot[s].u0), nu = uniform_int(P.slot[s].nu);
    const int t0 = uniform_int(P.slot[s].t0), nt = uniform_int(P.slot[s].nt);
    const int64_t urow = uniform_i64(P.slot[s].u_row), trow = uniform_i64(P.slot[s].t_row);
    const int64_t at_b = uniform_i64(P.slot[s].at_b);
    const int kp = C.npm / C.np, kt = C.ntm / C.nt;
    int32_t *rng = (int32_t *)smem;                       // [nu][4]
    double *acc = (double *)(smem + ((16 * (size_t)C.ntm + 15) & ~(size_t)15));
    for (int k = tid; k < nu; k += DMAT_BAND_PASS_BLOCK) {
        rng[4 * k] = rng[4 * k + 2] = INT_MAX;
        rng[4 * k + 1] = rng[4 * k + 3] = -1;
    }
    if (tid == 0) {
        s_in = 0;
        s_special = 0;
        s_const = M;   // published by the first __syncthreads below
    }
    const double *__restrict__ Br = F.r + q.ob;
    const double *__restrict__ Bd = F.d + q.ob;
    const double mul_t = q.sin_half * M.inv_t;
    uint64_t n_in = 0;
    for (int uc0 = u0; uc0 < u0 + nu; uc0 += band_rows) {
        const int rows = min(band_rows, u0 + nu - uc0);
        const int stride = rows * C.npm;
        for (int k = tid; k < DMAT_BAND_SUMS * stride; k += DMAT_BAND_PASS_BLOCK) acc[k] = 0.0;
        __syncthreads();
        for (int c0 = wave * 64; c0 < q.la; c0 += PASS_WAVES * 64) {
            const int i = c0 + lane;
            bool active = i < q.la;
            double r1 = 0, d1 = 0, z1 = 0, w1 = 0, l1 = 0, f1 = 0;
            if (active) {
                r1 = F.r[q.oa + i];
                d1 = F.d[q.oa + i];
                z1 = F.z[q.oa + i];
                w1 = F.w[q.oa + i];
                l1 = F.dll[q.oa + i];
                f1 = F.zfa[q.oa + i];
                active = w1 != 0;
            }
            if (__ballot(active) == 0) continue;
            // the wave's window of delta2, widened far above the rounding of the separations
            const double reach = C.rpmax / q.cos_half;
            double lo_r = wave_min(active ? r1 : INFINITY) - reach;
            double hi_r = wave_max(active ? r1 : -INFINITY) + reach;
            double d_lim = C.rtmax / q.sin_half - wave_min(active ? d1 : INFINITY);
            lo_r -= 1e-6 + 1e-12 * fabs(lo_r);
            hi_r += 1e-6 + 1e-12 * fabs(hi_r);
            d_lim += 1e-6 + 1e-12 * fabs(d_lim);
            WalkTask T;
            T.j_lo = uniform_int(wave_search<true>(Br, q.lb, lo_r, lane));
            T.j_hi = uniform_int(min(wave_search<false>(Br, q.lb, hi_r, lane),
                                     wave_search<false>(Bd, q.lb, d_lim, lane)));
            if (T.j_lo >= T.j_hi) continue;
            T.cos_half = q.cos_half;
            T.sin_half = q.sin_half;
            T.cp = uniform_f64(q.cos_half * M.inv_p);
            T.st = uniform_f64(mul_t);
            T.rc = uniform_f64(Br[q.lb >> 1]);
            T.dc = uniform_f64(Bd[q.lb >> 1]);
            T.q0 = 1.0;
            if (T.j_hi - T.j_lo >= 2) {
                const double span = (uniform_f64(Br[T.j_hi - 1]) - uniform_f64(Br[T.j_lo])) * T.cp;
                if (span > 0) T.q0 = (double)(T.j_hi - 1 - T.j_lo) / span;
            }
            WalkLane L{r1, d1, z1 * 0.5, w1, w1 * f1};
            L.j_lo = T.j_lo;
            L.j_hi = T.j_hi;
            if (nu > band_rows && active) {
                // the lane's pixels of this band of rows
                const BandAxis A = band_trans_axis(d1, mul_t, q.sin_half, C.rtmax, C.ntm,
                                                   M.fast_t);
                const BandTable B = load_table(W.table_d + at_b, Bd, q.lb);
                auto v = [&](int p) { return Bd[p]; };
                if (uc0 > u0) L.j_lo = max(T.j_lo, band_edge(A, B, v, uc0));
                if (uc0 + rows < u0 + nu) L.j_hi = min(T.j_hi, band_edge(A, B, v, uc0 + rows));
                if (L.j_lo >= L.j_hi) {
                    active = false;
                    L.j_lo = T.j_lo;
                }
            }
            BandPassMem mem{Br, Bd, F.w + q.ob, F.z + q.ob, W.pre_b + at_b, acc, rng,
                            &s_special, stride, nu, uc0 * C.npm, u0, i, l1, &s_const, 0, -1, 0, 0};
            walk_lane<false, true, DmatAcc>(M, T, L, mem, active);
            mem.note();
            n_in += mem.n_in;
        }
        __syncthreads();
        // this band's rows: S per data bin, eta5..eta8 and the effective sums per model bin
        for (int k = tid; k < rows / kt * C.np; k += DMAT_BAND_PASS_BLOCK) {
            const int tt = k / C.np, rp = k - tt * C.np;
            double sum[4] = {0, 0, 0, 0};
            for (int x = 0; x < kt; ++x)
                for (int y = 0; y < kp; ++y) {
                    const double *b = acc + (tt * kt + x) * C.npm + rp * kp + y;
                    for (int c = 0; c < 4; ++c) sum[c] += b[c * stride];
                }
            const int64_t row = trow + (uc0 - u0) / kt + tt;
            for (int c = 0; c < 4; ++c) W.S[(row * 4 + c) * C.np + rp] = sum[c];
        }
        for (int k = tid; k < stride; k += DMAT_BAND_PASS_BLOCK) {
            const int uu = k / C.npm, mrp = k - uu * C.npm;
            const double *b = acc + k;
            const int64_t row = urow + (uc0 - u0) + uu;
            double *e = W.eta + row * 4 * C.npm + mrp;
            e[0] = b[4 * stride] * q.inv_w1 * q.inv_w2;
            e[C.npm] = q.order2 ? b[5 * stride] * q.inv_w1 * q.inv_s2 : 0.0;
            e[2 * C.npm] = q.order1 ? b[6 * stride] * q.inv_s1 * q.inv_w2 : 0.0;
            e[3 * C.npm] = q.order1 && q.order2 ? b[7 * stride] * q.inv_s1 * q.inv_s2 : 0.0;
            double *f = W.eff + row * 5 * C.npm + mrp;
            f[0] = b[8 * stride];
            f[C.npm] = b[9 * stride];
            f[2 * C.npm] = b[10 * stride];
            f[3 * C.npm] = b[0];
            f[4 * C.npm] = b[4 * stride];
        }
        __syncthreads();
    }
    n_in = wave_sum_u64(n_in);
    if (lane == 0) atomicAdd(&s_in, (unsigned long long)n_in);
    __syncthreads();
    const bool special = s_special != 0;
    const bool live = !special && s_in > 0;
    if (tid == 0) {
        if (special) W.redo[atomicAdd(W.num_redo, 1)] = P.first + s;
        if (live) {
            atomicAdd(&W.stats[DMAT_STAT_IN_RANGE], s_in);
            atomicAdd(&W.stats[DMAT_STAT_SELECTED], s_in);
        }
    }
    // pixel ranges of the pair's rows; a row that the pair does not reach stays empty
    for (int k = tid; k < nu; k += DMAT_BAND_PASS_BLOCK)
        W.rng_u[urow + k] = live ? make_int4(rng[4 * k], rng[4 * k + 1], rng[4 * k + 2],
                                             rng[4 * k + 3])
                                 : make_int4(INT_MAX, -1, INT_MAX, -1);
    for (int k = tid; k < nt; k += DMAT_BAND_PASS_BLOCK) {
        int4 v = make_int4(INT_MAX, -1, INT_MAX, -1);
        for (int x = 0; x < kt && live; ++x) {
            const int32_t *r = rng + 4 * (k * kt + x);
            v = make_int4(min(v.x, r[0]), max(v.y, r[1]), min(v.z, r[2]), max(v.w, r[3]));
        }
        W.rng_t[trow + k] = v;
    }
    if (!live) return;   // uniform over the workgroup
    // (each thread reads back the workspace entries it wrote: the loops run as above)
    for (int uc0 = u0; uc0 < u0 + nu; uc0 += band_rows) {
        const int rows = min(band_rows, u0 + nu - uc0);
        for (int k = tid; k < rows / kt * C.np; k += DMAT_BAND_PASS_BLOCK) {
            const int tt = k / C.np, rp = k - tt * C.np;
            const int64_t row = trow + (uc0 - u0) / kt + tt;
            const double v = W.S[row * 4 * C.np + rp];
            const int t = t0 + (uc0 - u0) / kt + tt;
            if (v != 0) unsafeAtomicAdd(&O.weights_dmat[rp * C.nt + t], v);
        }
        for (int k = tid; k < rows * C.npm; k += DMAT_BAND_PASS_BLOCK) {
            const int uu = k / C.npm, mrp = k - uu * C.npm;
            const double *f = W.eff + (urow + (uc0 - u0) + uu) * 5 * C.npm + mrp;
            const int u = uc0 + uu;
            const int kb = mrp * C.ntm + u;
            if (f[0] != 0 || f[C.npm] != 0 || f[2 * C.npm] != 0 || f[3 * C.npm] != 0) {
                unsafeAtomicAdd(&O.r_par_eff[kb], f[0]);
                unsafeAtomicAdd(&O.r_trans_eff[kb], f[C.npm]);
                unsafeAtomicAdd(&O.z_eff[kb], f[2 * C.npm]);
                unsafeAtomicAdd(&O.weight_eff[kb], f[3 * C.npm]);
            }
            const int64_t A = (int64_t)(mrp / kp) * C.nt + u / kt;
            if (f[4 * C.npm] != 0) unsafeAtomicAdd(&O.dmat[A * C.nm + kb], f[4 * C.npm]);
        }
    }
}

// The rank-4 term needs every (t, u) of a pair with a non-empty row t and row u, also where no
// pixel reaches both; S and eta of such a tile are dense.
__global__ __launch_bounds__(256) void dmat_band_count_kernel(DmatConst C, DmatBandSlots P,
                                                              DmatBandWork W) {
    const int s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= P.count) return;
    const DmatBandSlot q = P.slot[s];
    for (int t = 0; t < q.nt; ++t) {
        const int4 rt = W.rng_t[q.t_row + t];
        if (rt.x > rt.y) continue;
        for (int u = 0; u < q.nu; ++u) {
            const int4 ru = W.rng_u[q.u_row + u];
            if (ru.x <= ru.y) atomicAdd(&W.tile_count[(q.t0 + t) * C.ntm + q.u0 + u], 1);
        }
    }
}

// One workgroup: list offsets of the tiles and their work items of at most item_pairs pairs.
__global__ __launch_bounds__(1024) void dmat_band_scan_kernel(int tiles, int item_pairs,
                                                              DmatBandWork W) {
    __shared__ int s_list[16], s_item[16];   // of a wave
    const int tid = threadIdx.x;
    const int per = (tiles + 1023) / 1024;
    const int k0 = min(tiles, tid * per), k1 = min(tiles, k0 + per);
    int n = 0, m = 0;
    for (int k = k0; k < k1; ++k) {
        n += W.tile_count[k];
        m += (W.tile_count[k] + item_pairs - 1) / item_pairs;
    }
    // exclusive sums over the threads: inside each wave, then over the waves
    int a = n, b = m;
    const int lane = tid & 63, wave = tid >> 6;
    for (int d = 1; d < 64; d <<= 1) {
        const int x = __shfl_up(a, d, 64), y = __shfl_up(b, d, 64);
        if (lane >= d) {
            a += x;
            b += y;
        }
    }
    if (lane == 63) {
        s_list[wave] = a;
        s_item[wave] = b;
    }
    __syncthreads();
    int before = 0, items_before = 0;
    for (int k = 0; k < wave; ++k) {
        before += s_list[k];
        items_before += s_item[k];
    }
    if (tid == 1023) {
        *W.num_items = items_before + b;
        *W.queue = 0;
    }
    int first = before + a - n, item = items_before + b - m;
    for (int k = k0; k < k1; ++k) {
        const int count = W.tile_count[k];
        W.tile_count[k] = first;   // fill position of the list kernel
        for (int c = 0; c < count; c += item_pairs)
            W.items[item++] = make_int4(k, first + c, min(item_pairs, count - c), 0);
        first += count;
    }
}

__global__ __launch_bounds__(256) void dmat_band_list_kernel(DmatConst C, DmatBandSlots P,
                                                             DmatBandWork W) {
    const int s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= P.count) return;
    const DmatBandSlot q = P.slot[s];
    for (int t = 0; t < q.nt; ++t) {
        const int4 rt = W.rng_t[q.t_row + t];
        if (rt.x > rt.y) continue;
        for (int u = 0; u < q.nu; ++u) {
            const int4 ru = W.rng_u[q.u_row + u];
            if (ru.x <= ru.y)
                W.list[atomicAdd(&W.tile_count[(q.t0 + t) * C.ntm + q.u0 + u], 1)] = s;
        }
    }
}

namespace {

// The sums per r_par bin of one pixel per group of 16 lanes over its partner's pixels [j0, j1),
// whose bins are k0 .. k0 + kn - 1: lane li takes bin edges 15 at a time, and add(k, x, y,
// first, end) gets a bin, the differences of the two prefix sums over its pixels [first, end).
// pre: the prefix records' pair of sums (stride 4).  Every lane of the wave takes part.
template <class Add>
__device__ __forceinline__ void band_bins(const BandAxis &A, const BandTable &T,
                                          const double *__restrict__ v,
                                          const double2 *__restrict__ pre, int j0, int j1, int k0,
                                          int kn, int li, Add add) {
    const int groups = wave_max_int((kn + 14) / 15);
    for (int g = 0; g < groups; ++g) {
        // lane li: the first pixel of bin k; the sums of bin k lie between its edge and the
        // next lane's
        const int at = 15 * g + li;
        const int k = k0 + at;
        double2 here = make_double2(0.0, 0.0);
        int e = 0;
        if (at <= kn && kn > 0) {
            e = at == 0 ? j0 : j1;
            if (at > 0 && at < kn) e = band_edge(A, T, [&](int p) { return v[p]; }, k);
            here = pre[4 * (int64_t)e];
        }
        const double x = dpp_f64<DPP_ROW_SHL1>(here.x) - here.x;
        const double y = dpp_f64<DPP_ROW_SHL1>(here.y) - here.y;
        const int end = dpp_int<DPP_ROW_SHL1>(e);
        if (at < kn && li < 15) add(k, x, y, e, end);
    }
}

}  // namespace

__global__ __launch_bounds__(DMAT_BAND_FILL_BLOCK, 3) void dmat_band_fill_kernel(
    XiConst M, DmatConst C, DmatForests F, DmatBandSlots P, DmatBandWork W, DmatOut O) {
    extern __shared__ __align__(16) double panel[];   // [PX][VLEN]
    __shared__ int s_item;
    __shared__ unsigned int s_cols;   // 16-column blocks of eta with an entry, of this panel
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = tid >> 6;
    // v_mfma_f64_16x16x4f64 operands: lane l holds A[l % 16][l / 16] and B[l / 16][l % 16];
    // register r of the result holds row 4 r + l / 16, column l % 16 of the 16 x 16 block.
    // Wave w owns the data r_par bins 16 w .. 16 w + 15 of the chunk and every model bin.
    const int li = lane & 15;
    const int lk = lane >> 4;
    const int row = 16 * wave + li;
    uint32_t n_mfma = 0;
    for (;;) {
        __syncthreads();
        if (tid == 0) s_item = atomicAdd(W.queue, 1);
        __syncthreads();
        const int item = s_item;
        if (item >= *W.num_items) break;
        const int4 work = W.items[item];
        const int tile = uniform_int(work.x);
        const int t = tile / C.ntm, u = tile - t * C.ntm;
        for (int rp0 = 0; rp0 < C.np; rp0 += DMAT_CHUNK_RP) {
            for (int mrp0 = 0; mrp0 < C.npm; mrp0 += DMAT_CHUNK_MRP) {
                const int nrp = min(DMAT_CHUNK_RP, C.np - rp0);
                const int nmrp = min(DMAT_CHUNK_MRP, C.npm - mrp0);
                double4_t acc[FILL_CB];
#pragma unroll
                for (int b = 0; b < FILL_CB; ++b) acc[b] = (double4_t){0.0, 0.0, 0.0, 0.0};
                for (int e = 0; e < work.z; ++e) {
                    const int s = uniform_int(W.list[work.y + e]);
                    const BandPair q = load_band_pair(F, P, s);
                    const int64_t trow = uniform_i64(P.slot[s].t_row) +
                                         (t - uniform_int(P.slot[s].t0));
                    const int64_t urow = uniform_i64(P.slot[s].u_row) +
                                         (u - uniform_int(P.slot[s].u0));
                    // rank-4 term S[., t] x eta5..8[., u]: one K = 4 product per block
                    double *vS = panel, *vE = panel + 4 * DMAT_CHUNK_RP;
                    __syncthreads();   // the last panel has been read
                    for (int k = tid; k < 4 * DMAT_CHUNK_RP; k += DMAT_BAND_FILL_BLOCK) {
                        const int c = k / DMAT_CHUNK_RP, r = k - c * DMAT_CHUNK_RP;
                        vS[k] = r < nrp ? W.S[(trow * 4 + c) * C.np + rp0 + r] : 0.0;
                    }
                    for (int k = tid; k < 4 * DMAT_CHUNK_MRP; k += DMAT_BAND_FILL_BLOCK) {
                        const int c = k / DMAT_CHUNK_MRP, m = k - c * DMAT_CHUNK_MRP;
                        vE[k] = m < nmrp ? W.eta[(urow * 4 + c) * C.npm + mrp0 + m] : 0.0;
                    }
                    __syncthreads();
                    const double sa = vS[lk * DMAT_CHUNK_RP + row];
                    if (__ballot(sa != 0.0) != 0) {
                        n_mfma += FILL_CB;
#pragma unroll
                        for (int b = 0; b < FILL_CB; ++b)
                            acc[b] = __builtin_amdgcn_mfma_f64_16x16x4f64(
                                sa, vE[lk * DMAT_CHUNK_MRP + 16 * b + li], acc[b], 0, 0, 0);
                    }
                    const int4 rt = W.rng_t[trow], ru = W.rng_u[urow];
                    // bins per unit of r_comov and dist_m: data and model
                    const double mul_pd = q.cos_half * C.np / C.span_p;
                    const double mul_pm = q.cos_half * C.npm / C.span_p;
                    const double mul_td = q.sin_half * C.nt / C.rtmax;
                    const double mul_tm = q.sin_half * C.ntm / C.rtmax;
                    // pixels of delta1 (their partners: delta2), then of delta2
                    for (int side = 0; side < 2; ++side) {
                        const int64_t os = side ? q.ob : q.oa, op = side ? q.oa : q.ob;
                        const int np_ = side ? q.la : q.lb;   // pixels of the partner
                        const double *__restrict__ Pr = F.r + op;
                        const double *__restrict__ Pd = F.d + op;
                        const int64_t at = uniform_i64(side ? P.slot[s].at_a   // of the partner
                                                            : P.slot[s].at_b);
                        const double2 *__restrict__ pre =
                            (const double2 *)((side ? W.pre_a : W.pre_b) + at);
                        const BandTable Tr = load_table(W.table_r + at, Pr, np_);
                        const BandTable Td = load_table(W.table_d + at, Pd, np_);
                        const double inv_w = side ? q.inv_w1 : q.inv_w2;
                        const double inv_s = side ? (q.order1 ? q.inv_s1 : 0.0)
                                                  : (q.order2 ? q.inv_s2 : 0.0);
                        const double *__restrict__ zf = (side ? F.zfb : F.zfa) + os;
                        const int p0 = uniform_int(side ? max(rt.z, ru.z) : max(rt.x, ru.x));
                        const int p1 = uniform_int(side ? min(rt.w, ru.w) : min(rt.y, ru.y));
                        for (int base = p0; base <= p1; base += PX) {
                            __syncthreads();   // the last panel (or the rank-4 rows) is read
                            for (int k = tid; k < PX * VLEN / 2; k += DMAT_BAND_FILL_BLOCK)
                                ((double2 *)panel)[k] = make_double2(0.0, 0.0);
                            if (tid == 0) s_cols = 0;
                            // lane group lk: pixel base + 4 wave + lk
                            const int p = base + 4 * wave + lk;
                            const int64_t ps = os + min(p, p1);
                            const double rs = F.r[ps], ds = F.d[ps];
                            const double ws = p <= p1 ? F.w[ps] : 0.0;
                            const double fz = zf[min(p, p1)];
                            // edges of the partner's pixels in row t (lanes 0, 1), in row u
                            // (2, 3) and in the r_par range (4, 5)
                            int edge = 0;
                            if (li < 6 && ws != 0) {
                                const bool par = li >= 4, model = li >= 2;
                                const BandAxis A =
                                    par ? band_par_axis(rs, mul_pm, q.cos_half, C.span_p, C.npm,
                                                        M.fast_p)
                                        : band_trans_axis(ds, model ? mul_tm : mul_td,
                                                          q.sin_half, C.rtmax,
                                                          model ? C.ntm : C.nt, M.fast_t);
                                const int K = par ? (li == 4 ? -C.npm : C.npm)
                                                  : (model ? u : t) + (li & 1);
                                const double *__restrict__ V = par ? Pr : Pd;
                                edge = band_edge(A, par ? Tr : Td, [&](int x) { return V[x]; },
                                                 K);
                            }
                            const int first = lane & 48;
                            const int r_lo = __shfl(edge, first + 4, 64);
                            const int r_hi = __shfl(edge, first + 5, 64);
                            int j0[2], j1[2], k0[2], kn[2];
#pragma unroll
                            for (int h = 0; h < 2; ++h) {   // 0: data bins in row t, 1: model, u
                                j0[h] = max(__shfl(edge, first + 2 * h, 64), r_lo);
                                j1[h] = min(__shfl(edge, first + 2 * h + 1, 64), r_hi);
                                // r_par bins of the first and last of these pixels
                                const BandAxis A = band_par_axis(
                                    rs, h ? mul_pm : mul_pd, q.cos_half, C.span_p,
                                    h ? C.npm : C.np, M.fast_p);
                                k0[h] = kn[h] = 0;
                                if (j0[h] < j1[h]) {
                                    k0[h] = band_key(A, Pr[j0[h]]);
                                    kn[h] = band_key(A, Pr[j1[h] - 1]) - k0[h] + 1;
                                }
                            }
                            __syncthreads();
                            double *px = panel + (4 * wave + lk) * VLEN;
                            uint32_t cols = 0;
#pragma unroll
                            for (int h = 0; h < 2; ++h) {
                                const int bins = h ? C.npm : C.np;
                                const BandAxis A = band_par_axis(rs, h ? mul_pm : mul_pd,
                                                                 q.cos_half, C.span_p, bins,
                                                                 M.fast_p);
                                const double f1 = h ? fz * inv_w : ws;
                                const double f2 = h ? fz * inv_s : ws;
                                const int chunk = h ? mrp0 : rp0, count = h ? nmrp : nrp;
                                double *dst = px + (h ? VE : VP);
                                const int second = h ? VE2 - VE : VP2 - VP;
                                band_bins(A, Tr, Pr, pre + h, j0[h], j1[h], k0[h], kn[h], li,
                                          [&](int k, double x, double y, int, int) {
                                    const int b = (k >= 0 ? k : -k - 1) - chunk;
                                    if (b < 0 || b >= count) return;
                                    if (h) cols |= 1u << (b >> 4);
                                    lds_add(dst + b, f1 * x);
                                    lds_add(dst + second + b, f2 * y);
                                });
                            }
                            if (cols) atomicOr(&s_cols, cols);
                            __syncthreads();
                            // acc -= P x eta + P' x eta', K = the pixels, four at a time
                            const uint32_t blocks = (uint32_t)uniform_int((int)s_cols);
#pragma unroll
                            for (int k4 = 0; k4 < PX / 4; ++k4) {
                                const double *v = panel + (4 * k4 + lk) * VLEN;
                                const double a1 = -v[VP + row], a2 = -v[VP2 + row];
                                // no pair of these pixels in this wave's data bins
                                if (__ballot(a1 != 0.0 || a2 != 0.0) == 0) continue;
#pragma unroll
                                for (int b = 0; b < FILL_CB; ++b) {
                                    if (!((blocks >> b) & 1u)) continue;
                                    n_mfma += 2;
                                    acc[b] = __builtin_amdgcn_mfma_f64_16x16x4f64(
                                        a1, v[VE + 16 * b + li], acc[b], 0, 0, 0);
                                    acc[b] = __builtin_amdgcn_mfma_f64_16x16x4f64(
                                        a2, v[VE2 + 16 * b + li], acc[b], 0, 0, 0);
                                }
                            }
                        }
                    }
                }
                // block -> dmat
#pragma unroll
                for (int a = 0; a < 4; ++a) {
                    const int r = 16 * wave + 4 * a + lk;
#pragma unroll
                    for (int b = 0; b < FILL_CB; ++b) {
                        const int m = 16 * b + li;
                        if (r < nrp && m < nmrp && acc[b][a] != 0) {
                            const int64_t A = (int64_t)(rp0 + r) * C.nt + t;
                            const int64_t k = (int64_t)(mrp0 + m) * C.ntm + u;
                            unsafeAtomicAdd(&O.dmat[A * C.nm + k], acc[b][a]);
                        }
                    }
                }
            }
        }
    }
    if (lane == 0 && n_mfma) atomicAdd(&W.stats[DMAT_STAT_MFMA], (unsigned long long)n_mfma);
}

// ---------------------------------------------------------------------------------------
// Forest x quasar pairs: delta2 is one unprojected pixel (py/picca/xcf.py:427-658), whose pairs
// leave the identity and the Q eta2 + Q' eta4 terms.  No pass: a pair's rows come from its
// edges, the matrix-core panel holds 16 pairs (K = the pairs), and the tile of a data row and
// its own model rows adds the pair-bin term, weights_dmat and the effective sums.  With a pair
// per workgroup and one quasar pixel a tile, the general pass and fill leave 15 of 16 lanes and
// rows of K idle: 3000 forests, 145k kept pairs, 100 x 50 bins take 2.4 ms here, 36 ms (fill) and
// 11 ms (pass) there.  Bound by the chain of table, probe and prefix loads of an edge.

// Rows that each pair reaches (as non-empty pixel ranges for the tile lists), and the pairs
// whose bins do not follow the runs: a pixel at the end of a range whose bin rounds past it, or
// r_par == r_par_min exactly, which xcf's count pass leaves out.  One thread per pair.
__global__ __launch_bounds__(256) void dmat_quasar_rows_kernel(XiConst M, DmatConst C,
                                                               DmatForests F, DmatBandSlots P,
                                                               DmatBandWork W) {
    const int s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= P.count) return;
    const DmatBandSlot q = P.slot[s];
    const int64_t oa = F.off[q.a], ob = F.off[q.b];
    const int n = (int)(F.off[q.a + 1] - oa);
    const double *__restrict__ R = F.r + oa;
    const double *__restrict__ D = F.d + oa;
    const double cos_half = P.cs[2 * s], sin_half = P.cs[2 * s + 1];
    const double rq = F.r[ob], dq = F.d[ob];
    const BandTable Tr{W.table_r + q.at_a, R[0], 1.0 / band_mean_step(R[0], R[n - 1], n), n};
    const BandTable Td{W.table_d + q.at_a, D[0], 1.0 / band_mean_step(D[0], D[n - 1], n), n};
    auto r = [&](int p) { return R[p]; };
    auto d = [&](int p) { return D[p]; };
    const BandAxis Ap = band_signed_axis(rq, cos_half * C.npm / C.span_p, cos_half, C.rpmin,
                                         C.span_p, C.npm, M.fast_p);
    const int lo = band_edge(Ap, Tr, r, 0), hi = band_edge(Ap, Tr, r, C.npm);
    const BandAxis At = band_trans_axis(dq, sin_half * C.ntm / C.rtmax, sin_half, C.rtmax, C.ntm,
                                        M.fast_t);
    const int top = band_edge(At, Td, d, C.ntm);
    const bool special = (lo < n && !((R[lo] - rq) * cos_half > C.rpmin)) ||
                         (hi < n && (R[hi] - rq) * cos_half < C.rpmax) ||
                         (top < n && (D[top] + dq) * sin_half < C.rtmax);
    if (special) W.redo[atomicAdd(W.num_redo, 1)] = P.first + s;
    const int4 empty = make_int4(INT_MAX, -1, INT_MAX, -1), full = make_int4(0, 0, 0, 0);
    int first = band_edge(At, Td, d, q.u0);
    const int kt = C.ntm / C.nt;
    bool any = false;
    for (int u = 0; u < q.nu; ++u) {
        const int end = band_edge(At, Td, d, q.u0 + u + 1);
        const bool in = !special && max(first, lo) < min(end, hi);
        W.rng_u[q.u_row + u] = in ? full : empty;
        any = any || in;
        if ((u + 1) % kt == 0) {
            W.rng_t[q.t_row + u / kt] = any ? full : empty;
            any = false;
        }
        first = end;
    }
}

__global__ __launch_bounds__(DMAT_BAND_FILL_BLOCK, 3) void dmat_quasar_fill_kernel(
    XiConst M, DmatConst C, DmatForests F, DmatBandSlots P, DmatBandWork W, DmatOut O) {
    extern __shared__ __align__(16) double panel[];   // [PX][VLEN]
    // effective sums, weight and pair-bin term of the tile's model bins (own rows' tiles only)
    __shared__ double s_eff[5][DMAT_CHUNK_MRP];
    __shared__ int s_item;
    __shared__ unsigned int s_cols;
    __shared__ unsigned long long s_in;
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = tid >> 6;
    const int li = lane & 15;
    const int lk = lane >> 4;
    const int row = 16 * wave + li;
    const int kp = C.npm / C.np, kt = C.ntm / C.nt;
    uint32_t n_mfma = 0;
    for (;;) {
        __syncthreads();
        if (tid == 0) {
            s_item = atomicAdd(W.queue, 1);
            s_in = 0;
        }
        __syncthreads();
        const int item = s_item;
        if (item >= *W.num_items) break;
        const int4 work = W.items[item];
        const int tile = uniform_int(work.x);
        const int t = tile / C.ntm, u = tile - t * C.ntm;
        const bool own = u / kt == t;   // model row u lies in data row t
        for (int rp0 = 0; rp0 < C.np; rp0 += DMAT_CHUNK_RP) {
            for (int mrp0 = 0; mrp0 < C.npm; mrp0 += DMAT_CHUNK_MRP) {
                const int nrp = min(DMAT_CHUNK_RP, C.np - rp0);
                const int nmrp = min(DMAT_CHUNK_MRP, C.npm - mrp0);
                const bool eff = own && rp0 == 0;
                double4_t acc[FILL_CB];
#pragma unroll
                for (int b = 0; b < FILL_CB; ++b) acc[b] = (double4_t){0.0, 0.0, 0.0, 0.0};
                for (int k = tid; k < 5 * DMAT_CHUNK_MRP; k += DMAT_BAND_FILL_BLOCK)
                    (&s_eff[0][0])[k] = 0.0;
                for (int base = 0; base < work.z; base += PX) {
                    __syncthreads();   // the last panel is read
                    for (int k = tid; k < PX * VLEN / 2; k += DMAT_BAND_FILL_BLOCK)
                        ((double2 *)panel)[k] = make_double2(0.0, 0.0);
                    if (tid == 0) s_cols = 0;
                    // lane group lk: pair base + 4 wave + lk of the item
                    const int e = base + 4 * wave + lk;
                    const int s = W.list[work.y + min(e, work.z - 1)];
                    const DmatBandSlot q = P.slot[s];
                    const int64_t oa = F.off[q.a], ob = F.off[q.b];
                    const int n = (int)(F.off[q.a + 1] - oa);
                    const double *__restrict__ Pr = F.r + oa;
                    const double *__restrict__ Pd = F.d + oa;
                    const DmatPrefix *__restrict__ rec = W.pre_a + q.at_a;
                    const double2 *__restrict__ pre = (const double2 *)rec;
                    const BandTable Tr{W.table_r + q.at_a, Pr[0],
                                       1.0 / band_mean_step(Pr[0], Pr[n - 1], n), n};
                    const BandTable Td{W.table_d + q.at_a, Pd[0],
                                       1.0 / band_mean_step(Pd[0], Pd[n - 1], n), n};
                    const double cos_half = P.cs[2 * s], sin_half = P.cs[2 * s + 1];
                    const double rq = F.r[ob], dq = F.d[ob], zq = F.z[ob];
                    const double wq = e < work.z ? F.w[ob] : 0.0;
                    const double fq = F.zfb[ob];
                    auto par = [&](bool model) {
                        const int bins = model ? C.npm : C.np;
                        return band_signed_axis(rq, cos_half * bins / C.span_p, cos_half,
                                                C.rpmin, C.span_p, bins, M.fast_p);
                    };
                    int edge = 0;
                    if (li < 6 && wq != 0) {
                        const bool p = li >= 4, model = li >= 2;
                        const int bins = model ? C.ntm : C.nt;
                        const BandAxis A =
                            p ? par(true)
                              : band_trans_axis(dq, sin_half * bins / C.rtmax, sin_half, C.rtmax,
                                                bins, M.fast_t);
                        const int K = p ? (li == 4 ? 0 : C.npm) : (model ? u : t) + (li & 1);
                        const double *__restrict__ V = p ? Pr : Pd;
                        edge = band_edge(A, p ? Tr : Td, [&](int x) { return V[x]; }, K);
                    }
                    const int first = lane & 48;
                    const int r_lo = __shfl(edge, first + 4, 64);
                    const int r_hi = __shfl(edge, first + 5, 64);
                    int j0[2], j1[2], k0[2], kn[2];
#pragma unroll
                    for (int h = 0; h < 2; ++h) {
                        j0[h] = max(__shfl(edge, first + 2 * h, 64), r_lo);
                        j1[h] = min(__shfl(edge, first + 2 * h + 1, 64), r_hi);
                        k0[h] = kn[h] = 0;
                        if (j0[h] < j1[h]) {
                            const BandAxis A = par(h != 0);
                            k0[h] = band_key(A, Pr[j0[h]]);
                            kn[h] = band_key(A, Pr[j1[h] - 1]) - k0[h] + 1;
                        }
                    }
                    const double inv_w = 1.0 / F.sum_w[q.a];
                    const double inv_s = F.order[q.a] == 1 ? 1.0 / F.sw_dll[q.a] : 0.0;
                    __syncthreads();
                    double *px = panel + (4 * wave + lk) * VLEN;
                    uint32_t cols = 0;
                    if (eff && mrp0 == 0 && li == 0 && kn[1] > 0)
                        atomicAdd(&s_in, (unsigned long long)(rec[j1[1]].c - rec[j0[1]].c));
                    band_bins(par(false), Tr, Pr, pre, j0[0], j1[0], k0[0], kn[0], li,
                              [&](int k, double x, double y, int, int) {
                        const int b = k - rp0;
                        if (b < 0 || b >= nrp) return;
                        lds_add(px + VP + b, wq * x);
                        lds_add(px + VP2 + b, wq * y);
                    });
                    band_bins(par(true), Tr, Pr, pre + 1, j0[1], j1[1], k0[1], kn[1], li,
                              [&](int k, double x, double y, int j, int end) {
                        const int b = k - mrp0;
                        if (b < 0 || b >= nmrp) return;
                        cols |= 1u << (b >> 4);
                        lds_add(px + VE + b, fq * inv_w * x);
                        lds_add(px + VE2 + b, fq * inv_s * y);
                        if (!eff) return;
                        // over the bin's pixels: w2 sum w1 (r1 - r2) cos and so on
                        const DmatPrefix a = rec[j], z = rec[end];
                        const double w = wq * (z.w - a.w);
                        const double rc = Pr[n / 2], dc = Pd[n / 2];
                        lds_add(&s_eff[0][b], cos_half * (wq * (z.r - a.r) + (rc - rq) * w));
                        lds_add(&s_eff[1][b], sin_half * (wq * (z.d - a.d) + (dc + dq) * w));
                        lds_add(&s_eff[2][b], 0.5 * (wq * (z.z - a.z) + zq * w));
                        lds_add(&s_eff[3][b], w);
                        lds_add(&s_eff[4][b], wq * fq * x);
                    });
                    if (cols) atomicOr(&s_cols, cols);
                    __syncthreads();
                    // acc -= Q x eta2 + Q' x eta4, K = the pairs, four at a time
                    const uint32_t blocks = (uint32_t)uniform_int((int)s_cols);
#pragma unroll
                    for (int k4 = 0; k4 < PX / 4; ++k4) {
                        const double *v = panel + (4 * k4 + lk) * VLEN;
                        const double a1 = -v[VP + row], a2 = -v[VP2 + row];
                        if (__ballot(a1 != 0.0 || a2 != 0.0) == 0) continue;
#pragma unroll
                        for (int b = 0; b < FILL_CB; ++b) {
                            if (!((blocks >> b) & 1u)) continue;
                            n_mfma += 2;
                            acc[b] = __builtin_amdgcn_mfma_f64_16x16x4f64(
                                a1, v[VE + 16 * b + li], acc[b], 0, 0, 0);
                            acc[b] = __builtin_amdgcn_mfma_f64_16x16x4f64(
                                a2, v[VE2 + 16 * b + li], acc[b], 0, 0, 0);
                        }
                    }
                }
                __syncthreads();
                // block -> dmat
#pragma unroll
                for (int a = 0; a < 4; ++a) {
                    const int r = 16 * wave + 4 * a + lk;
#pragma unroll
                    for (int b = 0; b < FILL_CB; ++b) {
                        const int m = 16 * b + li;
                        if (r < nrp && m < nmrp && acc[b][a] != 0) {
                            const int64_t A = (int64_t)(rp0 + r) * C.nt + t;
                            const int64_t k = (int64_t)(mrp0 + m) * C.ntm + u;
                            unsafeAtomicAdd(&O.dmat[A * C.nm + k], acc[b][a]);
                        }
                    }
                }
                if (eff) {
                    for (int m = tid; m < nmrp; m += DMAT_BAND_FILL_BLOCK) {
                        const int kb = (mrp0 + m) * C.ntm + u;
                        const int64_t A = (int64_t)((mrp0 + m) / kp) * C.nt + t;
                        if (s_eff[3][m] != 0)
                            unsafeAtomicAdd(&O.weights_dmat[A], s_eff[3][m]);
                        if (s_eff[3][m] != 0 || s_eff[0][m] != 0 || s_eff[1][m] != 0 ||
                            s_eff[2][m] != 0) {
                            unsafeAtomicAdd(&O.r_par_eff[kb], s_eff[0][m]);
                            unsafeAtomicAdd(&O.r_trans_eff[kb], s_eff[1][m]);
                            unsafeAtomicAdd(&O.z_eff[kb], s_eff[2][m]);
                            unsafeAtomicAdd(&O.weight_eff[kb], s_eff[3][m]);
                        }
                        if (s_eff[4][m] != 0) unsafeAtomicAdd(&O.dmat[A * C.nm + kb], s_eff[4][m]);
                    }
                }
                __syncthreads();
            }
        }
        if (tid == 0 && s_in) {
            atomicAdd(&W.stats[DMAT_STAT_IN_RANGE], s_in);
            atomicAdd(&W.stats[DMAT_STAT_SELECTED], s_in);
        }
    }
    if (lane == 0 && n_mfma) atomicAdd(&W.stats[DMAT_STAT_MFMA], (unsigned long long)n_mfma);
}

size_t dmat_band_pass_lds(const DmatConst &C, int rows) {
    return ((16 * (size_t)C.ntm + 15) & ~(size_t)15) +
           sizeof(double) * DMAT_BAND_SUMS * (size_t)C.npm * rows;
}

hipError_t launch_dmat_prefix(const DmatForests &F, const DmatListed &T, DmatPrefix *pa,
                              DmatPrefix *pb, int32_t *table_r, int32_t *table_d,
                              hipStream_t stream) {
    if (T.count <= 0) return hipSuccess;
    const dim3 forests((unsigned)T.count);
    if (pb)
        hipLaunchKernelGGL(dmat_prefix_kernel<true>, forests, dim3(64), 0, stream, F, T, pa, pb);
    else
        hipLaunchKernelGGL(dmat_prefix_kernel<false>, forests, dim3(64), 0, stream, F, T, pa, pb);
    hipLaunchKernelGGL(dmat_table_kernel, dim3((unsigned)T.count, 2), dim3(256), 0, stream, F, T,
                       table_r, table_d);
    return hipGetLastError();
}

hipError_t launch_dmat_band_pass(const XiConst &M, const DmatConst &C, const DmatForests &F,
                                 const DmatBandSlots &P, const DmatBandWork &W,
                                 const DmatOut &O, int band_rows, hipStream_t stream) {
    if (P.count <= 0) return hipSuccess;
    const size_t lds = dmat_band_pass_lds(C, band_rows);
    hipError_t err = hipFuncSetAttribute((const void *)dmat_band_pass_kernel,
                                         hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (err != hipSuccess) return err;
    hipLaunchKernelGGL(dmat_band_pass_kernel, dim3(P.count), dim3(DMAT_BAND_PASS_BLOCK), lds,
                       stream, M, C, F, P, W, O, band_rows);
    return hipGetLastError();
}

// the work items of the tiles, whose rows the pass or the rows kernel has set
static hipError_t launch_tile_lists(const DmatConst &C, const DmatBandSlots &P,
                                    const DmatBandWork &W, int item_pairs, hipStream_t stream) {
    const dim3 pairs((unsigned)((P.count + 255) / 256));
    hipLaunchKernelGGL(dmat_band_count_kernel, pairs, dim3(256), 0, stream, C, P, W);
    hipLaunchKernelGGL(dmat_band_scan_kernel, dim3(1), dim3(1024), 0, stream, C.nt * C.ntm,
                       item_pairs, W);
    hipLaunchKernelGGL(dmat_band_list_kernel, pairs, dim3(256), 0, stream, C, P, W);
    return hipGetLastError();
}

hipError_t launch_dmat_band_fill(const XiConst &M, const DmatConst &C, const DmatForests &F,
                                 const DmatBandSlots &P, const DmatBandWork &W,
                                 const DmatOut &O, bool quasar, int num_cus,
                                 hipStream_t stream) {
    if (P.count <= 0) return hipSuccess;
    hipError_t err = launch_tile_lists(C, P, W, quasar ? DMAT_QUASAR_ITEM : DMAT_BAND_ITEM, stream);
    if (err != hipSuccess) return err;
    const size_t lds = sizeof(double) * PX * VLEN;
    auto kern = quasar ? dmat_quasar_fill_kernel : dmat_band_fill_kernel;
    err = hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize,
                              (int)lds);
    if (err != hipSuccess) return err;
    hipLaunchKernelGGL(kern, dim3(3 * num_cus), dim3(DMAT_BAND_FILL_BLOCK), lds, stream, M, C, F,
                       P, W, O);
    return hipGetLastError();
}

hipError_t launch_dmat_quasar_rows(const XiConst &M, const DmatConst &C, const DmatForests &F,
                                   const DmatBandSlots &P, const DmatBandWork &W,
                                   hipStream_t stream) {
    if (P.count <= 0) return hipSuccess;
    hipLaunchKernelGGL(dmat_quasar_rows_kernel, dim3((unsigned)((P.count + 255) / 256)),
                       dim3(256), 0, stream, M, C, F, P, W);
    return hipGetLastError();
}

}  // namespace picca
