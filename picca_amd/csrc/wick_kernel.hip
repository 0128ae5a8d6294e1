// Wick covariance terms T1, T2, T3 of the auto-correlation on gfx950 (MI355X):
// compute_wickT123_pairs of py/picca/cf.py:1486-1602 for a batch of forest pairs.
//
// For each pair the reference lists its in-range pixel pairs (i, j) with bin p, adds
// w1w2 to weights_wick[p], 1 to num_pairs_wick[p] and w1w2 zev1 zev2 to T1[p, p], and then,
// for every two listed pairs a < b, adds one product to [p_a, p_b] and [p_b, p_a]:
//     i_a == i_b:  Wx2[j_a, j_b] w1[i] zev1[i]                        -> T2
//     j_a == j_b:  Wx1[i_a, i_b] w2[j] zev2[j]                        -> T2
//     otherwise:   Wx1[i_a, i_b] Wx2[j_a, j_b]                        -> T3
// (Wx the forests' weighted 1-D correlations).  That is T[P, Q] = sum over a in P, b in Q,
// b != a, of the product.  The pixel pairs of one pixel j in one bin are runs of consecutive i
// (segments); over two segments a and b the products share Wx2[j_a, j_b] (or w2 zev2), so their
// sum needs only
//     D = sum_{i_a in a} sum_{i_b in b} Wx1[i_a, i_b],
// less the terms i_a == i_b, which are T2 products with w1 zev1 (or a itself for j_a == j_b):
//   wick_segment_kernel  a thread per pixel j of a pair walks the pixels i: first the segments
//                     per bin, the bins' sums and T1, then (after a prefix sum) the segments
//                     themselves, by bin; wick_sort_kernel orders each bin's by j;
//   wick_rsum_kernel  a wave per segment a: the prefix sums over i_b of sum_{i_a in a}
//                     Wx1[i_a, i_b];
//   wick_row_kernel   one workgroup per task (pair, bin P) and part of the pair's segments b,
//                     one segment per lane: the segments a of P are staged through LDS and
//                     walked in step, D being one difference of a's prefix sums, and each lane's
//                     sums go to an LDS row of T2 / T3 (at its segment's bin), which goes to
//                     HBM at the end.
// A step per two segments replaces one per pixel pair and segment (7 pixels a segment on the
// 0.8 A grid), and the prefix sums of every row of Wx1, which took 7.0 ms of the kernels' 22 ms
// on 24 pairs (2.6e7 values of Wx) where the segments' sums take 0.49 ms and the rows 2.2 ms
// (11.1 ms before); the pixel pairs are walked by a thread per pixel of delta2 (twice 0.3 ms on
// those pairs, 3.6 ms for one workgroup per pair).
// FP64 throughout; bins by truncation after divide-then-multiply, as the reference.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "device_util.h"
#include "engine.h"

namespace picca {

namespace {

__device__ __forceinline__ void lds_add(double *p, double v) {
    __hip_atomic_fetch_add(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

// bin of pixel pair (i, j) or -1 when out of range; r_trans from the comoving distances
__device__ __forceinline__ int wick_bin(const WickConst &C, double r1, double r2, double c,
                                        double s) {
    double r_par = (r1 - r2) * c;
    if (!C.xcorr) r_par = fabs(r_par);
    const double r_trans = (r1 + r2) * s;
    if (!(r_par < C.rpmax && r_trans < C.rtmax && r_par >= C.rpmin)) return -1;
    const int bp = (int)((r_par - C.rpmin) / C.span * C.np);
    const int bt = (int)(r_trans / C.rtmax * C.nt);
    const int p = bt + C.nt * bp;
    return p < C.nb ? p : -2;   // -2: rounds up to np (the reference writes out of bounds)
}

}  // namespace

// PLACE false: per pair and bin the number of segments, and the bins' sums and T1.  PLACE true:
// the segments, at the positions that seg_pos holds.
template <bool PLACE>
__global__ __launch_bounds__(WICK_BLOCK) void wick_segment_kernel(WickConst C, WickInputs I,
                                                                  WickPairs P, WickWork W,
                                                                  WickOut O) {
    extern __shared__ __align__(16) unsigned char smem[];
    double *hw = (double *)smem;          // [nb] sum w1 w2
    double *ht = hw + C.nb;               // [nb] sum w1 w2 zev1 zev2
    int *cnt = (int *)(ht + C.nb);        // [nb] pixel pairs per bin
    int *scnt = cnt + C.nb;               // [nb] segments per bin
    __shared__ unsigned long long s_over, s_in;
    const int s = blockIdx.y;
    const int tid = threadIdx.x;
    const int a = uniform_int(P.a[s]), b = uniform_int(P.b[s]);
    const int64_t oa = uniform_i64(I.off[a]), ob = uniform_i64(I.off[b]);
    const int n1 = (int)(uniform_i64(I.off[a + 1]) - oa);
    const int n2 = (int)(uniform_i64(I.off[b + 1]) - ob);
    if ((int)(blockIdx.x * WICK_BLOCK) >= n2) return;
    const double c = uniform_f64(P.cs[2 * s]), sn = uniform_f64(P.cs[2 * s + 1]);
    if (!PLACE) {
        for (int k = tid; k < C.nb; k += WICK_BLOCK) {
            hw[k] = 0.0;
            ht[k] = 0.0;
            cnt[k] = 0;
            scnt[k] = 0;
        }
        if (tid == 0) {
            s_over = 0;
            s_in = 0;
        }
        __syncthreads();
    }
    const int j = blockIdx.x * WICK_BLOCK + tid;
    if (j < n2) {
        const double r2 = I.r[ob + j];
        const double w2 = I.w[ob + j], z2 = I.zev2[ob + j];
        int run = -1, first = 0;
        double sw = 0.0, sz = 0.0;
        uint32_t over = 0;
        auto close = [&](int end) {   // the segment [first, end) of bin `run`
            if (run < 0) return;
            if (PLACE) {
                const int pos = atomicAdd(&W.seg_pos[(int64_t)s * C.nb + run], 1);
                W.seg_raw[pos] = make_int4(run, j, first, end - 1);
            } else {
                atomicAdd(&cnt[run], end - first);
                atomicAdd(&scnt[run], 1);
                lds_add(hw + run, w2 * sw);
                lds_add(ht + run, w2 * z2 * sz);
            }
        };
        for (int i = 0; i < n1; ++i) {
            const int p = wick_bin(C, I.r[oa + i], r2, c, sn);
            if (p != run) {
                close(i);
                run = p;
                first = i;
                sw = sz = 0.0;
            }
            if (!PLACE) {
                over += p == -2 ? 1u : 0u;
                const double w1 = I.w[oa + i];
                sw += w1;
                sz += w1 * I.zev1[oa + i];
            }
        }
        close(n1);
        if (over) atomicAdd(&s_over, (unsigned long long)over);
    }
    if (PLACE) return;
    __syncthreads();
    unsigned long long in = 0;
    for (int k = tid; k < C.nb; k += WICK_BLOCK) {
        if (cnt[k] == 0) continue;
        in += cnt[k];
        unsafeAtomicAdd(O.weights_wick + k, hw[k]);
        atomicAdd(O.num_pairs_wick + k, (unsigned long long)cnt[k]);
        unsafeAtomicAdd(O.t1 + (int64_t)k * C.nb + k, ht[k]);
        atomicAdd(&W.seg_count[(int64_t)s * C.nb + k], scnt[k]);
    }
    if (in) atomicAdd(&s_in, in);
    __syncthreads();
    if (tid == 0) {
        if (s_over) atomicAdd(O.stats + WICK_STAT_OVERFLOW, s_over);
        atomicAdd(O.stats + WICK_STAT_IN_RANGE, s_in);
    }
}

namespace {

// v of the lane that DPP names, 0 for the lanes it does not write
template <int CTRL, int ROWS>
__device__ __forceinline__ double dpp_or_zero(double v) {
    const uint64_t b = (uint64_t)__double_as_longlong(v);
    const uint32_t lo = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)b, CTRL, ROWS, 0xf,
                                                              true);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)(b >> 32), CTRL,
                                                              ROWS, 0xf, true);
    return __longlong_as_double((long long)(((uint64_t)hi << 32) | lo));
}

// Inclusive prefix sum over the wave (row_shr 1, 2, 4, 8, then row_bcast 15 and 31); every lane
// is active.
__device__ __forceinline__ double wave_scan(double v) {
    v += dpp_or_zero<0x111, 0xf>(v);
    v += dpp_or_zero<0x112, 0xf>(v);
    v += dpp_or_zero<0x114, 0xf>(v);
    v += dpp_or_zero<0x118, 0xf>(v);
    v += dpp_or_zero<0x142, 0xa>(v);
    v += dpp_or_zero<0x143, 0xc>(v);
    return v;
}

// out[k + 1] = sum_{m <= k} value(m) for m in [0, n), out[0] = 0; one wave
template <class Value>
__device__ __forceinline__ void wave_prefix(int n, int lane, double *__restrict__ out,
                                            Value value) {
    if (lane == 0) out[0] = 0.0;
    double carry = 0.0;
    for (int k0 = 0; k0 < n; k0 += 256) {
        // four stretches of 64: their values are read together, then scanned
        double v[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int k = k0 + 64 * u + lane;
            v[u] = k < n ? value(k) : 0.0;
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int k = k0 + 64 * u + lane;
            v[u] = carry + wave_scan(v[u]);
            if (k < n) out[k + 1] = v[u];
            carry = __shfl(v[u], 63, 64);
        }
    }
}

}  // namespace

// Prefix sums of the diagonal of Wx and of w zev1 of each listed forest: one wave each.
__global__ __launch_bounds__(64) void wick_diag_kernel(WickInputs I,
                                                       const int32_t *__restrict__ forests,
                                                       double *__restrict__ diag,
                                                       double *__restrict__ wz) {
    const int f = forests[blockIdx.x];
    const int lane = threadIdx.x;
    const int64_t o = I.off[f];
    const int n = (int)(I.off[f + 1] - o);
    const double *m = I.wx + I.wx_off[f];
    wave_prefix(n, lane, diag + o + f, [&](int k) { return m[(int64_t)k * n + k]; });
    wave_prefix(n, lane, wz + o + f, [&](int k) { return I.w[o + k] * I.zev1[o + k]; });
}

// Segments of each task by rising j (and i), so that the lanes of the row kernel read
// neighbouring entries of a row: each finds its rank among the task's segments.  Longer lists
// than the stage holds keep the order in which their pixels came.
__global__ __launch_bounds__(WICK_BLOCK) void wick_sort_kernel(WickWork W) {
    __shared__ int64_t key[WICK_SORT];
    const WickTask t = W.task[blockIdx.x];
    const int4 *__restrict__ in = W.seg_raw + t.start;
    int4 *__restrict__ out = W.seg + t.start;
    if (t.count > WICK_SORT) {
        for (int k = threadIdx.x; k < t.count; k += WICK_BLOCK) out[k] = in[k];
        return;
    }
    for (int k = threadIdx.x; k < t.count; k += WICK_BLOCK)
        key[k] = ((int64_t)in[k].y << 32) | (uint32_t)in[k].z;
    __syncthreads();
    for (int k = threadIdx.x; k < t.count; k += WICK_BLOCK) {
        const int64_t mine = key[k];
        int rank = 0;
        for (int q = 0; q < t.count; ++q) rank += key[q] < mine ? 1 : 0;
        out[rank] = in[k];
    }
}

// The segments' sums: row r of a task's segment holds the prefix sums over i_b of
// sum_{i_a in segment} Wx1[i_a, i_b].  Waves take segments, lanes the pixels i_b.
__global__ __launch_bounds__(WICK_BLOCK) void wick_rsum_kernel(WickInputs I, WickPairs P,
                                                               WickWork W, int split) {
    const WickTask t = W.task[blockIdx.x / split];
    const int part = blockIdx.x % split;
    const int lane = threadIdx.x & 63;
    const int fa = P.a[t.pair];
    const int n1 = (int)(I.off[fa + 1] - I.off[fa]);
    const double *__restrict__ wx1 = I.wx + I.wx_off[fa];
    for (int k = part * (WICK_BLOCK / 64) + (threadIdx.x >> 6); k < t.count;
         k += split * (WICK_BLOCK / 64)) {
        const int4 e = W.seg[t.start + k];
        const int lo = uniform_int(e.z), hi = uniform_int(e.w);
        wave_prefix(n1, lane, W.rsum + t.rows + (int64_t)k * (n1 + 1), [&](int ib) {
            double v = 0.0;
            for (int ia = lo; ia <= hi; ++ia) v += wx1[(int64_t)ia * n1 + ib];
            return v;
        });
    }
}

// segment a of the task's bin as the row kernel stages it
struct WickA {
    int32_t lo, hi, ja, row;
    double w2z2;   // w2 zev2 at j_a
    double pad;
};
static_assert(sizeof(WickA) == 32, "WickA layout");
constexpr int WICK_ASTAGE = 256;   // segments a staged in LDS at a time

__global__ __launch_bounds__(WICK_BLOCK) void wick_row_kernel(WickConst C, WickInputs I,
                                                              WickPairs P, WickWork W,
                                                              WickOut O, int split) {
    extern __shared__ __align__(16) unsigned char smem[];
    double *r2 = (double *)smem;                  // [nb] row of T2
    double *r3 = r2 + C.nb;                       // [nb] row of T3
    WickA *sa = (WickA *)(r3 + C.nb);             // [WICK_ASTAGE] staged segments a
    __shared__ unsigned long long s_products;
    // workgroup g of `split` for task blockIdx / split takes part g of the pair's segments
    const int task = blockIdx.x / split;
    const int g = blockIdx.x - task * split;
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = tid >> 6;
    const WickTask t = W.task[task];
    const int part = (t.pair_count + split - 1) / split;
    const int lo = min(t.pair_count, g * part), hi = min(t.pair_count, lo + part);
    if (lo >= hi) return;   // uniform over the workgroup
    const int fa = P.a[t.pair], fb = P.b[t.pair];
    const int64_t oa = I.off[fa], ob = I.off[fb];
    const int n1 = (int)(I.off[fa + 1] - oa), n2 = (int)(I.off[fb + 1] - ob);
    const double *__restrict__ wx2 = I.wx + I.wx_off[fb];
    const double *__restrict__ rsum = W.rsum + t.rows;
    const double *__restrict__ diag = W.diag + oa + fa;
    const double *__restrict__ wz = W.wz + oa + fa;
    const int4 *__restrict__ segs = W.seg + t.pair_start;
    for (int k = tid; k < C.nb; k += WICK_BLOCK) {
        r2[k] = 0.0;
        r3[k] = 0.0;
    }
    if (tid == 0) s_products = 0;
    // Lanes own segments b; the wave walks the staged segments a in step, so every read of a
    // step is in one row: a's prefix sums and row j_a of the symmetric Wx2.
    uint64_t products = 0;
    for (int a0 = 0; a0 < t.count; a0 += WICK_ASTAGE) {
        const int na = min(WICK_ASTAGE, t.count - a0);
        __syncthreads();
        for (int k = tid; k < na; k += WICK_BLOCK) {
            const int4 e = W.seg[t.start + a0 + k];
            WickA A;
            A.lo = e.z;
            A.hi = e.w;
            A.ja = e.y;
            A.row = a0 + k;
            A.w2z2 = I.w[ob + e.y] * I.zev2[ob + e.y];
            A.pad = 0.0;
            sa[k] = A;
        }
        __syncthreads();
        for (int c0 = lo + wave * 64; c0 < hi; c0 += WICK_BLOCK) {
            const int sidx = c0 + lane;
            const bool live = sidx < hi;
            // (bin, j_b, i_lo, i_hi); a dead lane's empty segment reads entry 0 twice
            const int4 e = live ? segs[sidx] : make_int4(0, -1, 0, -1);
            const int len = e.w - e.z + 1;
            double acc2 = 0.0, acc3 = 0.0;
#pragma unroll 4
            for (int k = 0; k < na; ++k) {
                const WickA A = sa[k];
                const double *__restrict__ row = rsum + (int64_t)A.row * (n1 + 1);
                const bool same_j = e.y == A.ja;
                // Wx2[j_a, j_b], 0 for j_b == j_a (those products are T2) and dead lanes
                double x2 = 0.0;
                if (live && !same_j) x2 = wx2[(int64_t)A.ja * n2 + e.y];
                double d = row[e.w + 1] - row[e.z];
                products += (uint32_t)(A.hi - A.lo + 1) * (uint32_t)len;
                // pixels in both segments: i_b == i_a
                const int olo = max(A.lo, e.z), ohi = min(A.hi, e.w);
                double v = 0.0;
                if (olo <= ohi) {
                    d -= diag[ohi + 1] - diag[olo];
                    v = wz[ohi + 1] - wz[olo];
                    if (same_j) products -= (uint32_t)(ohi - olo + 1);
                }
                acc3 = fma(x2, d, acc3);
                // same j: Wx1[i_a, i_b] w2 zev2; i_b == i_a: Wx2[j_a, j_b] w1 zev1
                acc2 = fma(same_j ? A.w2z2 : x2, same_j ? d : v, acc2);
            }
            if (live) {
                if (acc2 != 0.0) lds_add(r2 + e.x, acc2);
                if (acc3 != 0.0) lds_add(r3 + e.x, acc3);
            }
        }
    }
    const uint64_t wp = wave_sum_u64(products);
    if (lane == 0) atomicAdd(&s_products, (unsigned long long)wp);
    __syncthreads();
    const int64_t row = (int64_t)t.bin * C.nb;
    for (int k = tid; k < C.nb; k += WICK_BLOCK) {
        if (r2[k] != 0.0) unsafeAtomicAdd(O.t2 + row + k, r2[k]);
        if (r3[k] != 0.0) unsafeAtomicAdd(O.t3 + row + k, r3[k]);
    }
    if (tid == 0) atomicAdd(O.stats + WICK_STAT_PRODUCTS, s_products);
}

size_t wick_list_lds(const WickConst &C) { return (size_t)C.nb * (8 + 8 + 4 + 4); }
size_t wick_row_lds(const WickConst &C) {
    return (size_t)C.nb * 16 + (size_t)WICK_ASTAGE * sizeof(WickA);
}

hipError_t launch_wick_diag(const WickInputs &I, const int32_t *forests, int32_t num_forests,
                            double *diag, double *wz, hipStream_t stream) {
    if (num_forests <= 0) return hipSuccess;
    hipLaunchKernelGGL(wick_diag_kernel, dim3(num_forests), dim3(64), 0, stream, I, forests, diag,
                       wz);
    return hipGetLastError();
}

hipError_t launch_wick_segments(bool place, const WickConst &C, const WickInputs &I,
                                const WickPairs &P, const WickWork &W, const WickOut &O,
                                int64_t longest, hipStream_t stream) {
    if (P.count <= 0 || longest <= 0) return hipSuccess;
    const dim3 grid((unsigned)((longest + WICK_BLOCK - 1) / WICK_BLOCK), (unsigned)P.count);
    if (place) {
        hipLaunchKernelGGL(wick_segment_kernel<true>, grid, dim3(WICK_BLOCK), 0, stream, C, I, P,
                           W, O);
        return hipGetLastError();
    }
    const size_t lds = wick_list_lds(C);
    hipError_t err = hipFuncSetAttribute((const void *)wick_segment_kernel<false>,
                                         hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (err != hipSuccess) return err;
    hipLaunchKernelGGL(wick_segment_kernel<false>, grid, dim3(WICK_BLOCK), lds, stream, C, I, P,
                       W, O);
    return hipGetLastError();
}

hipError_t launch_wick_sort(const WickWork &W, int64_t tasks, hipStream_t stream) {
    if (tasks <= 0) return hipSuccess;
    hipLaunchKernelGGL(wick_sort_kernel, dim3((unsigned)tasks), dim3(WICK_BLOCK), 0, stream, W);
    return hipGetLastError();
}

hipError_t launch_wick_rows(const WickConst &C, const WickInputs &I, const WickPairs &P,
                            const WickWork &W, const WickOut &O, int64_t tasks,
                            hipStream_t stream) {
    if (tasks <= 0) return hipSuccess;
    const size_t lds = wick_row_lds(C);
    hipError_t err = hipFuncSetAttribute((const void *)wick_row_kernel,
                                         hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (err != hipSuccess) return err;
    // enough workgroups for about eight waves per SIMD: each task's list split in parts
    const int64_t want = 8 * 1024 / (WICK_BLOCK / 64);
    const int split = (int)std::max<int64_t>(1, std::min<int64_t>(64, (want + tasks - 1) / tasks));
    hipLaunchKernelGGL(wick_rsum_kernel, dim3((unsigned)(tasks * 2 * split)), dim3(WICK_BLOCK), 0,
                       stream, I, P, W, 2 * split);
    hipLaunchKernelGGL(wick_row_kernel, dim3((unsigned)(tasks * split)), dim3(WICK_BLOCK), lds,
                       stream, C, I, P, W, O, split);
    return hipGetLastError();
}

}  // namespace picca
