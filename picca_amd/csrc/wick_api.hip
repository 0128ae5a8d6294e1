// C-ABI of the Wick covariance terms (declared in include/picca_hip.h).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <string>
#include <vector>

#include "context.h"

extern "C" {

int picca_wick_t123(picca_ctx *ctx, const picca_cf_params *params, int64_t num_pairs,
                    const int32_t *pair_a, const int32_t *pair_b, const double *pair_ang,
                    const double *zev1, const double *zev2, const int64_t *wx_offsets,
                    int64_t wx_size, const double *wx, double *weights_wick,
                    int64_t *num_pairs_wick, double *t1, double *t2, double *t3,
                    picca_wick_report *report) {
    if (!ctx) return fail(PICCA_E_VALUE, "ctx is NULL");
    if (!params) return fail(PICCA_E_VALUE, "params is NULL");
    if (ctx->num_forests <= 0) return fail(PICCA_E_RUNTIME, "no forest store");
    const int np = params->num_bins_r_par, nt = params->num_bins_r_trans;
    if (np <= 0 || nt <= 0) return fail(PICCA_E_VALUE, "bin counts must be positive");
    if ((int64_t)np * nt > 8192) return fail(PICCA_E_VALUE, "more than 8192 bins");
    if (!(params->r_par_max > params->r_par_min) || !(params->r_trans_max > 0))
        return fail(PICCA_E_VALUE, "empty separation range");
    if (num_pairs < 0 || wx_size < 0) return fail(PICCA_E_VALUE, "negative size");
    const int64_t nf = ctx->num_forests, npix = ctx->num_pixels;
    if (!zev1 || !zev2 || !wx_offsets || (wx_size > 0 && !wx))
        return fail(PICCA_E_VALUE, "input arrays must not be NULL");
    if (num_pairs > 0 && (!pair_a || !pair_b || !pair_ang))
        return fail(PICCA_E_VALUE, "pair arrays must not be NULL");
    if (!weights_wick || !num_pairs_wick || !t1 || !t2 || !t3)
        return fail(PICCA_E_VALUE, "output arrays must not be NULL");
    const std::vector<int64_t> &off = ctx->h_offsets;
    for (int64_t k = 0; k < num_pairs; ++k) {
        if (pair_a[k] < 0 || pair_a[k] >= nf || pair_b[k] < 0 || pair_b[k] >= nf)
            return fail(PICCA_E_VALUE, "pair index out of range of the forest store");
        if (!(pair_ang[k] >= 0.0) || !(pair_ang[k] <= M_PI))
            return fail(PICCA_E_VALUE, "pair angle outside [0, pi]");
        for (int32_t f : {pair_a[k], pair_b[k]}) {
            const int64_t n = off[f + 1] - off[f];
            if (n >= (1 << 20)) return fail(PICCA_E_VALUE, "forest longer than 2^20 pixels");
            if (wx_offsets[f] < 0 || wx_offsets[f] + n * n > wx_size)
                return fail(PICCA_E_VALUE, "weighted 1-D correlation missing for a forest");
        }
    }
    for (int64_t k = 0; k < npix; ++k)
        if (!std::isfinite(zev1[k]) || !std::isfinite(zev2[k]))
            return fail(PICCA_E_VALUE, "evolution factors must be finite");

    picca::WickConst C;
    std::memset(&C, 0, sizeof(C));
    C.np = np;
    C.nt = nt;
    C.nb = np * nt;
    C.xcorr = params->x_correlation != 0;
    C.rpmin = params->r_par_min;
    C.rpmax = params->r_par_max;
    C.rtmax = params->r_trans_max;
    C.span = params->r_par_max - params->r_par_min;
    const int64_t nb = C.nb;
    if ((int64_t)(picca::wick_row_lds(C) + 1024) > ctx->lds_limit ||
        (int64_t)(picca::wick_list_lds(C) + 2048) > ctx->lds_limit)
        return fail(PICCA_E_VALUE, "too many bins for the workgroup's LDS");

    PICCA_HIP_CHECK(hipSetDevice(ctx->device));
    PICCA_HIP_CHECK(ctx->wk_zev1.upload(zev1, (size_t)npix, ctx->stream));
    PICCA_HIP_CHECK(ctx->wk_zev2.upload(zev2, (size_t)npix, ctx->stream));
    PICCA_HIP_CHECK(ctx->wk_wx.upload(wx, (size_t)wx_size, ctx->stream));
    PICCA_HIP_CHECK(ctx->wk_wxoff.upload(wx_offsets, (size_t)nf, ctx->stream));
    PICCA_HIP_CHECK(ctx->o_wdm.reserve((size_t)nb));
    PICCA_HIP_CHECK(ctx->wk_nb.reserve((size_t)nb));
    PICCA_HIP_CHECK(ctx->o_dmat.reserve((size_t)(3 * nb * nb)));
    PICCA_HIP_CHECK(ctx->wk_stats.reserve(picca::WICK_NSTATS));
    PICCA_HIP_CHECK(picca::launch_zero_u64((unsigned long long *)ctx->o_wdm.ptr, nb, ctx->stream));
    PICCA_HIP_CHECK(picca::launch_zero_u64(ctx->wk_nb.ptr, nb, ctx->stream));
    PICCA_HIP_CHECK(picca::launch_zero_u64((unsigned long long *)ctx->o_dmat.ptr, 3 * nb * nb,
                                           ctx->stream));
    PICCA_HIP_CHECK(picca::launch_zero_u64(ctx->wk_stats.ptr, picca::WICK_NSTATS, ctx->stream));
    // prefix sums of the diagonal and of w zev1 for every forest of the pairs
    std::vector<int32_t> forests;
    {
        std::vector<char> used((size_t)nf, 0);
        for (int64_t k = 0; k < num_pairs; ++k) used[(size_t)pair_a[k]] = used[(size_t)pair_b[k]] = 1;
        for (int64_t f = 0; f < nf; ++f)
            if (used[(size_t)f]) forests.push_back((int32_t)f);
    }
    PICCA_HIP_CHECK(ctx->wk_forests.upload(forests.data(), forests.size(), ctx->stream));
    PICCA_HIP_CHECK(ctx->wk_diag.reserve((size_t)(npix + nf)));
    PICCA_HIP_CHECK(ctx->wk_wz.reserve((size_t)(npix + nf)));
    picca::WickInputs I{ctx->off.ptr,     ctx->r.ptr,       ctx->w.ptr,       ctx->wk_zev1.ptr,
                        ctx->wk_zev2.ptr, ctx->wk_wx.ptr,   ctx->wk_wxoff.ptr};
    PICCA_HIP_CHECK(picca::launch_wick_diag(I, ctx->wk_forests.ptr, (int32_t)forests.size(),
                                            ctx->wk_diag.ptr, ctx->wk_wz.ptr, ctx->stream));
    picca::WickOut O{ctx->o_wdm.ptr, ctx->wk_nb.ptr, ctx->o_dmat.ptr, ctx->o_dmat.ptr + nb * nb,
                     ctx->o_dmat.ptr + 2 * nb * nb, ctx->wk_stats.ptr};

    // batches of pairs: at most 2^20 (pair, bin) counts and 2^27 pixel pairs (the segments are
    // fewer); inside a batch, runs of tasks, or of parts of them, whose segment sums fit 1 GiB
    const int64_t pixel_budget = (int64_t)1 << 27, count_budget = (int64_t)1 << 20;
    const int64_t rsum_budget = (int64_t)1 << 27;
    double total_ms = 0.0;
    int64_t batches = 0;
    std::vector<double> cs;
    std::vector<int32_t> seg_count, seg_pos;
    std::vector<picca::WickTask> tasks, rows_of;
    auto add_time = [&]() -> int {
        PICCA_HIP_CHECK(hipEventRecord(ctx->ev_stop, ctx->stream));
        PICCA_HIP_CHECK(hipStreamSynchronize(ctx->stream));
        float ms = 0.f;
        PICCA_HIP_CHECK(hipEventElapsedTime(&ms, ctx->ev_start, ctx->ev_stop));
        total_ms += ms;
        return PICCA_OK;
    };
    for (int64_t p0 = 0; p0 < num_pairs;) {
        int64_t p1 = p0, entries = 0, longest = 0;
        while (p1 < num_pairs && (p1 == p0 || (p1 - p0 + 1) * nb <= count_budget) &&
               p1 - p0 < 65535) {
            const int64_t n1 = off[pair_a[p1] + 1] - off[pair_a[p1]];
            const int64_t n2 = off[pair_b[p1] + 1] - off[pair_b[p1]];
            if (p1 > p0 && entries + n1 * n2 > pixel_budget) break;
            entries += n1 * n2;
            longest = std::max(longest, n2);
            ++p1;
        }
        const int64_t count = p1 - p0;
        cs.assign((size_t)(2 * count), 0.0);
        for (int64_t k = 0; k < count; ++k) {
            cs[2 * k] = std::cos(pair_ang[p0 + k] / 2);
            cs[2 * k + 1] = std::sin(pair_ang[p0 + k] / 2);
        }
        PICCA_HIP_CHECK(ctx->dpa.upload(pair_a + p0, (size_t)count, ctx->stream));
        PICCA_HIP_CHECK(ctx->dpb.upload(pair_b + p0, (size_t)count, ctx->stream));
        PICCA_HIP_CHECK(ctx->dcs.upload(cs.data(), cs.size(), ctx->stream));
        // (zeroed in 64-bit words)
        const int64_t cells = count * nb;
        PICCA_HIP_CHECK(ctx->wk_segcount.reserve((size_t)cells + 1));
        PICCA_HIP_CHECK(picca::launch_zero_u64((unsigned long long *)ctx->wk_segcount.ptr,
                                               (cells + 1) / 2, ctx->stream));
        picca::WickPairs P{ctx->dpa.ptr, ctx->dpb.ptr, ctx->dcs.ptr, (int32_t)count};
        picca::WickWork W{ctx->wk_segcount.ptr, nullptr, nullptr, nullptr, nullptr, nullptr,
                          ctx->wk_diag.ptr, ctx->wk_wz.ptr};
        PICCA_HIP_CHECK(hipEventRecord(ctx->ev_start, ctx->stream));
        PICCA_HIP_CHECK(picca::launch_wick_segments(false, C, I, P, W, O, longest, ctx->stream));
        int status = add_time();
        if (status != PICCA_OK) return status;
        seg_count.resize((size_t)cells);
        PICCA_HIP_CHECK(hipMemcpyAsync(seg_count.data(), ctx->wk_segcount.ptr,
                                       sizeof(int32_t) * (size_t)cells, hipMemcpyDeviceToHost,
                                       ctx->stream));
        PICCA_HIP_CHECK(hipStreamSynchronize(ctx->stream));
        // tasks in (pair, bin) order and the segments' positions
        seg_pos.resize((size_t)cells);
        tasks.clear();
        int64_t segs = 0;
        for (int64_t k = 0; k < count; ++k) {
            const int64_t start = segs;
            const size_t first_task = tasks.size();
            for (int64_t p = 0; p < nb; ++p) {
                const int32_t n = seg_count[(size_t)(k * nb + p)];
                if (n < 0 || segs + n > INT32_MAX)   // a forest pair whose pixels hardly rise
                    return fail(PICCA_E_VALUE, "more than 2^31 segments in one pair");
                seg_pos[(size_t)(k * nb + p)] = (int32_t)segs;
                if (n > 0)
                    tasks.push_back(picca::WickTask{(int32_t)k, (int32_t)p, (int32_t)segs, n,
                                                    (int32_t)start, 0, 0});
                segs += n;
            }
            for (size_t t = first_task; t < tasks.size(); ++t)
                tasks[t].pair_count = (int32_t)(segs - start);
        }
        ++batches;
        if (!tasks.empty()) {
            // The row kernel's tasks: a (pair, bin) each, in parts where its segment sums exceed
            // the budget, and runs of them whose sums fit it, from row 0 in each run.
            rows_of.clear();
            std::vector<int64_t> run_begin{0};
            int64_t rows = 0, most = 0;
            for (const picca::WickTask &task : tasks) {
                const int32_t f = pair_a[p0 + task.pair];
                const int64_t row = off[f + 1] - off[f] + 1;
                const int32_t part = (int32_t)std::min<int64_t>(
                    task.count, std::max<int64_t>(1, rsum_budget / row));
                for (int32_t first = 0; first < task.count; first += part) {
                    picca::WickTask t = task;
                    t.start += first;
                    t.count = std::min(part, task.count - first);
                    if (rows > 0 && rows + t.count * row > rsum_budget) {
                        run_begin.push_back((int64_t)rows_of.size());
                        rows = 0;
                    }
                    t.rows = rows;
                    rows += t.count * row;
                    most = std::max(most, rows);
                    rows_of.push_back(t);
                }
            }
            run_begin.push_back((int64_t)rows_of.size());
            PICCA_HIP_CHECK(ctx->wk_segpos.upload(seg_pos.data(), (size_t)cells, ctx->stream));
            PICCA_HIP_CHECK(ctx->wk_task.upload(tasks.data(), tasks.size(), ctx->stream));
            PICCA_HIP_CHECK(ctx->wk_rows.upload(rows_of.data(), rows_of.size(), ctx->stream));
            PICCA_HIP_CHECK(ctx->wk_seg_raw.reserve((size_t)segs));
            PICCA_HIP_CHECK(ctx->wk_seg.reserve((size_t)segs));
            PICCA_HIP_CHECK(ctx->wk_rsum.reserve((size_t)most));
            W.seg_pos = ctx->wk_segpos.ptr;
            W.seg_raw = ctx->wk_seg_raw.ptr;
            W.seg = ctx->wk_seg.ptr;
            W.rsum = ctx->wk_rsum.ptr;
            PICCA_HIP_CHECK(hipEventRecord(ctx->ev_start, ctx->stream));
            PICCA_HIP_CHECK(picca::launch_wick_segments(true, C, I, P, W, O, longest,
                                                        ctx->stream));
            W.task = ctx->wk_task.ptr;
            PICCA_HIP_CHECK(picca::launch_wick_sort(W, (int64_t)tasks.size(), ctx->stream));
            for (size_t r = 0; r + 1 < run_begin.size(); ++r) {
                W.task = ctx->wk_rows.ptr + run_begin[r];
                PICCA_HIP_CHECK(picca::launch_wick_rows(C, I, P, W, O,
                                                        run_begin[r + 1] - run_begin[r],
                                                        ctx->stream));
            }
            status = add_time();
            if (status != PICCA_OK) return status;
        }
        p0 = p1;
    }

    std::vector<double> h_w((size_t)nb), h_t((size_t)(3 * nb * nb));
    std::vector<unsigned long long> h_n((size_t)nb);
    unsigned long long h_stats[picca::WICK_NSTATS];
    PICCA_HIP_CHECK(hipMemcpyAsync(h_w.data(), ctx->o_wdm.ptr, sizeof(double) * nb,
                                   hipMemcpyDeviceToHost, ctx->stream));
    PICCA_HIP_CHECK(hipMemcpyAsync(h_n.data(), ctx->wk_nb.ptr, sizeof(unsigned long long) * nb,
                                   hipMemcpyDeviceToHost, ctx->stream));
    PICCA_HIP_CHECK(hipMemcpyAsync(h_t.data(), ctx->o_dmat.ptr, sizeof(double) * 3 * nb * nb,
                                   hipMemcpyDeviceToHost, ctx->stream));
    PICCA_HIP_CHECK(hipMemcpyAsync(h_stats, ctx->wk_stats.ptr, sizeof(h_stats),
                                   hipMemcpyDeviceToHost, ctx->stream));
    PICCA_HIP_CHECK(hipStreamSynchronize(ctx->stream));
    for (int64_t k = 0; k < nb; ++k) {
        weights_wick[k] += h_w[k];
        num_pairs_wick[k] += (int64_t)h_n[k];
    }
    for (int64_t k = 0; k < nb * nb; ++k) {
        t1[k] += h_t[k];
        t2[k] += h_t[nb * nb + k];
        t3[k] += h_t[2 * nb * nb + k];
    }
    if (report) {
        report->in_range_pairs = (int64_t)h_stats[picca::WICK_STAT_IN_RANGE];
        // the row kernel walks every listed pair a against every b != a, so it sees each
        // unordered pair {a, b} twice; the reference's loop (py/picca/cf.py:1573-1600)
        // visits index1 < index2 only, one product per unordered pair
        report->products = (int64_t)(h_stats[picca::WICK_STAT_PRODUCTS] / 2);
        report->overflow_pairs = (int64_t)h_stats[picca::WICK_STAT_OVERFLOW];
        report->batches = batches;
        report->kernel_ms = total_ms;
    }
    return PICCA_OK;
}

}  // extern "C"
