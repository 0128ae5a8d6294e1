// Device context of the C-ABI (shared by the entry points of the library).
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cstring>
#include <string>
#include <thread>
#include <memory>
#include <vector>

#include "../../include/picca_hip.h"
#include "engine.h"
#include "download.h"
#include "dmat_band.h"
#include "xi_walk.h"

namespace picca_host {

// message of the last failure on the calling thread (picca_last_error)
std::string &last_error();

inline int fail(int code, const std::string &msg) {
    last_error() = msg;
    return code;
}

#define PICCA_HIP_CHECK(expr)                                                              \
    do {                                                                                   \
        hipError_t err_ = (expr);                                                          \
        if (err_ != hipSuccess)                                                            \
            return picca_host::fail(PICCA_E_HIP,                                           \
                                    std::string(#expr) + ": " + hipGetErrorString(err_));  \
    } while (0)

template <typename T>
struct DeviceBuffer {
    T *ptr = nullptr;
    size_t count = 0;
    DeviceBuffer() = default;
    DeviceBuffer(const DeviceBuffer &) = delete;
    DeviceBuffer &operator=(const DeviceBuffer &) = delete;
    ~DeviceBuffer() { release(); }
    void release() {
        if (ptr) (void)hipFree(ptr);
        ptr = nullptr;
        count = 0;
    }
    hipError_t reserve(size_t n) {
        if (n <= count && ptr) return hipSuccess;
        release();
        size_t bytes = std::max<size_t>(n, 1) * sizeof(T);
        hipError_t err = hipMalloc((void **)&ptr, bytes);
        if (err != hipSuccess) {
            ptr = nullptr;
            return err;
        }
        count = n;
        return hipSuccess;
    }
    hipError_t upload(const T *host, size_t n, hipStream_t stream) {
        hipError_t err = reserve(n);
        if (err != hipSuccess || n == 0) return err;
        return hipMemcpyAsync(ptr, host, n * sizeof(T), hipMemcpyHostToDevice, stream);
    }
    // n values followed by `pad` zeros (kernels may read a few elements past the end)
    hipError_t upload_padded(const T *host, size_t n, size_t pad, hipStream_t stream) {
        hipError_t err = reserve(n + pad);
        if (err != hipSuccess) return err;
        if (n > 0) err = hipMemcpyAsync(ptr, host, n * sizeof(T), hipMemcpyHostToDevice, stream);
        if (err != hipSuccess) return err;
        return hipMemsetAsync(ptr + n, 0, pad * sizeof(T), stream);
    }
};

// Runs body(begin, end) over [0, n) on up to hardware_concurrency threads, on the calling one
// alone below 65536 elements of work (`work`: of n items that are several each, as forests; a
// started thread takes as long as a few thousand forest pixels, so those count half).
template <typename F>
inline void parallel_for(int64_t n, F body, int64_t work = 0) {
    unsigned hw = std::thread::hardware_concurrency();
    int64_t nthreads = std::max<int64_t>(1, std::min<int64_t>(hw ? hw : 1, 16));
    if (std::max(n, work) < 65536) nthreads = 1;
    if (nthreads == 1) {
        body(0, n);
        return;
    }
    std::vector<std::thread> pool;
    int64_t step = (n + nthreads - 1) / nthreads;
    for (int64_t t = 0; t < nthreads; ++t) {
        int64_t lo = t * step, hi = std::min(n, lo + step);
        if (lo >= hi) break;
        pool.emplace_back([=] { body(lo, hi); });
    }
    for (auto &th : pool) th.join();
}

// All of [0, n) pass ok(k), a test of a few instructions: on several threads from 2^20 on (on
// 3e5 values starting them took longer than the tests, 0.13 ms of a covariance).
template <typename F>
inline bool parallel_all(int64_t n, F ok) {
    std::atomic<bool> all{true};
    auto range = [&](int64_t lo, int64_t hi) {
        bool good = true;
        for (int64_t k = lo; k < hi; ++k) good = good && ok(k);
        if (!good) all.store(false, std::memory_order_relaxed);
    };
    if (n < ((int64_t)1 << 20)) range(0, n);
    else parallel_for(n, range);
    return all.load();
}

}  // namespace picca_host

using picca_host::DeviceBuffer;
using picca_host::download_values;
using picca_host::fail;
using picca_host::parallel_all;
using picca_host::parallel_for;

struct picca_ctx {
    int device = 0;
    hipStream_t stream = nullptr;
    hipEvent_t ev_start = nullptr, ev_stop = nullptr, ev_mid = nullptr;
    picca_host::DownloadRing ring;
    // distortion matrix: events around each batch's pass and fill kernels (a pool that
    // grows with the batches of a run) and the last run's report
    std::vector<hipEvent_t> dmat_events;
    picca_dmat_report dmat_report = {0.0, 0.0, 0, 0};
    int num_cus = 0;
    int64_t lds_limit = 0;
    unsigned long long *scratch = nullptr;   // this GPU's no-allocation scratch array

    // forest store
    int64_t num_forests = 0;
    int64_t num_pixels = 0;
    double max_abs_r = 0;   // largest |r_comov| and |dist_m| of the store: bound the
    double max_abs_d = 0;   // rounding of the pre-scaled coordinates of the fast loop
    bool negative_d = false;   // some dist_m is negative
    bool has_log_lambda = false;
    bool has_order = false;
    std::vector<int32_t> h_order;   // host copy of the fit orders (< 0: unprojected)
    std::vector<int64_t> h_offsets;
    std::vector<double> h_dmin, h_dmax;   // per forest: smallest / largest dist_m
    std::vector<double2> h_spc;           // per forest: smallest steps (ForestView::spc)
    std::vector<uint8_t> h_mono;          // per forest: ForestView::mono
    std::vector<uint8_t> h_fit;           // per forest: sum w and sum w dll^2 are positive
    DeviceBuffer<double> z, r, d, w, dw, ll, zq;
    DeviceBuffer<picca::PixelRecord> pix;
    DeviceBuffer<int64_t> off;
    DeviceBuffer<int32_t> order;
    DeviceBuffer<uint8_t> mono;
    // run walk of the xi kernel (xi_walk.h)
    DeviceBuffer<double2> rd, spc;
    DeviceBuffer<picca::PrefixPair> pre;
    int32_t xi_schedule = 0;   // PICCA_XI_SCHEDULE_*
    double median_step_r = 0;  // median over forests of the mean r_comov step between pixels
    // the xi launch sequence (zero kernels + pair kernel) as a HIP graph, replayed while
    // its launch arguments stay the same
    bool xi_use_graph = true;
    hipGraph_t xi_graph = nullptr;
    hipGraphExec_t xi_graph_exec = nullptr;
    std::vector<unsigned char> xi_graph_key;

    // xi pairs
    int64_t num_pairs = 0;
    int32_t num_rows = 0;
    DeviceBuffer<int32_t> pa, pb, pchunks;
    DeviceBuffer<double> pang, pcs;
    DeviceBuffer<uint8_t> pflags;
    std::vector<int64_t> h_group_begin;
    std::vector<int32_t> h_group_row;
    DeviceBuffer<int64_t> gbegin;
    DeviceBuffer<int32_t> grow;

    // distortion-matrix inputs (stores given with log_lambda): per-forest sums of
    // compute_dmat_forest_pairs_fast (py/picca/cf.py:577-594) and the pixel redshifts
    std::vector<double> h_z;
    DeviceBuffer<double> dll, sum_w, sw_dll, zfa, zfb;

    // dmat batches
    DeviceBuffer<int32_t> dpa, dpb;
    DeviceBuffer<double> dang, dcs;
    DeviceBuffer<uint8_t> dflags;
    DeviceBuffer<double> ws_S, ws_eta;
    DeviceBuffer<uint32_t> ws_U;
    DeviceBuffer<int32_t> ws_band, ws_rng, ws_cnt;
    DeviceBuffer<int64_t> ws_pix;
    DeviceBuffer<unsigned long long> ws_touched;
    DeviceBuffer<double> o_wdm, o_dmat;
    DeviceBuffer<double> o_matrix;   // MatrixBlock of a distortion matrix
    // forest pairs without cuts: prefix sums of both roles (64 bytes a pixel of the call's
    // forests and role, 8 of index tables) and the workspace of a batch
    int64_t dmat_batch_bytes = PICCA_DMAT_BATCH_BYTES, dmat_prefix_bytes = INT64_MAX;
    int64_t dmat_routes[PICCA_DMAT_ROUTES] = {0, 0, 0, 0};
    DeviceBuffer<picca::DmatPrefix> db_pre_a, db_pre_b;
    DeviceBuffer<picca::DmatBandSlot> db_slot;
    DeviceBuffer<double> db_cs, db_S, db_eta, db_eff;
    DeviceBuffer<int4> db_rng_t, db_rng_u, db_items;
    DeviceBuffer<int32_t> db_tile, db_list, db_redo, db_num, db_table_r, db_table_d;
    DeviceBuffer<picca::DmatListedForest> db_listed;
    void release_dmat_band() {
        db_pre_a.release();
        db_pre_b.release();
        db_table_r.release();
        db_table_d.release();
        db_S.release();
        db_eta.release();
        db_eff.release();
        db_list.release();
        db_items.release();
    }

    // metal distortion matrix: absorber tables per slot (store order) and per-pass tasks
    struct MetalSlot {
        bool set = false;
        int64_t pixels = 0;
        DeviceBuffer<double> z, r, d, w, f;
        DeviceBuffer<picca::MetalRecord> rec;   // num_pixels + METAL_REC_PAD records
    };
    MetalSlot metal[4];
    DeviceBuffer<int64_t> m_task_begin;
    DeviceBuffer<int32_t> m_task_pair;

    // subsampling covariance: rows, weights, per-bin means and weight sums, matrix
    DeviceBuffer<double> cv_xi, cv_w, cv_y, cv_s, cv_cov;

    // Wick terms: evolution factors, weighted 1-D correlations, per-batch segments and tasks
    DeviceBuffer<double> wk_zev1, wk_zev2, wk_wx, wk_rsum, wk_diag, wk_wz;
    DeviceBuffer<int64_t> wk_wxoff;
    DeviceBuffer<int32_t> wk_segcount, wk_segpos, wk_forests;
    DeviceBuffer<int4> wk_seg, wk_seg_raw;
    DeviceBuffer<picca::WickTask> wk_task, wk_rows;   // (pair, bin); the row kernel's parts
    DeviceBuffer<unsigned long long> wk_nb, wk_stats;

    // continuum fit: resident spectra (forest pixels) and per-forest results
    int64_t cont_forests = 0;
    int64_t cont_pixels = 0;
    DeviceBuffer<int64_t> c_off;
    DeviceBuffer<int32_t> c_class;   // forests ordered by the waves their fit takes
    int64_t cont_class_begin[picca::CONT_CLASSES + 1] = {0, 0, 0, 0, 0, 0};
    DeviceBuffer<double> c_flux, c_ivar, c_mean, c_x, c_eta, c_lss, c_fudge;
    DeviceBuffer<int32_t> c_order;
    DeviceBuffer<double> c_a0, c_b0;
    // the fit's a, b, chi2, then ndata, status, evaluations, one array after the other
    DeviceBuffer<double> c_fit;
    picca::ContOut cont_out() const {
        const size_t n = (size_t)cont_forests;
        int32_t *whole = (int32_t *)(c_fit.ptr + 3 * n);
        return {c_fit.ptr, c_fit.ptr + n, c_fit.ptr + 2 * n, whole, whole + n, whole + 2 * n};
    }
    // DR16 iteration: per pixel rest-frame log lambda, transmission correction, rest-frame
    // bin; the stacked sums; the mean continuum's interpolation nodes
    DeviceBuffer<double> c_llr, c_trans, c_stack, c_xs, c_ys;
    DeviceBuffer<int32_t> c_bin;
    int32_t cont_nbins = 0;     // 0: no rest frame set for the resident forests
    bool cont_fitted = false;   // a fit of the resident forests is on the device

    // seed network: parameters, Adam state, training data and scratch
    int32_t mlp_in = 0, mlp_hidden = 0;
    int64_t mlp_step = 0;   // Adam time step
    DeviceBuffer<float> m_w1t, m_b1, m_w2, m_b2;
    DeviceBuffer<uint16_t> m_w1t_bf16;
    DeviceBuffer<float> g_w1t, g_b1, g_w2, g_b2, g_loss;
    DeviceBuffer<float> a_m, a_v;
    DeviceBuffer<float> m_x, m_t, m_h, m_y, m_dh;
    DeviceBuffer<int32_t> m_rows;
    int64_t mlp_rows = 0;   // rows of the resident training data

    // forest x quasar pairs (cross-correlation)
    int64_t xcf_pairs = 0;
    int32_t xcf_rows = 0;
    DeviceBuffer<picca::XcfPairRecord> x_rec;
    DeviceBuffer<int32_t> x_forest, x_row;
    DeviceBuffer<int64_t> x_begin, x_chunk;
    int64_t xcf_groups = 0, xcf_chunks = 0;
    // host copies of the groups and, per pair in record order, the smallest and largest
    // r_trans any pixel of its forest can have with the quasar (for the row windows)
    std::vector<int64_t> hx_begin;
    std::vector<int32_t> hx_forest, hx_row;
    std::vector<double> hx_rt_lo, hx_rt_hi;
    // row windows of the last plan: per window, the pair indices and groups on the device
    struct XcfWindow {
        int32_t t0 = 0, rows = 0;
        int64_t groups = 0;
        int64_t chunks = 0;
        DeviceBuffer<int64_t> idx, begin, chunk;
        DeviceBuffer<int32_t> forest, row;
    };
    std::vector<std::unique_ptr<XcfWindow>> x_windows;
    int64_t x_plan_version = -1;
    int32_t x_plan_nt = 0, x_plan_rows = 0;
    double x_plan_rtmax = 0;
    int64_t x_pairs_version = 0;

    // xi results
    int64_t out_nb = 0;
    int32_t out_rows = 0;
    bool have_result = false;
    DeviceBuffer<picca::XiBin> o_bins;
    DeviceBuffer<unsigned long long> queue, stats;
};

// A distortion matrix's results on the device, in one block that one copy fetches: counters, then
// weights_dmat, the four effective sums and the matrix.
constexpr int MATRIX_COUNTERS = 16;
struct MatrixBlock {
    unsigned long long *counters;
    double *weights, *eff, *matrix;
    int64_t nb, nm;
    int64_t words() const { return MATRIX_COUNTERS + nb + 4 * nm + nb * nm; }
};

// The block in the context, cleared by the stream.
inline hipError_t make_matrix_block(picca_ctx *ctx, int64_t nb, int64_t nm, MatrixBlock &B) {
    B = MatrixBlock{nullptr, nullptr, nullptr, nullptr, nb, nm};
    const hipError_t err = ctx->o_matrix.reserve((size_t)B.words());
    if (err != hipSuccess) return err;
    B.counters = (unsigned long long *)ctx->o_matrix.ptr;
    B.weights = ctx->o_matrix.ptr + MATRIX_COUNTERS;
    B.eff = B.weights + nb;
    B.matrix = B.eff + 4 * nm;
    return picca::launch_zero_u64(B.counters, B.words(), ctx->stream);
}

// Fetches the counters when the stream is done and, if accept(counters), adds the results to the
// caller's arrays.  A matrix of up to 1 MB is copied with its counters.
template <class Accept>
inline hipError_t fetch_matrix(picca_ctx *ctx, const MatrixBlock &B, const Accept &accept,
                               double *weights_dmat, double *dmat, double *r_par_eff,
                               double *r_trans_eff, double *z_eff, double *weight_eff) {
    constexpr int64_t HEAD = 8 * MATRIX_COUNTERS;
    struct Field {
        double *to;
        int64_t size;
    };
    const Field fields[6] = {{weights_dmat, 8 * B.nb}, {r_par_eff, 8 * B.nm},
                             {r_trans_eff, 8 * B.nm},  {z_eff, 8 * B.nm},
                             {weight_eff, 8 * B.nm},   {dmat, 8 * B.nb * B.nm}};
    // bytes [lo, hi) of the results (behind the counters), whose first is at src
    auto add = [&](const char *src, int64_t lo, int64_t hi) {
        int64_t first = 0;
        for (const Field &f : fields) {
            const int64_t p = std::max(lo, first), q = std::min(hi, first + f.size);
            const double *s = (const double *)(src + (p - lo));
            double *o = f.to + (p - first) / 8;
            for (int64_t k = 0; k < (q - p) / 8; ++k) o[k] += s[k];
            first += f.size;
        }
    };
    const int64_t bytes = 8 * B.words();
    const bool whole = bytes <= picca_host::DownloadRing::SMALL;
    hipError_t err = ctx->ring.ensure(bytes);
    if (err == hipSuccess) err = ctx->ring.fetch(B.counters, whole ? bytes : HEAD, ctx->stream);
    if (err != hipSuccess) return err;
    unsigned long long counters[MATRIX_COUNTERS];
    std::memcpy(counters, ctx->ring.memory, HEAD);
    if (!accept(counters)) return hipSuccess;
    if (!whole)
        return picca_host::download(ctx->ring, B.weights, bytes - HEAD, ctx->stream, add);
    add(ctx->ring.memory + HEAD, 0, bytes - HEAD);
    return hipSuccess;
}

