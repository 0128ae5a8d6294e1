// Batched quasar-continuum fit on gfx950 (MI355X).
//
// Minimises, for every forest independently, the objective of picca's continuum fit
// (LeastsSquaresContModel.__call__,
// py/picca/delta_extraction/least_squares/least_squares_cont_model.py:65-95):
//     chi2(a, b) = sum_{ivar>0} (f - C)^2 W - sum_{ivar>0} log W,   C = (a + b x) m,
// with x = (log_lambda - Lmin) / (Lmax - Lmin), m the mean continuum and
// W = 1 / C^2 / (eta var_pipe + var_lss + fudge / var_pipe), var_pipe = 1 / ivar / C^2
// (:141-192).  Substituting var_pipe, W = 1 / D(C) with
//     D(C) = eta / ivar + var_lss C^2 + fudge ivar C^4,
// so chi2 = sum (f - C)^2 / D + log D: smooth in (a, b), with closed-form first and second
// derivatives.  With use_constant_weight W = 1 and chi2 is the plain sum of squares.
//
// One workgroup of 1, 2, 4 or 8 waves per forest, ten pixels a lane: the pixels' inputs are
// read once and stay in registers over the whole fit (flux, mean continuum, x, eta / ivar,
// var_lss, fudge ivar).  The six sums (chi2, gradient, Hessian) are reduced across the waves
// (DPP, then LDS), and every lane runs the same Levenberg-Marquardt iteration on them (damped
// Newton; a step is taken only when it lowers chi2).  Reading the 56 bytes of a pixel again for
// every evaluation (5.4 of them) bound the fit by HBM: 827 us for 20000 forests of 143 to 621
// pixels at 4.6 TB/s; from registers it takes 333 us, of which the one read is 145 us at the
// card's copy rate and the rest the divisions and the sums.  Ten pixels a lane (two waves per
// SIMD) put a forest of the log10-lambda grid on one wave; six (three waves per SIMD, two waves
// a forest, which repeat the serial step and meet at a barrier) took 518 us.  The sum of log W
// takes one logarithm per lane: the mantissas of D are multiplied and their exponents added.
// Forests beyond 8 x 64 x 10 pixels read their inputs per evaluation, one wave each.
//
// The fit stops when the Newton decrement g^T H^-1 g / 2 (Migrad's EDM) falls below tol * max(1,
// |chi2|).  The slope stays at 0 for order-0 forests (py/picca/delta_extraction/
// expected_fluxes/utils.py:109).  The validity checks of compute_continuum (:111-120:
// not converged, then negative, then all-zero continuum, each overriding the previous)
// run on the final parameters.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "device_util.h"
#include "engine.h"

namespace picca {

namespace {

struct Sums {
    double chi, ga, gb, haa, hab, hbb;
};

__device__ __forceinline__ double wave_sum(double v) {
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
    return v;
}

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

// Sum over the wave, in every lane (row_shr 1, 2, 4, 8, then row_bcast 15 and 31: lane 63 holds
// the total).  Every lane of the wave is active.
__device__ __forceinline__ double wave_total(double v) {
    v += dpp_or_zero<0x111, 0xf>(v);
    v += dpp_or_zero<0x112, 0xf>(v);
    v += dpp_or_zero<0x114, 0xf>(v);
    v += dpp_or_zero<0x118, 0xf>(v);
    v += dpp_or_zero<0x142, 0xa>(v);
    v += dpp_or_zero<0x143, 0xc>(v);
    const uint64_t b = (uint64_t)__double_as_longlong(v);
    const uint32_t lo = __builtin_amdgcn_readlane((uint32_t)b, 63);
    const uint32_t hi = __builtin_amdgcn_readlane((uint32_t)(b >> 32), 63);
    return __longlong_as_double((long long)(((uint64_t)hi << 32) | lo));
}

// A lane's pixels of the register kernel.
constexpr int PPL = CONT_PIXELS_PER_LANE;
struct LanePixels {
    double f[PPL], m[PPL], x[PPL];
    double p[PPL], lss[PPL], q[PPL];   // eta / ivar, var_lss, fudge ivar
    uint32_t used;                     // bit k: pixel k has ivar > 0
};

// The six sums at (a, b) of a lane's pixels, then of the forest.  CONSTANT: all weights 1.
template <int WAVES, bool CONSTANT>
__device__ Sums evaluate_lanes(const LanePixels &P, double a, double b, double (*part)[6],
                               int wave) {
    Sums s{0, 0, 0, 0, 0, 0};
    double mant = 1.0;
    int expo = 0;
#pragma unroll
    for (int k = 0; k < PPL; ++k) {
        if (!((P.used >> k) & 1u)) continue;
        const double m = P.m[k], x = P.x[k];
        const double C = fma(b, x, a) * m;
        const double r = P.f[k] - C;
        double dT, d2T;
        if (CONSTANT) {
            s.chi = fma(r, r, s.chi);
            dT = -2.0 * r;
            d2T = 2.0;
        } else {
            const double C2 = C * C;
            const double qc = P.q[k] * C2;
            const double D = fma(C2, P.lss[k] + qc, P.p[k]);
            const double D1 = C * fma(4.0, qc, 2.0 * P.lss[k]);    // dD/dC
            const double D2 = fma(12.0, qc, 2.0 * P.lss[k]);       // d2D/dC2
            const double inv = 1.0 / D;
            const double g = r * inv;                               // r / D
            const double h = D1 * inv;
            const double w = fma(-g, g, inv);                       // 1 / D - r^2 / D^2
            s.chi = fma(r, g, s.chi);
            if (D > 0 && D < INFINITY) {
                mant *= __builtin_amdgcn_frexp_mant(D);
                expo += __builtin_amdgcn_frexp_exp(D);
            } else {
                s.chi += log(D);
            }
            // dT/dC = -2 r / D - r^2 D' / D^2 + D' / D
            dT = fma(D1, w, -2.0 * g);
            // d2T/dC2 = 2/D + 4 r D'/D^2 + 2 r^2 D'^2/D^3 - r^2 D''/D^2 + D''/D - D'^2/D^2
            d2T = fma(D2, w, fma(h, fma(2.0 * g * g, D1, fma(4.0, g, -h)), 2.0 * inv));
        }
        const double mx = m * x;
        const double t = d2T * m, tx = d2T * mx;
        s.ga = fma(dT, m, s.ga);
        s.gb = fma(dT, mx, s.gb);
        s.haa = fma(t, m, s.haa);
        s.hab = fma(t, mx, s.hab);
        s.hbb = fma(tx, mx, s.hbb);
    }
    if (!CONSTANT) s.chi += fma((double)expo, 0.69314718055994530942, log(mant));
    s.chi = wave_total(s.chi);
    s.ga = wave_total(s.ga);
    s.gb = wave_total(s.gb);
    s.haa = wave_total(s.haa);
    s.hab = wave_total(s.hab);
    s.hbb = wave_total(s.hbb);
    if constexpr (WAVES > 1) {
        // every wave adds the waves' sums in one order, so that all take the same steps
        if ((threadIdx.x & 63) == 0) {
            double *o = part[wave];
            o[0] = s.chi;
            o[1] = s.ga;
            o[2] = s.gb;
            o[3] = s.haa;
            o[4] = s.hab;
            o[5] = s.hbb;
        }
        __syncthreads();
        double t[6] = {0, 0, 0, 0, 0, 0};
        for (int v = 0; v < WAVES; ++v)
#pragma unroll
            for (int c = 0; c < 6; ++c) t[c] += part[v][c];
        s = Sums{t[0], t[1], t[2], t[3], t[4], t[5]};
    }
    return s;
}

__device__ Sums evaluate(const ContIn &I, int64_t o, int n, double a, double b, bool constant,
                         int lane) {
    Sums s{0, 0, 0, 0, 0, 0};
    for (int k = lane; k < n; k += 64) {
        const double iv = I.ivar[o + k];
        if (!(iv > 0)) continue;
        const double m = I.mean_cont[o + k];
        const double x = I.x[o + k];
        const double f = I.flux[o + k];
        const double C = (a + b * x) * m;
        const double r = f - C;
        double T, dT, d2T;
        if (constant) {
            T = r * r;
            dT = -2.0 * r;
            d2T = 2.0;
        } else {
            const double eta = I.eta[o + k];
            const double lss = I.var_lss[o + k];
            const double fud = I.fudge[o + k];
            const double C2 = C * C;
            const double D = eta / iv + lss * C2 + fud * iv * C2 * C2;
            const double D1 = 2.0 * lss * C + 4.0 * fud * iv * C2 * C;   // dD/dC
            const double D2 = 2.0 * lss + 12.0 * fud * iv * C2;           // d2D/dC2
            const double inv = 1.0 / D;
            const double q = r * inv;                                     // r / D
            T = r * q + log(D);
            // dT/dC = -2 r / D - r^2 D' / D^2 + D' / D
            dT = -2.0 * q - q * q * D1 + D1 * inv;
            // d2T/dC2 = 2/D + 4 r D'/D^2 + 2 r^2 D'^2/D^3 - r^2 D''/D^2 + D''/D - D'^2/D^2
            d2T = 2.0 * inv + 4.0 * q * D1 * inv + 2.0 * q * q * D1 * D1 * inv -
                  q * q * D2 + D2 * inv - D1 * D1 * inv * inv;
        }
        const double mx = m * x;
        s.chi += T;
        s.ga += dT * m;
        s.gb += dT * mx;
        s.haa += d2T * m * m;
        s.hab += d2T * m * mx;
        s.hbb += d2T * mx * mx;
    }
    s.chi = wave_sum(s.chi);
    s.ga = wave_sum(s.ga);
    s.gb = wave_sum(s.gb);
    s.haa = wave_sum(s.haa);
    s.hab = wave_sum(s.hab);
    s.hbb = wave_sum(s.hbb);
    return s;
}

// Newton (lambda = 0) or damped step; false when the damped Hessian is not positive
__device__ __forceinline__ bool solve_step(const Sums &s, bool free_b, double lambda,
                                           double &da, double &db) {
    const double haa = s.haa * (1.0 + lambda);
    if (!free_b) {
        if (!(haa > 0)) return false;
        da = -s.ga / haa;
        db = 0.0;
        return true;
    }
    const double hbb = s.hbb * (1.0 + lambda);
    const double det = haa * hbb - s.hab * s.hab;
    if (!(haa > 0) || !(det > 0)) return false;
    da = -(hbb * s.ga - s.hab * s.gb) / det;
    db = -(haa * s.gb - s.hab * s.ga) / det;
    return true;
}

}  // namespace

namespace {

// Levenberg-Marquardt from (a, b); `evaluate(a, b)` gives the sums.  Returns the status.
template <class Evaluate>
__device__ __forceinline__ int fit_forest(const ContConst &K, bool free_b, double &a, double &b,
                                          Sums &s, int &evals, Evaluate evaluate) {
    s = evaluate(a, b);
    evals = 1;
    int status = 1;   // 1: not converged within max_iter
    double lambda = 0.0;
    for (int it = 0; it < K.max_iter; ++it) {
        // convergence: Newton decrement at the current point
        double na, nb;
        if (solve_step(s, free_b, 0.0, na, nb)) {
            const double edm = -0.5 * (s.ga * na + s.gb * nb);
            if (edm < K.tol * fmax(1.0, fabs(s.chi)) || edm < K.tol_abs) {
                status = 0;
                break;
            }
        }
        double da, db;
        if (!solve_step(s, free_b, lambda, da, db)) {
            lambda = lambda == 0.0 ? 1e-3 : lambda * 10.0;
            if (lambda > 1e12) break;
            continue;
        }
        const Sums t = evaluate(a + da, b + db);
        ++evals;
        if (t.chi < s.chi) {
            a += da;
            b += db;
            s = t;
            lambda = lambda * 0.1;
            if (lambda < 1e-9) lambda = 0.0;
        } else {
            lambda = lambda == 0.0 ? 1e-3 : lambda * 10.0;
            if (lambda > 1e12) {   // no representable improvement left: at the minimum
                status = 0;
                break;
            }
        }
    }
    return status;
}

// the reference's checks of the final continuum in its order, later ones overriding earlier ones
__device__ __forceinline__ int check_fit(int status, const Sums &s, bool negative, bool nonzero) {
    if (status == 0 && !(s.chi == s.chi)) status = 4;
    if (negative) status = 2;
    if (!nonzero) status = 3;
    return status;
}

}  // namespace

template <int WAVES, bool CONSTANT>
__global__ __launch_bounds__(64 * WAVES, 2) void cont_fit_lanes_kernel(
    ContConst K, ContIn I, ContOut O, const int32_t *__restrict__ forests) {
    __shared__ double part[2][WAVES][6];
    __shared__ int s_flags[2];
    __shared__ int s_ndata;
    const int64_t f = forests[blockIdx.x];
    const int tid = threadIdx.x;
    const int wave = tid >> 6;
    const int64_t o = I.off[f];
    const int n = (int)(I.off[f + 1] - o);
    LanePixels P;
    P.used = 0;
#pragma unroll
    for (int k = 0; k < PPL; ++k) {
        const int at = tid + 64 * WAVES * k;
        const bool in = at < n;
        const int64_t p = o + (in ? at : 0);
        const double iv = in ? I.ivar[p] : 0.0;
        P.m[k] = in ? I.mean_cont[p] : 0.0;
        P.x[k] = in ? I.x[p] : 0.0;
        P.f[k] = in ? I.flux[p] : 0.0;
        if (!CONSTANT) {
            const bool use = iv > 0;
            P.lss[k] = in ? I.var_lss[p] : 0.0;
            P.p[k] = use ? I.eta[p] / iv : 0.0;
            P.q[k] = use ? I.fudge[p] * iv : 0.0;
        }
        P.used |= iv > 0 ? 1u << k : 0u;
    }
    if (tid < 2) s_flags[tid] = 0;
    if (tid == 0) s_ndata = 0;
    const bool free_b = I.order[f] != 0;
    double a = I.a0[f];
    double b = free_b ? I.b0[f] : 0.0;
    Sums s;
    int evals, turn = 0;
    int status = fit_forest(K, free_b, a, b, s, evals, [&](double at, double bt) {
        turn ^= 1;   // the waves' sums alternate between two buffers: one barrier a step
        return evaluate_lanes<WAVES, CONSTANT>(P, at, bt, part[turn], wave);
    });
    // validity of the final continuum over every pixel of the forest
    bool negative = false, nonzero = false;
#pragma unroll
    for (int k = 0; k < PPL; ++k) {
        const double C = (a + b * P.x[k]) * P.m[k];
        const bool in = tid + 64 * WAVES * k < n;
        negative |= in && C < 0;
        nonzero |= in && C != 0;
    }
    if (WAVES > 1) __syncthreads();   // s_flags and s_ndata are set
    const uint64_t neg = __ballot(negative), non = __ballot(nonzero);
    int nd = __popc(P.used);
    for (int off = 32; off > 0; off >>= 1) nd += __shfl_xor(nd, off, 64);
    if ((tid & 63) == 0) {
        if (neg) atomicOr(&s_flags[0], 1);
        if (non) atomicOr(&s_flags[1], 1);
        atomicAdd(&s_ndata, nd);
    }
    __syncthreads();
    if (tid == 0) {
        O.a[f] = a;
        O.b[f] = b;
        O.chi2[f] = s.chi;
        O.ndata[f] = s_ndata;
        O.status[f] = check_fit(status, s, s_flags[0] != 0, s_flags[1] != 0);
        O.evals[f] = evals;
    }
}

// Forests longer than the register kernel's pixels: one wave each.
__global__ __launch_bounds__(256) void cont_fit_kernel(ContConst K, ContIn I, ContOut O,
                                                       const int32_t *__restrict__ forests,
                                                       int32_t count) {
    const int lane = threadIdx.x & 63;
    const int k = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (k >= count) return;   // whole waves leave together
    const int64_t f = forests[k];
    const int64_t o = I.off[f];
    const int n = (int)(I.off[f + 1] - o);
    const bool free_b = I.order[f] != 0;
    const bool constant = K.use_constant_weight != 0;
    double a = I.a0[f];
    double b = free_b ? I.b0[f] : 0.0;
    Sums s;
    int evals;
    int status = fit_forest(K, free_b, a, b, s, evals, [&](double at, double bt) {
        return evaluate(I, o, n, at, bt, constant, lane);
    });
    // validity of the final continuum over every pixel of the forest
    bool negative = false, nonzero = false;
    int ndata = 0;
    for (int k = lane; k < n; k += 64) {
        const double C = (a + b * I.x[o + k]) * I.mean_cont[o + k];
        negative |= C < 0;
        nonzero |= C != 0;
        ndata += I.ivar[o + k] > 0 ? 1 : 0;
    }
    negative = __ballot(negative) != 0;
    nonzero = __ballot(nonzero) != 0;
    for (int off = 32; off > 0; off >>= 1) ndata += __shfl_xor(ndata, off, 64);
    status = check_fit(status, s, negative, nonzero);
    if (lane == 0) {
        O.a[f] = a;
        O.b[f] = b;
        O.chi2[f] = s.chi;
        O.ndata[f] = ndata;
        O.status[f] = status;
        O.evals[f] = evals;
    }
}

template <int WAVES>
static void launch_fit_lanes(const ContConst &K, const ContIn &I, const ContOut &O,
                             const int32_t *forests, int64_t count, hipStream_t stream) {
    if (count <= 0) return;
    auto kern = K.use_constant_weight ? cont_fit_lanes_kernel<WAVES, true>
                                      : cont_fit_lanes_kernel<WAVES, false>;
    hipLaunchKernelGGL(kern, dim3((unsigned)count), dim3(64 * WAVES), 0, stream, K, I, O,
                       forests);
}

hipError_t launch_cont_fit(const ContConst &K, const ContIn &I, const ContOut &O,
                           const int32_t *forests, const int64_t *class_begin,
                           hipStream_t stream) {
    // the longest forests first: the short ones fill the grid's end
    const int64_t *c = class_begin;
    const int64_t rest = c[5] - c[4];
    if (rest > 0)
        hipLaunchKernelGGL(cont_fit_kernel, dim3((unsigned)((rest + 3) / 4)), dim3(256), 0,
                           stream, K, I, O, forests + c[4], (int32_t)rest);
    launch_fit_lanes<8>(K, I, O, forests + c[3], c[4] - c[3], stream);
    launch_fit_lanes<4>(K, I, O, forests + c[2], c[3] - c[2], stream);
    launch_fit_lanes<2>(K, I, O, forests + c[1], c[2] - c[1], stream);
    launch_fit_lanes<1>(K, I, O, forests + c[0], c[1] - c[0], stream);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------------------
// Mean-continuum update of the DR16 iteration
// (Dr16ExpectedFlux.compute_expected_flux, py/picca/delta_extraction/expected_fluxes/
// dr16_expected_flux.py:380-464).
//
// cont_stack_kernel: ExpectedFlux._compute_mean_cont (py/picca/delta_extraction/
// expected_flux.py:256-308) with the forest weights of Dr16ExpectedFlux.compute_forest_weights
// (dr16_expected_flux.py:466-488, var_lss_mod = 1): over the pixels of the forests whose
// last fit is valid, sum F / (C + 1e-16) * w and w in the pixel's rest-frame bin, with
// w = 1 / (eta var_pipe + var_lss + fudge / var_pipe), var_pipe = 1 / ivar / C^2 and
// w = 0 where ivar <= 0.  One wave per forest; the bins live in LDS per workgroup and are
// added to HBM once per workgroup.
__global__ void __launch_bounds__(256)
cont_stack_kernel(ContIn I, const double *__restrict__ a_fit, const double *__restrict__ b_fit,
                  const int32_t *__restrict__ status, const int32_t *__restrict__ bins,
                  int32_t nbins, double *__restrict__ sum_ratio,
                  double *__restrict__ sum_weight, int64_t n_forests) {
    extern __shared__ __align__(16) unsigned char smem[];
    double *h_ratio = reinterpret_cast<double *>(smem);
    double *h_weight = h_ratio + nbins;
    for (int k = threadIdx.x; k < nbins; k += blockDim.x) {
        h_ratio[k] = 0.0;
        h_weight[k] = 0.0;
    }
    __syncthreads();
    const int lane = threadIdx.x & 63;
    const int64_t waves = (int64_t)gridDim.x * (blockDim.x >> 6);
    for (int64_t f = (int64_t)blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6); f < n_forests;
         f += waves) {
        if (status[f] != 0) continue;
        const double a = a_fit[f], b = b_fit[f];
        const int64_t o = I.off[f];
        const int n = (int)(I.off[f + 1] - o);
        for (int k = lane; k < n; k += 64) {
            const double iv = I.ivar[o + k];
            if (!(iv > 0)) continue;
            const double C = (b * I.x[o + k] + a) * I.mean_cont[o + k];
            const double var_pipe = 1.0 / iv / (C * C);
            const double w = 1.0 / (I.eta[o + k] * var_pipe + I.var_lss[o + k] +
                                    I.fudge[o + k] / var_pipe);
            const double ratio = I.flux[o + k] / (C + 1e-16);
            const int bin = bins[o + k];
            atomicAdd(&h_ratio[bin], ratio * w);
            atomicAdd(&h_weight[bin], w);
        }
    }
    __syncthreads();
    for (int k = threadIdx.x; k < nbins; k += blockDim.x) {
        if (h_weight[k] != 0.0) {
            unsafeAtomicAdd(&sum_ratio[k], h_ratio[k]);
            unsafeAtomicAdd(&sum_weight[k], h_weight[k]);
        }
    }
}

// cont_interp_kernel: the new get_mean_cont, scipy's interp1d(x, y,
// fill_value="extrapolate") (linear, nearest end interval outside [x0, x_{n-1}]), at every
// pixel's rest-frame log lambda, times the transmission correction
// (py/picca/delta_extraction/expected_fluxes/utils.py:49-64).  The interval and the slope
// follow scipy's _call_linear: i = searchsorted(x, v) clipped to [1, n - 1],
// y = (y_i - y_{i-1}) / (x_i - x_{i-1}) * (v - x_{i-1}) + y_{i-1}.
__global__ void __launch_bounds__(256)
cont_interp_kernel(const double *__restrict__ ll_rest, const double *__restrict__ trans,
                   const double *__restrict__ xs, const double *__restrict__ ys, int32_t n,
                   double *__restrict__ mean_cont, int64_t npix) {
    extern __shared__ __align__(16) unsigned char smem[];
    double *sx = reinterpret_cast<double *>(smem);
    double *sy = sx + n;
    for (int k = threadIdx.x; k < n; k += blockDim.x) {
        sx[k] = xs[k];
        sy[k] = ys[k];
    }
    __syncthreads();
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; p < npix; p += stride) {
        const double v = ll_rest[p];
        // first index with sx[i] >= v (numpy searchsorted, side "left")
        int lo = 0, hi = n;
        while (lo < hi) {
            const int mid = (lo + hi) >> 1;
            if (sx[mid] < v) lo = mid + 1;
            else hi = mid;
        }
        const int i = lo < 1 ? 1 : (lo > n - 1 ? n - 1 : lo);
        const double x_lo = sx[i - 1], x_hi = sx[i];
        const double y_lo = sy[i - 1], y_hi = sy[i];
        const double slope = (y_hi - y_lo) / (x_hi - x_lo);
        mean_cont[p] = (slope * (v - x_lo) + y_lo) * trans[p];
    }
}

hipError_t launch_cont_stack(const ContIn &I, const double *a, const double *b,
                             const int32_t *status, const int32_t *bins, int32_t nbins,
                             double *sum_ratio, double *sum_weight, int64_t n_forests,
                             int num_cus, hipStream_t stream) {
    if (n_forests <= 0 || nbins <= 0) return hipSuccess;
    const size_t lds = 2 * sizeof(double) * (size_t)nbins;
    int64_t blocks = (n_forests + 3) / 4;
    if (blocks > 8 * (int64_t)num_cus) blocks = 8 * (int64_t)num_cus;
    hipError_t err = hipFuncSetAttribute((const void *)cont_stack_kernel,
                                         hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (err != hipSuccess) return err;
    hipLaunchKernelGGL(cont_stack_kernel, dim3((unsigned)blocks), dim3(256), lds, stream, I, a,
                       b, status, bins, nbins, sum_ratio, sum_weight, n_forests);
    return hipGetLastError();
}

hipError_t launch_cont_interp(const double *ll_rest, const double *trans, const double *xs,
                              const double *ys, int32_t n, double *mean_cont, int64_t npix,
                              int num_cus, hipStream_t stream) {
    if (npix <= 0) return hipSuccess;
    const size_t lds = 2 * sizeof(double) * (size_t)n;
    int64_t blocks = (npix + 255) / 256;
    if (blocks > 16 * (int64_t)num_cus) blocks = 16 * (int64_t)num_cus;
    hipError_t err = hipFuncSetAttribute((const void *)cont_interp_kernel,
                                         hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (err != hipSuccess) return err;
    hipLaunchKernelGGL(cont_interp_kernel, dim3((unsigned)blocks), dim3(256), lds, stream,
                       ll_rest, trans, xs, ys, n, mean_cont, npix);
    return hipGetLastError();
}

}  // namespace picca
