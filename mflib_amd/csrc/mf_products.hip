// Per-detection products (gfx950): what SingleChannel::Detector::detect
// derives for every peak once PeakFinder has picked it
// (src/singleChannel/detector.cpp:537-664):
//   - the correlation coefficient at the peak, clamped to [-1, 1] (574-575);
//   - the sub-sample time shift, by a parabola through three lags
//     (quadraticRefinement, 38-89) or by Lanczos-windowed sinc
//     interpolation on a grid of shifts (lanczosRefinement, 91-152);
//   - the amplitude scaling factors of the detected window against the
//     template, Gibbons & Ringdal (2006) and Schaff & Richards (2014)
//     (src/singleChannel/relativeMagnitude.cpp:35-58, 273-388), when the
//     window fits the signal (detector.cpp:578-585) and is not constant
//     (relativeMagnitude.cpp:330-338).
// One wavefront per detection.  Everything is FP64 for both signal
// precisions, as the reference's double instantiation computes it; the
// float instantiation's own arithmetic is not reproduced (its Lanczos grid
// position optIndex + shift is rounded to FP32, which drops the fraction
// for lags beyond 2^23, and its detected-window "mean" is the float sum,
// relativeMagnitude.cpp:110-125).
#include <hip/hip_runtime.h>

#include <cfloat>

#include "mf_device.hpp"
#include "mf_kernels.hpp"

using namespace mfdev;

namespace mfk {

namespace {

// The refinements are compared bit for bit with a CPU restatement:
// no contraction of products into sums in this file.
#pragma clang fp contract(off)

constexpr int kWave = 64;

// sinc of the Lanczos kernel sinc(x) sinc(x / a) (detector.cpp:91-109):
// sinc(0) = 1 below |x| <= 100 eps; the window keeps every x with
// int(|x|) <= a.
__device__ __forceinline__ double sinc(double x)
{
    double r = 1.0;
    if (fabs(x) > DBL_EPSILON * 100) {
        const double pix = M_PI * x;
        r = sin(pix) / pix;
    }
    return r;
}

// std::min's selection rule, (b < a) ? b : a, which keeps `a` when either is NaN
__device__ __forceinline__ double std_min(double a, double b) { return (b < a) ? b : a; }

// quadraticRefinement (detector.cpp:38-89): the vertex of the parabola
// through lags p-1, p, p+1 (of |rho| when absval), 0 at either end or when
// lag p is neither the maximum nor the minimum of the three.
template <typename T>
__device__ double quadratic_shift(gptr<const T> xc, int n, int p, double dt, int absval)
{
    if (!(p > 0 && p < n - 1)) { return 0.0; }
    double y1 = static_cast<double>(xc[p - 1]);
    double y2 = static_cast<double>(xc[p]);
    double y3 = static_cast<double>(xc[p + 1]);
    if (absval) {
        y1 = fabs(y1);
        y2 = fabs(y2);
        y3 = fabs(y3);
    }
    if (y2 < y1 || y2 < y3) {
        if (y2 < y1 && y2 < y3) {
            y1 = -y1;
            y2 = -y2;
            y3 = -y3;
        } else {
            return 0.0;
        }
    }
    y1 = std_min(y2 - 100 * DBL_EPSILON, y1);
    y3 = std_min(y2 - 100 * DBL_EPSILON, y3);
    const double num = dt * (y1 - y3);
    const double den = 2 * (y1 - 2 * y2 + y3);
    return num / den;
}

// The larger of two grid points' values, equal values going to the smaller
// index; index 0 is no point.
__device__ __forceinline__ void keep_best(double &best, int &bestIdx, double ob, int oi)
{
    if (oi != 0 && (bestIdx == 0 || ob > best || (ob == best && oi < bestIdx))) {
        best = ob;
        bestIdx = oi;
    }
}

// cos and sin of pi j / a for the taps j = -a - 1 .. a - 1 of the Lanczos
// window (at most kLanczosTable of them), a block's own in LDS.
constexpr int kLanczosTable = 1024;
struct __align__(16) Turn {
    double c, s;
};

// lanczosRefinement (detector.cpp:111-152) over one block: thread l
// evaluates the interpolant at grid points idx = l + 1, l + 1 + NTH, ...
// (shift = -0.5 + idx / nRefine), summing its 2a + 1 taps in the
// reference's order; the result is the first grid point of the largest
// value, as the sequential strict '>' scan from -DBL_MAX picks it.
// With a table, the window's sine of a tap at frac + j is
// sin(pi frac / a) cos(pi j / a) + cos(pi frac / a) sin(pi j / a), two
// operations where a call of sin() took a hundred; the tap at frac - 1,
// which may be close to 0, keeps a sine of its own, so no tap's weight
// cancels.  Measured, 430 detections of FP64 rows, a = 51 and 99 grid points:
// 90 us with a sine per tap on one wave, 48 us with the table on two.
template <typename T, int NTH, bool TABLE>
__device__ double lanczos_shift(gptr<const T> xc, int n, int p, double dt, int absval, int a, int nRefine,
                                Turn *table, double *redV, int *redI)
{
    const int lane = threadIdx.x;
    const double dtWork = 1.0 / static_cast<double>(nRefine);
    if constexpr (TABLE) {
        for (int i = lane; i < 2 * a + 1; i += NTH) {
            const double ang = M_PI * (static_cast<double>(i - a - 1) / a);
            table[i] = Turn{cos(ang), sin(ang)};
        }
        __syncthreads();
    }
    double best = 0.0;
    int bestIdx = 0;  // 0: none (grid indices start at 1)
    for (int idx = lane + 1; idx < nRefine; idx += NTH) {
        const double shift = -0.5 + dtWork * idx;
        const double x = p + shift;
        const int fl = static_cast<int>(floor(x));
        // The taps sit at xi = frac + k - 1 (frac = x - floor(x), exact), so
        // sin(pi xi) = (-1)^(k-1) sin(pi frac): one sine per grid point for
        // the first sinc factor instead of one per tap.  The window's own
        // factor sinc(xi / a) keeps its sine per tap.
        const double frac = x - static_cast<double>(fl);
        const double sFrac = sin(M_PI * frac);
        double sWin = 0.0, cWin = 0.0, sOne = 0.0;  // of pi frac / a; sin of pi (frac - 1) / a
        if constexpr (TABLE) {
            sWin = sin(M_PI * (frac / a));
            cWin = cos(M_PI * (frac / a));
            sOne = sin(M_PI * ((frac - 1.0) / a));
        }
        double y = 0.0;
        for (int k = -a; k <= a; ++k) {
            const long long i = static_cast<long long>(fl) - k + 1;  // no int overflow near 2^31 lags
            const double xi = x - static_cast<double>(i);
            double v = 0.0;
            if (i >= 0 && i < n) { v = static_cast<double>(xc[i]); }
            double w = 0.0;
            if (static_cast<int>(fabs(xi)) <= a) {
                const double s1 = ((k - 1) & 1) ? -sFrac : sFrac;
                const double sinc1 = fabs(xi) > DBL_EPSILON * 100 ? s1 / (M_PI * xi) : 1.0;
                if constexpr (TABLE) {
                    // xi = frac + j; the interpolant's tap k has j = k - 1
                    const Turn t = table[k + a];
                    const double s2 = k == 0 ? sOne : sWin * t.c + cWin * t.s;
                    const double xa = xi / a;
                    w = sinc1 * (fabs(xa) > DBL_EPSILON * 100 ? s2 / (M_PI * xa) : 1.0);
                } else {
                    w = sinc1 * sinc(xi / a);
                }
            }
            y = y + v * w;
        }
        if (absval) { y = fabs(y); }
        // a lane's own points are visited in increasing idx: strict '>' keeps the first
        if (y > -DBL_MAX && (bestIdx == 0 || y > best)) {
            best = y;
            bestIdx = idx;
        }
    }
    // across lanes, then waves
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        const double ob = __shfl_xor(best, o, kWave);
        const int oi = __shfl_xor(bestIdx, o, kWave);
        keep_best(best, bestIdx, ob, oi);
    }
    if constexpr (NTH > kWave) {
        if (lane % kWave == 0) {
            redV[lane / kWave] = best;
            redI[lane / kWave] = bestIdx;
        }
        __syncthreads();
#pragma unroll
        for (int w = 0; w < NTH / kWave; ++w) { keep_best(best, bestIdx, redV[w], redI[w]); }
    }
    if (bestIdx == 0) { return 0.0; }
    const double shift = -0.5 + dtWork * bestIdx;
    return dt * shift;
}

// RelativeMagnitude's factors of y[0..Lt) against t[0..Lt) over one
// wavefront, two passes: the means, then the demeaned sums of squares and
// products.  Returns false for a constant window (no factors).
template <typename T>
__device__ bool amplitude_factors(gptr<const double> t, gptr<const T> y, int Lt, double &gr, double &sr)
{
    const int lane = threadIdx.x % kWave;
    double st = 0.0, sy = 0.0;
    for (int i = lane; i < Lt; i += kWave) {
        st += t[i];
        sy += static_cast<double>(y[i]);
    }
    const double mt = wave_sum(st) / Lt;
    const double my = wave_sum(sy) / Lt;
    double xx = 0.0, yy = 0.0, xy = 0.0;
    for (int i = lane; i < Lt; i += kWave) {
        const double dx = t[i] - mt;
        const double dy = static_cast<double>(y[i]) - my;
        xx += dx * dx;
        yy += dy * dy;
        xy += dx * dy;
    }
    xx = wave_sum(xx);
    yy = wave_sum(yy);
    xy = wave_sum(xy);
    if (yy == 0.0) { return false; }  // a constant window throws in the reference
    gr = fabs(xy) / xx;
    sr = sqrt(yy / xx);
    return true;
}

// One detection per block: one wave, or with WAVES = 2 the Lanczos grid on
// two waves and the window table in LDS.
template <typename T, int WAVES>
__global__ __launch_bounds__(WAVES * kWave) void products_kernel(const ProductJob *__restrict__ jobs, int absval,
                                                                int interp, int lanczosAlpha, int lanczosPoints,
                                                                ProductOut *__restrict__ out)
{
    constexpr bool TABLE = WAVES > 1;
    __shared__ Turn table[TABLE ? kLanczosTable : 1];
    __shared__ double redV[WAVES];
    __shared__ int redI[WAVES];
    const ProductJob job = jobs[blockIdx.x];
    const int lane = threadIdx.x;
    const gptr<const T> xc = to_global(static_cast<const T *>(job.rho));
    const int n = job.nOut;
    const int p = job.peak;

    double shift = 0.0;
    if (interp == kInterpQuadratic) {
        shift = quadratic_shift<T>(xc, n, p, job.dt, absval);
    } else if (interp == kInterpLanczos) {
        shift = lanczos_shift<T, WAVES * kWave, TABLE>(xc, n, p, job.dt, absval, lanczosAlpha, lanczosPoints, table,
                                                      redV, redI);
    }

    // amplitude scaling factors: two passes over the template and the window
    int flags = 0;
    double gr = 0.0, sr = 0.0;
    const int Lt = job.Lt;
    if (static_cast<long long>(p) + Lt > job.sigLen) {
        flags |= kProductTruncated;
    } else if (amplitude_factors<T>(to_global(job.tmpl), to_global(static_cast<const T *>(job.sig)) + p, Lt, gr,
                                    sr)) {
        flags |= kProductAmplitude;
    }

    if (lane == 0) {
        const double r = static_cast<double>(xc[p]);
        ProductOut o;
        o.rho = fmax(-1.0, fmin(1.0, r));  // NaN -> 1, as std::max(-1, std::min(1, NaN))
        o.shift = shift;
        o.alphaGR = gr;
        o.alphaSR = sr;
        o.flags = flags;
        o.pad = 0;
        out[blockIdx.x] = o;
    }
}

// One wavefront per window: window k is windows[k * ld .. k * ld + Lt).
template <typename T>
__global__ __launch_bounds__(kWave) void amplitude_kernel(const double *__restrict__ tmpl, int Lt,
                                                         const T *__restrict__ windows, long long ld,
                                                         ProductOut *__restrict__ out)
{
    double gr = 0.0, sr = 0.0;
    const bool ok = amplitude_factors<T>(to_global(tmpl), to_global(windows) + blockIdx.x * ld, Lt, gr, sr);
    if (threadIdx.x == 0) {
        ProductOut o{};
        o.alphaGR = gr;
        o.alphaSR = sr;
        o.flags = ok ? kProductAmplitude : 0;
        out[blockIdx.x] = o;
    }
}

}  // namespace

hipError_t launch_amplitude(int precision, const double *dTmpl, int Lt, const void *dWindows, long long ld,
                            int nWindows, ProductOut *dOut, hipStream_t stream)
{
    if (nWindows <= 0) { return hipSuccess; }
    if (precision == 0) {
        hipLaunchKernelGGL(amplitude_kernel<float>, dim3(nWindows), dim3(kWave), 0, stream, dTmpl, Lt,
                           static_cast<const float *>(dWindows), ld, dOut);
    } else {
        hipLaunchKernelGGL(amplitude_kernel<double>, dim3(nWindows), dim3(kWave), 0, stream, dTmpl, Lt,
                           static_cast<const double *>(dWindows), ld, dOut);
    }
    return hipGetLastError();
}

hipError_t launch_products(int precision, const ProductJob *dJobs, int nJobs, int absval, int interp,
                           int lanczosAlpha, int lanczosPoints, ProductOut *dOut, hipStream_t stream)
{
    if (nJobs <= 0) { return hipSuccess; }
    // a Lanczos window that fits the table runs on two waves (the default 51
    // taps a side does, and 99 grid points fill them); longer windows and
    // the other kinds on one
    const bool table = interp == kInterpLanczos && 2LL * lanczosAlpha + 1 <= kLanczosTable;
    const auto launch = [&](auto kernel, int threads) {
        hipLaunchKernelGGL(kernel, dim3(nJobs), dim3(threads), 0, stream, dJobs, absval, interp, lanczosAlpha,
                           lanczosPoints, dOut);
    };
    if (precision == 0) {
        table ? launch(products_kernel<float, 2>, 2 * kWave) : launch(products_kernel<float, 1>, kWave);
    } else {
        table ? launch(products_kernel<double, 2>, 2 * kWave) : launch(products_kernel<double, 1>, kWave);
    }
    return hipGetLastError();
}

}  // namespace mfk
