// k-space kernels of include/fft_kernels.h evaluated on the device, and the
// closed-form spectrum (power law times BBKS transfer function).
#pragma once

#include "api_util.h"

namespace mitos {

// include/fft_kernels.h:187
__host__ __device__ __forceinline__ double sinc_d(double x) { return x == 0 ? 1. : sin(x) / x; }

// Bardeen, Bond, Kaiser & Szalay (1986), eq. G3: q = k / Gamma (k in h/Mpc)
__host__ __device__ __forceinline__ double bbks_T(double k, double Gamma) {
#pragma clang fp contract(off)
    if (k == 0) return 1.0;
    const double q = k / Gamma;
    const double a = 2.34 * q;
    const double poly = 1.0 + 3.89 * q + pow(16.1 * q, 2) + pow(5.46 * q, 3) + pow(6.71 * q, 4);
    return log(1.0 + a) / a * pow(poly, -0.25);
}

// kernel value (re, im) at one wavevector; formulas of include/fft_kernels.h
__host__ __device__ __forceinline__ cx<double> ksp_value(const KSpec& ks, double kx, double ky,
                                                         double kz, double k) {
#pragma clang fp contract(off)
    switch (ks.id) {
        case KID_CONSTANT: return mk<double>(ks.p[0], 0);               // :28-31
        case KID_INV_POISSON: return mk<double>((k > 0) ? -1.0 / k / k : 1.0, 0);  // :96-99
        case KID_DX: return mk<double>(0, kx);                         // :101-104
        case KID_DY: return mk<double>(0, ky);
        case KID_DZ: return mk<double>(0, kz);
        case KID_POWER_NO_TRANSFER: {                                  // :116-121
            if (k == 0) return mk<double>(0, 0);                       // src/primordial.c:26
            const double A_s = ks.p[0], n_s = ks.p[1], k_pivot = ks.p[2];
            return mk<double>(sqrt(A_s * pow(k / k_pivot, n_s - 1.) * k * (2. * M_PI * M_PI)),
                              0);
        }
        case KID_UNDO_WINDOW: {                                        // :198-219
            if (k == 0) return mk<double>(1.0, 0);
            const double order = ks.p[0];
            const double N = ks.p[1];
            const double boxlen = ks.p[2];
            const double W_x = sinc_d(0.5 * kx * boxlen / N);
            const double W_y = sinc_d(0.5 * ky * boxlen / N);
            const double W_z = sinc_d(0.5 * kz * boxlen / N);
            const double W = pow(W_x * W_y * W_z, order);
            return mk<double>(1.0 / W, 0);
        }
        case KID_SQRT_POWER_LAW:
            if (k == 0) return mk<double>(0, 0);
            return mk<double>(sqrt(ks.p[0] * pow(k, ks.p[1])), 0);
        case KID_BBKS:
            if (k == 0) return mk<double>(0, 0);
            return mk<double>(bbks_T(k, ks.p[0]), 0);
        case KID_LOWPASS: return mk<double>((k < ks.p[0]) ? 1.0 : 0.0, 0);          // :33-37
        case KID_HIPASS: return mk<double>((k > ks.p[0]) ? 1.0 : 0.0, 0);           // :39-43
        case KID_TOPHAT:                                                             // :45-51
            return mk<double>((k >= ks.p[0] && k <= ks.p[1]) ? 1.0 : 0.0, 0);
        case KID_ELLIPTIC_TOPHAT: {                                                  // :54-68
            const double rx = ks.p[0], ry = ks.p[1], rz = ks.p[2], eta2 = ks.p[3];
            const double kr = kx * rx + ky * ry + kz * rz;
            const double kk = kx * kx + ky * ky + kz * kz;
            const double rr = rx * rx + ry * ry + rz * rz;
            const double theta = kk * rr + (eta2 - 1) * kr * kr;
            return mk<double>((theta <= 4 * M_PI * M_PI) ? 1.0 : 0.0, 0);
        }
        case KID_TRANSLATE: {                                                        // :70-79
            const double ph = ks.p[0] * kx + ks.p[1] * ky + ks.p[2] * kz;
            return mk<double>(cos(ph), sin(ph));
        }
        case KID_GAUSSIAN: {                                                         // :81-86
            const double kR = k * ks.p[0];
            return mk<double>(exp(-kR * kR), 0);
        }
        case KID_GAUSSIAN_INV: {                                                     // :88-93
            const double kR = k * ks.p[0];
            return mk<double>(exp(kR * kR), 0);
        }
    }
    return mk<double>(0, 0);
}

// kernel_(inv_)transfer_function (include/fft_kernels.h:131-180) on the
// device: one tabulated function at two neighbouring times, tau_index and
// tau_index + 1 (the rows lo and hi), interpolated bilinearly as
// perturbSplineInterp does (src/perturb_spline.c:141-160).
struct TransferTab {
    const double* k;   // k_size wavenumbers, increasing
    const double* lo;  // T(k_j) at tau_index
    const double* hi;  // T(k_j) at tau_index + 1
    int k_size;
    double u_tau;
    int invert;        // 1: kernel_inv_transfer_function (1/T)
};

// perturbSplineFindK (src/perturb_spline.c:100-138) returns the first i from
// its search start with k_i <= k <= k_{i+1}, i.e. the largest i with k_i < k
// (0 when k = k_0), and i = k_size - 2, u = 1 above the table.  The same
// interval by bisection; below k_0 (where the reference's search has no
// defined result) the first interval extrapolates linearly.
__host__ __device__ __forceinline__ double transfer_value(const TransferTab& t, double k) {
#pragma clang fp contract(off)
    const int n = t.k_size;
    int i;
    double u;
    if (k > t.k[n - 1]) {
        i = n - 2;
        u = 1.0;
    } else {
        int lo = 0, hi = n - 2;  // the answer lies in [lo, hi]
        while (lo < hi) {
            const int mid = (lo + hi + 1) >> 1;
            if (t.k[mid] < k)
                lo = mid;
            else
                hi = mid - 1;
        }
        i = lo;
        const double left = t.k[i], right = t.k[i + 1];
        u = (k - left) / (right - left);
    }
    const double T11 = t.lo[i], T21 = t.lo[i + 1], T12 = t.hi[i], T22 = t.hi[i + 1];
    const double v = (1 - t.u_tau) * ((1 - u) * T11 + u * T21) +
                     t.u_tau * ((1 - u) * T12 + u * T22);
    return t.invert ? 1.0 / v : v;
}

// ---- write = read * kernel over the half grid (src/fft.c:257-302) ----------------
// A work-group takes 1024 (K = 4) consecutive modes of the dense grid, so every access
// is whole lines whatever the row length; it divides its first index once, and
// a mode's row and z' follow from small offsets.  Bound by HBM: read and write
// once.  Against one mode per thread with 64-bit divisions, and sin and pow per
// mode: the TSC window and a derivative at 384^3 in FP64 0.68 -> 0.31 ms (5.9
// TB/s), the CIC window at 512^3 in FP32 1.19 -> 0.28 ms; a spectrum at 512^3 in
// FP64 1.6 -> 0.75 ms, bound by the scattered reads of its table.
// Below 2^21 modes a thread takes one (K = 1), as four leave too few waves (a
// derivative, call and wait: 32^3 17.5 -> 16.6 us, 128^3 22.6 -> 22.1 us).
constexpr int kApplyModes = 4;
constexpr long kApplySmall = 1L << 21;

// small / d for 0 <= small < 2^20, d >= 2
__device__ __forceinline__ int small_div(int small, int d, float inv) {
    int q = (int)((float)small * inv);
    const int r = small - q * d;
    return r < 0 ? q - 1 : (r >= d ? q + 1 : q);
}

// The block's modes of nx x-slabs from x0: load(id) of all of a thread's first
// (dense offsets; a store to w may alias a later load of r), then f(id, value,
// x, y, z).
template <int K, typename V, typename LOAD, typename F>
__device__ __forceinline__ void for_block_modes(int N, long x0, long nx, LOAD&& load, F&& f) {
    const int H = N / 2 + 1;
    const long n = nx * N * H;
    const long e0 = (long)blockIdx.x * (256 * K);
    V v[K];
#pragma unroll
    for (int j = 0; j < K; j++) {
        const long e = e0 + threadIdx.x + 256 * j;
        if (e < n) v[j] = load(e);
    }
    const long row0 = e0 / H;
    const int z0 = (int)(e0 - row0 * H);
    const long xs = row0 / N;
    const int y0 = (int)(row0 - xs * N);
    const float invH = 1.0f / H, invN = 1.0f / N;
#pragma unroll
    for (int j = 0; j < K; j++) {
        const int t = (int)threadIdx.x + 256 * j;
        if (e0 + t >= n) continue;
        const int dr = small_div(z0 + t, H, invH);
        const int z = z0 + t - dr * H;
        const int dx = small_div(y0 + dr, N, invN);
        f(e0 + t, v[j], (int)(x0 + xs) + dx, y0 + dr - dx * N, z);
    }
}

// How the value of a mode is found: directly from the kernel's formula, or from
// a table made by a small launch before.
//   APPLY_DIRECT   ksp_value
//   APPLY_WINDOW   the window kernel: tab[i] = sinc of axis index i, the factors
//                  of ksp_value with the same bits; the squares and cubes of the
//                  CIC and TSC windows are products
//   APPLY_RADIAL   a kernel of |k| alone: tab[n^2], n^2 = |k|^2 / dk^2
//   APPLY_TRANSFER transfer_value, DC ignored
enum { APPLY_DIRECT = 0, APPLY_WINDOW = 1, APPLY_RADIAL = 2, APPLY_TRANSFER = 3 };

// TW/TR may be float (the _float variants compute the product in double, as C
// does for fftwf_complex * double complex).  r is dense, w has rows of whs.
template <typename TW, typename TR, int HOW, int K>
__global__ void __launch_bounds__(256)
    k_apply_kernel(cx<TW>* w, long whs, const cx<TR>* r, int N, long x0, long nx, double boxlen,
                   KSpec ks, const double* __restrict__ tab, TransferTab t) {
#pragma clang fp contract(off)
    const double dk = 2 * M_PI / boxlen;
    auto load = [&](long id) { return ld(r + id); };
    for_block_modes<K, cx<TR>>(N, x0, nx, load, [&](long id, cx<TR> a, int x, int y, int z) {
        cx<double> kv;
        if constexpr (HOW == APPLY_DIRECT) {
            double kx, ky, kz, k;
            wavevec(x, y, z, N, dk, kx, ky, kz, k);
            kv = ksp_value(ks, kx, ky, kz, k);
        } else if constexpr (HOW == APPLY_TRANSFER) {
            double kx, ky, kz, k;
            wavevec(x, y, z, N, dk, kx, ky, kz, k);
            kv = mk<double>(k == 0 ? 0.0 : transfer_value(t, k), 0);
        } else if constexpr (HOW == APPLY_WINDOW) {
            const double W = tab[x] * tab[y] * tab[z];
            const double p = ks.p[0] == 2.0   ? W * W
                             : ks.p[0] == 3.0 ? W * W * W
                                              : pow(W, ks.p[0]);
            kv = mk<double>((x | y | z) == 0 ? 1.0 : 1.0 / p, 0);
        } else {
            const int nx_ = freq_index(x, N), ny = freq_index(y, N);
            kv = mk<double>(tab[(long)nx_ * nx_ + (long)ny * ny + (long)z * z], 0);
        }
        const double re = (double)a.re, im = (double)a.im;
        st(w + (((long)x - x0) * N + y) * whs + z,
           mk<TW>((TW)(re * kv.re - im * kv.im), (TW)(re * kv.im + im * kv.re)));
    });
}

// sinc factors of the window kernel per axis index
static __global__ void k_window_factors(KSpec ks, int N, double boxlen, double* tab) {
#pragma clang fp contract(off)
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= N) return;
    const double dk = 2 * M_PI / boxlen;
    const double k = (i > N / 2) ? (i - N) * dk : i * dk;
    tab[i] = sinc_d(0.5 * k * ks.p[2] / ks.p[1]);
}

// values of a radial kernel over n^2
static __global__ void k_radial_values(KSpec ks, long n, double boxlen, double* tab) {
#pragma clang fp contract(off)
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const double dk = 2 * M_PI / boxlen;
    tab[i] = ksp_value(ks, 0, 0, 0, sqrt((double)i) * dk).re;
}

// r2c operator: normalisation, then the Poisson kernel -1/k^2 (1 at k = 0)
struct OpScalePoisson {
    int N;
    double s, dk;
    __device__ __forceinline__ cx<double> pre(cx<double> v, int, int, int) const { return v; }
    __device__ __forceinline__ cx<double> post(cx<double> v, int x, int y, int z) const {
        const double kx = freq_index(x, N) * dk, ky = freq_index(y, N) * dk, kz = z * dk;
        const double k2 = kx * kx + ky * ky + kz * kz;
        return cscale(v, k2 > 0 ? -s / k2 : s);
    }
};

// write = read * m over nx x-slabs, m the kernel values evaluated on the host
// (dense N x N x (N/2+1) per slab)
template <typename TW, typename TR>
__global__ void k_apply_mult(cx<TW>* w, const cx<TR>* r, const cx<double>* __restrict__ m,
                             int N, long hs, long nx) {
#pragma clang fp contract(off)
    const long H = N / 2 + 1;
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= nx * N * H) return;
    const long z = i % H;
    const long xy = i / H;
    const long id = xy * hs + z;
    const cx<TR> a = r[id];
    const cx<double> kv = m[i];
    const double re = (double)a.re, im = (double)a.im;
    w[id] = mk<TW>((TW)(re * kv.re - im * kv.im), (TW)(re * kv.im + im * kv.re));
}

// elementwise complex scaling (normalisations)
template <typename T>
__global__ void k_scale_complex(cx<T>* a, long n, double s) {
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    cx<T> v = a[i];
    a[i] = mk<T>((T)((double)v.re * s), (T)((double)v.im * s));
}

template <typename T>
__global__ void k_div_real(T* a, long n, double d) {
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    a[i] = (T)((double)a[i] / d);
}

}  // namespace mitos
