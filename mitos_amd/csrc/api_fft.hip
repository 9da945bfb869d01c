// Drop-in FFT, k-space kernel, Poisson and 2LPT entry points
// (include/fft.h:90-116, include/fft_kernels.h, include/poisson.h:29-30,
//  include/2lpt.h:27-29, include/grids_interp.h:41-48).
#include <string.h>

#include <algorithm>
#include <thread>
#include <vector>

#include "../../include/mitos_hip.h"
#include "dropin.h"
#include "kspace.h"

using namespace mitos;

namespace {

inline long half_elems(int N) { return (long)N * N * (N / 2 + 1); }

inline double* kern_parts(struct kernel* k) { return reinterpret_cast<double*>(&k->kern); }

inline unsigned nblk(long n, int b = 256) { return (unsigned)((n + b - 1) / b); }

// Map a reference kernel callback to its device kernel.
int kspec_from_callback(void (*compute)(struct kernel*), const void* params, int N,
                        double boxlen, KSpec* ks) {
    memset(ks, 0, sizeof(*ks));
    (void)N;
    (void)boxlen;
    if (compute == kernel_constant) {
        if (!params) return MITOS_ERR_ARG;
        ks->id = KID_CONSTANT;
        ks->p[0] = *(const double*)params;
    } else if (compute == kernel_inv_poisson) {
        ks->id = KID_INV_POISSON;
    } else if (compute == kernel_dx) {
        ks->id = KID_DX;
    } else if (compute == kernel_dy) {
        ks->id = KID_DY;
    } else if (compute == kernel_dz) {
        ks->id = KID_DZ;
    } else if (compute == kernel_power_no_transfer) {
        if (!params) return MITOS_ERR_ARG;
        const struct cosmology* c = (const struct cosmology*)params;
        ks->id = KID_POWER_NO_TRANSFER;
        ks->p[0] = c->A_s;
        ks->p[1] = c->n_s;
        ks->p[2] = c->k_pivot;
    } else if (compute == kernel_undo_Hermite_window) {
        if (!params) return MITOS_ERR_ARG;
        const struct Hermite_kern_params* h = (const struct Hermite_kern_params*)params;
        ks->id = KID_UNDO_WINDOW;
        ks->p[0] = h->order;
        ks->p[1] = h->N;
        ks->p[2] = h->boxlen;
    } else if (compute == kernel_sqrt_power_law) {
        if (!params) return MITOS_ERR_ARG;
        const struct mitos_spectrum_params* p = (const struct mitos_spectrum_params*)params;
        ks->id = KID_SQRT_POWER_LAW;
        ks->p[0] = p->A;
        ks->p[1] = p->n_s;
    } else if (compute == kernel_bbks_transfer) {
        if (!params) return MITOS_ERR_ARG;
        const struct mitos_spectrum_params* p = (const struct mitos_spectrum_params*)params;
        ks->id = KID_BBKS;
        ks->p[0] = p->Gamma;
    } else if (compute == kernel_lowpass || compute == kernel_hipass ||
               compute == kernel_gaussian || compute == kernel_gaussian_inv) {
        if (!params) return MITOS_ERR_ARG;
        ks->id = compute == kernel_lowpass   ? KID_LOWPASS
                 : compute == kernel_hipass  ? KID_HIPASS
                 : compute == kernel_gaussian ? KID_GAUSSIAN
                                              : KID_GAUSSIAN_INV;
        ks->p[0] = *(const double*)params;
    } else if (compute == kernel_tophat) {
        if (!params) return MITOS_ERR_ARG;
        ks->id = KID_TOPHAT;
        memcpy(ks->p, params, 2 * sizeof(double));
    } else if (compute == kernel_elliptic_tophat) {
        if (!params) return MITOS_ERR_ARG;
        ks->id = KID_ELLIPTIC_TOPHAT;
        memcpy(ks->p, params, 4 * sizeof(double));
    } else if (compute == kernel_translate) {
        if (!params) return MITOS_ERR_ARG;
        ks->id = KID_TRANSLATE;
        memcpy(ks->p, params, 3 * sizeof(double));
    } else {
        return MITOS_ERR_UNSUPPORTED;
    }
    return MITOS_OK;
}

template <int HOW, typename TW, typename TR>
int issue_apply(cx<TW>* w, const cx<TR>* r, int N, long x0, long nx, double boxlen,
                 const KSpec& ks, const double* tab, const TransferTab& t = TransferTab{}) {
    const long n = nx * N * (N / 2 + 1);
    if (n <= 0) return MITOS_ERR_DEVICE;  // as a launch of no work-groups fails
    const bool small = n < kApplySmall;
    const auto kern = small ? k_apply_kernel<TW, TR, HOW, 1>
                            : k_apply_kernel<TW, TR, HOW, kApplyModes>;
    const int modes = small ? 256 : 256 * kApplyModes;
    hipLaunchKernelGGL(kern, dim3(nblk(n, modes)), dim3(256), 0, api_stream(), w,
                       (long)(N / 2 + 1), r, N, x0, nx, boxlen, ks, tab, t);
    return launch_status();
}

// kernel_(inv_)transfer_function: the k vector and the selected function's
// two time rows go to the device, the modes are evaluated there
template <typename TW, typename TR>
int apply_transfer(cx<TW>* w, const cx<TR>* r, int N, long x0, long nx, double boxlen,
                   const struct spline_params* sp, int invert) {
    if (!sp || !sp->spline || !sp->spline->ptdat) return MITOS_ERR_ARG;
    const struct perturb_data* pt = sp->spline->ptdat;
    const int ks = pt->k_size, ts = pt->tau_size;
    if (ks < 2 || ts < 2 || !pt->k || !pt->delta || sp->index_src < 0 ||
        sp->index_src >= pt->n_functions || sp->tau_index < 0 || sp->tau_index > ts - 2)
        return MITOS_ERR_ARG;
    {
        ScratchLock hold;
        double* d = (double*)workspace(5, sizeof(double) * 3 * ks);
        if (!d) return MITOS_ERR_ALLOC;
        const double* rows =
            pt->delta + (size_t)sp->index_src * ks * ts + (size_t)ks * sp->tau_index;
        MITOS_HIP_CHECK(copy_sync(d, pt->k, sizeof(double) * ks, hipMemcpyHostToDevice));
        MITOS_HIP_CHECK(copy_sync(d + ks, rows, sizeof(double) * 2 * ks, hipMemcpyHostToDevice));
        TransferTab t{d, d + ks, d + 2 * ks, ks, sp->u_tau, invert};
        MITOS_TRY((issue_apply<APPLY_TRANSFER>(w, r, N, x0, nx, boxlen, KSpec{}, nullptr, t)));
    }
    return api_sync();
}

// Any other callback: evaluated on the host for every mode with the
// reference's protocol (src/fft.c:279-291: {kx, ky, kz, k, 0, params} in,
// kern out), a chunk of x-slabs at a time over host threads (the callback
// runs concurrently, as under the reference's OpenMP loop), copied to the
// device through two pinned buffers, and multiplied in there.
template <typename TW, typename TR>
int apply_kernel_host(cx<TW>* w, const cx<TR>* r, int N, long x0, long nx, double boxlen,
                      void (*compute)(struct kernel*), const void* params) {
    const long H = N / 2 + 1;
    const long plane = (long)N * H;
    const long bytes_slab = plane * (long)sizeof(cx<double>);
    const long per = std::max(1L, (32L << 20) / bytes_slab);  // slabs per chunk
    const size_t cbytes = (size_t)(per * bytes_slab);
    cx<double>* hbuf[2] = {nullptr, nullptr};
    cx<double>* dbuf = (cx<double>*)workspace(4, 2 * cbytes);
    if (!dbuf) return MITOS_ERR_ALLOC;
    hipEvent_t used[2] = {nullptr, nullptr};
    int rc = MITOS_OK;
    for (int b = 0; b < 2 && rc == MITOS_OK; b++) {
        if (hipHostMalloc((void**)&hbuf[b], cbytes, hipHostMallocDefault) != hipSuccess ||
            hipEventCreateWithFlags(&used[b], hipEventDisableTiming) != hipSuccess)
            rc = MITOS_ERR_ALLOC;
    }
    const double dk = 2 * M_PI / boxlen;
    const int nthreads = (int)std::min(16u, std::max(1u, std::thread::hardware_concurrency()));
    for (long c = 0, it = 0; c < nx && rc == MITOS_OK; c += per, it++) {
        const long ns = std::min(per, nx - c);
        const int b = (int)(it & 1);
        if (it >= 2 && hipEventSynchronize(used[b]) != hipSuccess) {
            rc = MITOS_ERR_DEVICE;
            break;
        }
        cx<double>* hb = hbuf[b];
        auto worker = [&](int tid) {
            for (long row = tid; row < ns * N; row += nthreads) {
                const int x = (int)(x0 + c + row / N), y = (int)(row % N);
                for (int z = 0; z < H; z++) {
                    struct kernel kk;
                    wavevec(x, y, z, N, dk, kk.kx, kk.ky, kk.kz, kk.k);
                    double* kp = kern_parts(&kk);
                    kp[0] = 0;
                    kp[1] = 0;
                    kk.params = params;
                    compute(&kk);
                    hb[row * H + z] = mk<double>(kp[0], kp[1]);
                }
            }
        };
        std::vector<std::thread> pool;
        for (int t = 1; t < nthreads; t++) pool.emplace_back(worker, t);
        worker(0);
        for (auto& th : pool) th.join();
        cx<double>* db = dbuf + (size_t)b * per * plane;
        if (hipMemcpyAsync(db, hb, (size_t)(ns * bytes_slab), hipMemcpyHostToDevice,
                           api_stream()) != hipSuccess) {
            rc = MITOS_ERR_DEVICE;
            break;
        }
        const long off = c * N * H;
        hipLaunchKernelGGL((k_apply_mult<TW, TR>), dim3(nblk(ns * plane)), dim3(256), 0,
                           api_stream(), w + off, r + off, db, N, H, ns);
        rc = launch_status();
        if (rc == MITOS_OK && hipEventRecord(used[b], api_stream()) != hipSuccess)
            rc = MITOS_ERR_DEVICE;
    }
    if (rc == MITOS_OK) rc = api_sync();
    else (void)api_sync();
    for (int b = 0; b < 2; b++) {
        if (hbuf[b]) hipHostFree(hbuf[b]);
        if (used[b]) hipEventDestroy(used[b]);
    }
    return rc;
}

// a kernel with a device form, issued on the library stream
template <typename TW, typename TR>
int device_apply(cx<TW>* w, const cx<TR>* r, int N, long x0, long nx, double boxlen,
                 const KSpec& ks) {
    // Tables of a window's N factors, and of the spectra's powers and logarithms over
    // n^2: a launch more, so where there are enough modes, for the spectra also enough
    // per entry (a slab has few).  Direct against table, call and wait: window 64^3 (2^17
    // modes) 19.6, 19.8 us, 128^3 (2^20) 38, 24 us; power law 64^3 18.5, 20.8 us, 128^3
    // 30, 25 us; of 1024^3 in FP32 four planes (2.7 modes an entry) power law 39, 42 us,
    // BBKS 70, 54 us, sixteen planes 100, 77 us and 220, 89 us.  Where no scratch can be
    // had they are evaluated directly as well.
    ScratchLock hold;
    const long n = nx * N * (N / 2 + 1), n2 = 3L * (N / 2) * (N / 2) + 1;
    if (ks.id == KID_UNDO_WINDOW && n >= (1L << 18)) {
        if (double* tab = (double*)workspace(SLOT_APPLY_TABLE, sizeof(double) * N)) {
            hipLaunchKernelGGL(k_window_factors, dim3(nblk(N)), dim3(256), 0, api_stream(), ks,
                               N, boxlen, tab);
            return issue_apply<APPLY_WINDOW>(w, r, N, x0, nx, boxlen, ks, tab);
        }
    }
    if ((ks.id == KID_POWER_NO_TRANSFER || ks.id == KID_SQRT_POWER_LAW || ks.id == KID_BBKS) &&
        n >= (1L << 19) && n >= (ks.id == KID_BBKS ? 2 : 8) * n2) {
        if (double* tab = (double*)workspace(SLOT_APPLY_TABLE, sizeof(double) * n2)) {
            hipLaunchKernelGGL(k_radial_values, dim3(nblk(n2)), dim3(256), 0, api_stream(), ks,
                               n2, boxlen, tab);
            return issue_apply<APPLY_RADIAL>(w, r, N, x0, nx, boxlen, ks, tab);
        }
    }
    return issue_apply<APPLY_DIRECT>(w, r, N, x0, nx, boxlen, ks, nullptr);
}

template <typename TW, typename TR>
int apply_kernel(cx<TW>* w, const cx<TR>* r, int N, long x0, long nx, double boxlen,
                 void (*compute)(struct kernel*), const void* params) {
    if (!w || !r || N < 2 || !compute) return MITOS_ERR_ARG;
    if (compute == kernel_transfer_function || compute == kernel_inv_transfer_function)
        return apply_transfer<TW, TR>(w, r, N, x0, nx, boxlen,
                                      (const struct spline_params*)params,
                                      compute == kernel_inv_transfer_function);
    KSpec ks;
    const int kr = kspec_from_callback(compute, params, N, boxlen, &ks);
    if (kr == MITOS_ERR_UNSUPPORTED)
        return apply_kernel_host<TW, TR>(w, r, N, x0, nx, boxlen, compute, params);
    MITOS_TRY(kr);
    MITOS_TRY((device_apply<TW, TR>(w, r, N, x0, nx, boxlen, ks)));
    return api_sync();
}

template <typename T>
int scale_complex(cx<T>* a, long n, double s) {
    if (!a) return MITOS_ERR_ARG;
    hipLaunchKernelGGL((k_scale_complex<T>), dim3(nblk(n)), dim3(256), 0, api_stream(), a, n, s);
    MITOS_TRY(launch_status());
    return api_sync();
}

// Work grids of a transform and their row stride: whole lines, dense rows where only
// those fit.  Two up to 32 MB each (128^3), else one used twice (see c2r_3d).
template <typename T>
bool work_grids(int N, cx<T>** w1, cx<T>** w2, long* hs) {
    const size_t bytes = work_grid_bytes<T>(N), second = bytes <= (32u << 20) ? bytes : 0;
    *hs = work_row<T>(N);
    *w1 = (cx<T>*)workspace(SLOT_FFT, bytes + second);
    if (*w1) {
        *w2 = *w1 + second / sizeof(cx<T>);
        return true;
    }
    *hs = N / 2 + 1;
    *w1 = *w2 = (cx<T>*)workspace(SLOT_FFT, sizeof(cx<T>) * half_elems(N));
    return *w1 != nullptr;
}

// r2c of an N^3 array with row stride rs into the (N, N, N/2+1) layout, times
// scale, issued on the library stream; in place in the output where no work grid fits
template <typename T, typename OPX>
int r2c_issue(int N, const T* in, long rs, cx<T>* out, OPX ox) {
    if (!in || !out) return MITOS_ERR_ARG;
    if (!size_supported(N)) return MITOS_ERR_UNSUPPORTED;
    ScratchLock hold;
    cx<T>*w1, *w2;
    long hs;
    if (!work_grids(N, &w1, &w2, &hs)) w1 = w2 = out;
    RealRowLoader<T> ld{in, rs, 0};
    return r2c_3d<T>(N, ld, w1, w2, hs, out, N / 2 + 1, ox, api_stream());
}

template <typename T>
int c2r_issue(int N, const cx<T>* in, T* out, long rs, double scale) {
    if (!in || !out) return MITOS_ERR_ARG;
    if (!size_supported(N)) return MITOS_ERR_UNSUPPORTED;
    ScratchLock hold;
    cx<T>*w1, *w2;
    long hs;
    if (!work_grids(N, &w1, &w2, &hs)) return MITOS_ERR_ALLOC;
    return c2r_3d<T>(N, in, N / 2 + 1, w1, w2, hs, out, rs, (T)scale, OpNone(), api_stream());
}

// unnormalised r2c of an N^3 array with row stride rs into the (N, N, N/2+1) layout
template <typename T>
int r2c_plain(int N, const T* in, long rs, cx<T>* out) {
    MITOS_TRY((r2c_issue<T>(N, in, rs, out, OpNone())));
    return api_sync();
}

template <typename T>
int c2r_plain(int N, const cx<T>* in, T* out, long rs, double scale) {
    MITOS_TRY(c2r_issue<T>(N, in, out, rs, scale));
    return api_sync();
}

}  // namespace

// ---- kernel callbacks (host evaluation; addresses select device kernels) ----------
extern "C" void kernel_constant(struct kernel* the_kernel) {
    double* k = kern_parts(the_kernel);
    k[0] = *((const double*)the_kernel->params);
    k[1] = 0;
}
extern "C" void kernel_inv_poisson(struct kernel* the_kernel) {
    double* k = kern_parts(the_kernel);
    const double kk = the_kernel->k;
    k[0] = (kk > 0) ? -1.0 / kk / kk : 1.0;
    k[1] = 0;
}
extern "C" void kernel_dx(struct kernel* the_kernel) {
    double* k = kern_parts(the_kernel);
    k[0] = 0;
    k[1] = the_kernel->kx;
}
extern "C" void kernel_dy(struct kernel* the_kernel) {
    double* k = kern_parts(the_kernel);
    k[0] = 0;
    k[1] = the_kernel->ky;
}
extern "C" void kernel_dz(struct kernel* the_kernel) {
    double* k = kern_parts(the_kernel);
    k[0] = 0;
    k[1] = the_kernel->kz;
}
extern "C" void kernel_power_no_transfer(struct kernel* the_kernel) {
    KSpec ks;
    kspec_from_callback(kernel_power_no_transfer, the_kernel->params, 0, 0, &ks);
    cx<double> v = ksp_value(ks, the_kernel->kx, the_kernel->ky, the_kernel->kz, the_kernel->k);
    double* k = kern_parts(the_kernel);
    k[0] = v.re;
    k[1] = v.im;
}
extern "C" void kernel_undo_Hermite_window(struct kernel* the_kernel) {
    KSpec ks;
    kspec_from_callback(kernel_undo_Hermite_window, the_kernel->params, 0, 0, &ks);
    cx<double> v = ksp_value(ks, the_kernel->kx, the_kernel->ky, the_kernel->kz, the_kernel->k);
    double* k = kern_parts(the_kernel);
    k[0] = v.re;
    k[1] = v.im;
}
extern "C" void kernel_sqrt_power_law(struct kernel* the_kernel) {
    KSpec ks;
    kspec_from_callback(kernel_sqrt_power_law, the_kernel->params, 0, 0, &ks);
    cx<double> v = ksp_value(ks, the_kernel->kx, the_kernel->ky, the_kernel->kz, the_kernel->k);
    double* k = kern_parts(the_kernel);
    k[0] = v.re;
    k[1] = v.im;
}
extern "C" void kernel_bbks_transfer(struct kernel* the_kernel) {
    KSpec ks;
    kspec_from_callback(kernel_bbks_transfer, the_kernel->params, 0, 0, &ks);
    cx<double> v = ksp_value(ks, the_kernel->kx, the_kernel->ky, the_kernel->kz, the_kernel->k);
    double* k = kern_parts(the_kernel);
    k[0] = v.re;
    k[1] = v.im;
}

// host evaluation of a parameterised callback through its device formula
static void host_value(void (*self)(struct kernel*), struct kernel* the_kernel) {
    KSpec ks;
    kspec_from_callback(self, the_kernel->params, 0, 0, &ks);
    cx<double> v = ksp_value(ks, the_kernel->kx, the_kernel->ky, the_kernel->kz, the_kernel->k);
    double* k = kern_parts(the_kernel);
    k[0] = v.re;
    k[1] = v.im;
}
extern "C" void kernel_lowpass(struct kernel* the_kernel) { host_value(kernel_lowpass, the_kernel); }
extern "C" void kernel_hipass(struct kernel* the_kernel) { host_value(kernel_hipass, the_kernel); }
extern "C" void kernel_tophat(struct kernel* the_kernel) { host_value(kernel_tophat, the_kernel); }
extern "C" void kernel_elliptic_tophat(struct kernel* the_kernel) {
    host_value(kernel_elliptic_tophat, the_kernel);
}
extern "C" void kernel_translate(struct kernel* the_kernel) {
    host_value(kernel_translate, the_kernel);
}
extern "C" void kernel_gaussian(struct kernel* the_kernel) {
    host_value(kernel_gaussian, the_kernel);
}
extern "C" void kernel_gaussian_inv(struct kernel* the_kernel) {
    host_value(kernel_gaussian_inv, the_kernel);
}

// ---- FFTs on distributed grids (src/fft.c:219-254) ---------------------------------
extern "C" int fft_r2c_dg(struct distributed_grid* dg) {
    MITOS_TRY(set_last_error(dg_r2c_issue(dg, false)));
    return set_last_error(api_sync());
}

extern "C" int fft_c2r_dg(struct distributed_grid* dg) {
    MITOS_TRY(set_last_error(dg_c2r_issue(dg)));
    return set_last_error(api_sync());
}

extern "C" int fft_apply_kernel_dg(struct distributed_grid* dg_write,
                                   const struct distributed_grid* dg_read,
                                   void (*compute)(struct kernel* the_kernel),
                                   const void* params) {
    if (!dg_write || !dg_read) return set_last_error(MITOS_ERR_ARG);
    if (dg_read->NX != dg_write->NX || dg_read->N != dg_write->N)
        return set_last_error(MITOS_ERR_DIMS);
    if (dg_read->momentum_space != 1) return set_last_error(MITOS_ERR_NOT_MOMENTUM);
    MITOS_TRY(set_last_error(apply_kernel<double, double>(
        reinterpret_cast<cx<double>*>(dg_write->fbox),
        reinterpret_cast<const cx<double>*>(dg_read->fbox), dg_read->N, dg_read->X0,
        dg_read->NX, dg_read->boxlen, compute, params)));
    dg_write->momentum_space = 1;
    return MITOS_OK;
}

// ---- serial-array variants (src/fft.c:38-216) ----------------------------------------
extern "C" int fft_normalize_r2c(fftw_complex* arr, int N, double boxlen) {
    const double boxvol = boxlen * boxlen * boxlen;
    return set_last_error(scale_complex<double>(reinterpret_cast<cx<double>*>(arr),
                                                half_elems(N),
                                                boxvol / ((long long)N * N * N)));
}
extern "C" int fft_normalize_r2c_float(fftwf_complex* arr, int N, double boxlen) {
    const double boxvol = boxlen * boxlen * boxlen;
    return set_last_error(scale_complex<float>(reinterpret_cast<cx<float>*>(arr), half_elems(N),
                                               boxvol / ((long long)N * N * N)));
}
extern "C" int fft_normalize_r2c_float_mpi(fftwf_complex* farr, long int N, long int local_size,
                                           double boxlen) {
    const double boxvol = boxlen * boxlen * boxlen;
    return set_last_error(scale_complex<float>(reinterpret_cast<cx<float>*>(farr), local_size,
                                               boxvol / ((long long)N * N * N)));
}
extern "C" int fft_normalize_c2r(double* arr, int N, double boxlen) {
    if (!arr) return set_last_error(MITOS_ERR_ARG);
    const long n = (long)N * N * N;
    hipLaunchKernelGGL((k_div_real<double>), dim3(nblk(n)), dim3(256), 0, api_stream(), arr, n,
                       boxlen * boxlen * boxlen);
    MITOS_TRY(set_last_error(launch_status()));
    return set_last_error(api_sync());
}
extern "C" int fft_apply_kernel(fftw_complex* write, const fftw_complex* read, int N,
                                double boxlen, void (*compute)(struct kernel*),
                                const void* params) {
    return set_last_error(apply_kernel<double, double>(
        reinterpret_cast<cx<double>*>(write), reinterpret_cast<const cx<double>*>(read), N, 0,
        N, boxlen, compute, params));
}
extern "C" int fft_apply_kernel_float(fftwf_complex* write, const fftwf_complex* read, int N,
                                      double boxlen, void (*compute)(struct kernel*),
                                      const void* params) {
    return set_last_error(apply_kernel<float, float>(
        reinterpret_cast<cx<float>*>(write), reinterpret_cast<const cx<float>*>(read), N, 0, N,
        boxlen, compute, params));
}
extern "C" int fft_apply_kernel_float_mpi(fftwf_complex* write, const fftwf_complex* read,
                                          long int N, long int X0, long int NX, double boxlen,
                                          void (*compute)(struct kernel*),
                                          const void* params) {
    return set_last_error(apply_kernel<float, float>(
        reinterpret_cast<cx<float>*>(write), reinterpret_cast<const cx<float>*>(read), (int)N,
        X0, NX, boxlen, compute, params));
}

// ---- window functions (src/grids_interp.c:374-399, 430-455) ---------------------------
static int undo_window(void* farr, int N, double boxlen, int order, bool fp32) {
    struct Hermite_kern_params h;
    h.order = order;
    h.N = N;
    h.boxlen = boxlen;
    if (fp32)
        return apply_kernel<float, float>(reinterpret_cast<cx<float>*>(farr),
                                          reinterpret_cast<const cx<float>*>(farr), N, 0, N,
                                          boxlen, kernel_undo_Hermite_window, &h);
    return apply_kernel<double, double>(reinterpret_cast<cx<double>*>(farr),
                                        reinterpret_cast<const cx<double>*>(farr), N, 0, N,
                                        boxlen, kernel_undo_Hermite_window, &h);
}
extern "C" int undoCICWindow(fftw_complex* farr, int N, double boxlen) {
    return set_last_error(undo_window(farr, N, boxlen, 2, false));
}
extern "C" int undoTSCWindow(fftw_complex* farr, int N, double boxlen) {
    return set_last_error(undo_window(farr, N, boxlen, 3, false));
}
extern "C" int undoCICWindowFloat(fftwf_complex* farr, int N, double boxlen) {
    return set_last_error(undo_window(farr, N, boxlen, 2, true));
}
extern "C" int undoTSCWindowFloat(fftwf_complex* farr, int N, double boxlen) {
    return set_last_error(undo_window(farr, N, boxlen, 3, true));
}

// ---- FFTW-plan equivalents on unpadded arrays -------------------------------------------
extern "C" int mitos_fft_r2c(int N, const double* in, fftw_complex* out) {
    return set_last_error(r2c_plain<double>(N, in, N, reinterpret_cast<cx<double>*>(out)));
}
extern "C" int mitos_fft_c2r(int N, const fftw_complex* in, double* out) {
    return set_last_error(
        c2r_plain<double>(N, reinterpret_cast<const cx<double>*>(in), out, N, 1.0));
}
extern "C" int mitos_fft_r2c_float(int N, const float* in, fftwf_complex* out) {
    return set_last_error(r2c_plain<float>(N, in, N, reinterpret_cast<cx<float>*>(out)));
}
extern "C" int mitos_fft_c2r_float(int N, const fftwf_complex* in, float* out) {
    return set_last_error(
        c2r_plain<float>(N, reinterpret_cast<const cx<float>*>(in), out, N, 1.0));
}

// ---- Poisson (src/poisson.c:29-70) --------------------------------------------------------
namespace mitos {

// r2c with its normalisation and, when asked, the Poisson kernel on the stored
// modes (include/fft_kernels.h:96-99)
int dg_r2c_issue(struct distributed_grid* dg, bool poisson) {
    if (!dg || !dg->box || !dg->fbox) return MITOS_ERR_ARG;
    const int N = dg->N;
    const double s = dg->boxlen * dg->boxlen * dg->boxlen / ((long long)N * N * N);
    cx<double>* out = reinterpret_cast<cx<double>*>(dg->fbox);
    if (poisson)
        MITOS_TRY((r2c_issue<double>(N, dg->box, N + 2, out,
                                     OpScalePoisson{N, s, 2 * M_PI / dg->boxlen})));
    else
        MITOS_TRY((r2c_issue<double>(N, dg->box, N + 2, out, OpScale<double>{s})));
    dg->momentum_space = 1;
    return MITOS_OK;
}

int dg_c2r_issue(struct distributed_grid* dg) {
    if (!dg || !dg->box || !dg->fbox) return MITOS_ERR_ARG;
    const double boxvol = dg->boxlen * dg->boxlen * dg->boxlen;
    MITOS_TRY(c2r_issue<double>(dg->N, reinterpret_cast<const cx<double>*>(dg->fbox), dg->box,
                                dg->N + 2, 1.0 / boxvol));
    dg->momentum_space = 0;
    return MITOS_OK;
}

int apply_padded_issue(cx<double>* w, long whs, const struct distributed_grid* dg,
                       const KSpec& ks) {
    const int N = dg->N;
    const long n = (long)N * N * (N / 2 + 1);
    hipLaunchKernelGGL((k_apply_kernel<double, double, APPLY_DIRECT, kApplyModes>),
                       dim3(nblk(n, 256 * kApplyModes)), dim3(256), 0, api_stream(), w, whs,
                       reinterpret_cast<const cx<double>*>(dg->fbox), N, 0L, (long)N, dg->boxlen,
                       ks, (const double*)nullptr, TransferTab{});
    return launch_status();
}

}  // namespace mitos

extern "C" int solvePoisson_dg(struct distributed_grid* dg) {
    MITOS_TRY(set_last_error(dg_r2c_issue(dg, true)));
    MITOS_TRY(set_last_error(dg_c2r_issue(dg)));
    return set_last_error(api_sync());
}

extern "C" int solvePoisson(double* phi, double* f, int N, double boxlen) {
    if (!phi || !f) return set_last_error(MITOS_ERR_ARG);
    {
        ScratchLock hold;
        cx<double>* fbox = (cx<double>*)workspace(1, sizeof(cx<double>) * half_elems(N));
        if (!fbox) return set_last_error(MITOS_ERR_ALLOC);
        const double boxvol = boxlen * boxlen * boxlen;
        const double s = boxvol / ((long long)N * N * N);
        MITOS_TRY(set_last_error(
            (r2c_issue<double>(N, f, N, fbox, OpScalePoisson{N, s, 2 * M_PI / boxlen}))));
        MITOS_TRY(set_last_error((c2r_issue<double>(N, fbox, phi, N, 1.0 / boxvol))));
    }
    return set_last_error(api_sync());
}
