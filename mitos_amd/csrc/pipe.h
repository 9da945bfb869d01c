// The fused IC pipeline (struct Pipe) and its host-side tables, shared by the
// single-realization API (pipeline.hip) and the ensemble API (ensemble.hip).
#pragma once

#include <math.h>
#include <string.h>

#include <map>
#include <mutex>
#include <tuple>
#include <type_traits>
#include <vector>

#include "../../include/mitos_hip.h"
#include "cic_sort.h"
#include "pipeline_kernels.h"
#include "powerspec.h"

namespace mitos {


// ---- spectrum ------------------------------------------------------------------------
// A of P = A k^n_s T_BBKS^2 for sigma_R = sigma8 (sigma8.cpp)
double sigma8_amplitude(double n_s, double gamma, double sigma8, double R);

// Host: device table w[i] = 1/sinc(0.5 k_i boxlen/N)^order for i in [0, N),
// k_i = freq_index(i)*2pi/boxlen.  The window of include/fft_kernels.h:198-219
// is separable, 1/W(k) = w[x] w[y] w[z] (k != 0).  Cached per (N, boxlen, order).
inline const double* window_table(int N, double boxlen, int order) {
    static std::mutex mu;
    static std::map<std::tuple<int, int, double, int>, double*> cache;
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) return nullptr;
    auto key = std::make_tuple(dev, N, boxlen, order);
    std::lock_guard<std::mutex> lock(mu);
    auto it = cache.find(key);
    if (it != cache.end()) return it->second;
    std::vector<double> h(N);
    const double dk = 2 * M_PI / boxlen;
    for (int i = 0; i < N; i++) {
        const double k = freq_index(i, N) * dk;
        const double w = sinc_d(0.5 * k * boxlen / N);
        h[i] = 1.0 / pow(w, order);
    }
    double* d = nullptr;
    if (hipMalloc(&d, sizeof(double) * N) != hipSuccess) return nullptr;
    if (copy_sync(d, h.data(), sizeof(double) * N, hipMemcpyHostToDevice) != hipSuccess) {
        hipFree(d);
        return nullptr;
    }
    cache[key] = d;
    return d;
}

// Device table S[n] = 3/4 + cos(2 pi n/N)/4, n in [0, N): the DFT of the
// periodic lattice stencil (1/8, 3/4, 1/8).  Cached per (device, N, type).
template <typename V>
inline const V* smooth_table(int N) {
    static std::mutex mu;
    static std::map<std::pair<int, int>, V*> cache;
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) return nullptr;
    auto key = std::make_pair(dev, N);
    std::lock_guard<std::mutex> lock(mu);
    auto it = cache.find(key);
    if (it != cache.end()) return it->second;
    std::vector<V> h(N);
    for (int n = 0; n < N; n++) {
        // exact values at the quarter points
        double c;
        if (4 * n == N || 4 * n == 3 * N) c = 0.0;
        else if (2 * n == N) c = -1.0;
        else c = cos(2.0 * M_PI * n / N);
        h[n] = (V)(0.75 + 0.25 * c);
    }
    V* d = nullptr;
    if (hipMalloc(&d, sizeof(V) * N) != hipSuccess) return nullptr;
    if (copy_sync(d, h.data(), sizeof(V) * N, hipMemcpyHostToDevice) != hipSuccess) {
        hipFree(d);
        return nullptr;
    }
    cache[key] = d;
    return d;
}

// True when every lattice coordinate q*((float)L/N) (float, src/particle.c:
// 102-109) sits exactly on grid node q in the reference's cell units
// (double x*N/boxlen, src/grids_interp.c:269-271).  Then the TSC window of an
// unmoved coordinate is exactly (1/8, 3/4, 1/8) and the lattice stencils
// reproduce gridTSC_dg; otherwise (e.g. 2000 Mpc/h over 1536 cells, a spacing
// float rounds) the moves gather 27 taps at the actual positions.
inline bool lattice_on_nodes(int N, double L) {
    const float spacing = (float)L / N;
    for (int q = 0; q < N; q++) {
        const float x = (float)q * spacing;
        if ((double)x * N / L != (double)q) return false;
    }
    return true;
}

inline double amplitude_cached(double n_s, double gamma, double sigma8) {
    static std::mutex mu;
    static std::map<std::tuple<double, double, double>, double> cache;
    auto key = std::make_tuple(n_s, gamma, sigma8);
    std::lock_guard<std::mutex> lock(mu);
    auto it = cache.find(key);
    if (it != cache.end()) return it->second;
    const double A = sigma8_amplitude(n_s, gamma, sigma8, 8.0);
    cache[key] = A;
    return A;
}

// Device table over the integer n^2 = |k|^2/dk^2 of the amplitude taking white
// noise to phi1(k) = -delta(k)/k^2, delta = noise * sqrt(A k^n_s) T_BBKS(k)
// (the primordial kernel of src/mitos.c:224, the transfer kernel of
// src/generate_grids.c:52 and kernel_inv_poisson of src/2lpt.c:75).
inline std::vector<double> phi1_host(int N, double boxlen, double A, double n_s, double gamma) {
    const long n2max = 3L * (N / 2) * (N / 2);
    std::vector<double> h(n2max + 1);
    const double dk = 2 * M_PI / boxlen;
    h[0] = 0.0;
    for (long n2 = 1; n2 <= n2max; n2++) {
        const double k = sqrt((double)n2) * dk;
        const double p = sqrt(A * pow(k, n_s));
        const double t = bbks_T(k, gamma);
        h[n2] = (p * t) * (-1.0 / k / k);
    }
    return h;
}

inline const double* phi1_table(int N, double boxlen, double A, double n_s, double gamma) {
    static std::mutex mu;
    static std::map<std::tuple<int, int, double, double, double, double>, double*> cache;
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) return nullptr;
    auto key = std::make_tuple(dev, N, boxlen, A, n_s, gamma);
    std::lock_guard<std::mutex> lock(mu);
    auto it = cache.find(key);
    if (it != cache.end()) return it->second;
    if (cache.size() > 64) {  // bounded: one entry per (size, spectrum)
        hipDeviceSynchronize();
        for (auto& kv : cache) hipFree(kv.second);
        cache.clear();
    }
    const std::vector<double> h = phi1_host(N, boxlen, A, n_s, gamma);
    double* d = nullptr;
    if (hipMalloc(&d, sizeof(double) * h.size()) != hipSuccess) return nullptr;
    if (copy_sync(d, h.data(), sizeof(double) * h.size(), hipMemcpyHostToDevice) !=
        hipSuccess) {
        hipFree(d);
        return nullptr;
    }
    cache[key] = d;
    return d;
}

// The table of phi1_table times the noise factor sqrt(L^3/2) of k_grf (the
// same double expression), rounded to float: the FP32 noise kernel's values
inline const float* phi1_table_f(int N, double boxlen, double A, double n_s, double gamma) {
    static std::mutex mu;
    static std::map<std::tuple<int, int, double, double, double, double>, float*> cache;
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) return nullptr;
    auto key = std::make_tuple(dev, N, boxlen, A, n_s, gamma);
    std::lock_guard<std::mutex> lock(mu);
    auto it = cache.find(key);
    if (it != cache.end()) return it->second;
    if (cache.size() > 64) {
        hipDeviceSynchronize();
        for (auto& kv : cache) hipFree(kv.second);
        cache.clear();
    }
    const std::vector<double> h = phi1_host(N, boxlen, A, n_s, gamma);
    const double boxvol = boxlen * boxlen * boxlen;
    const double factor = sqrt(boxvol / 2);
    std::vector<float> f(h.size());
    for (size_t i = 0; i < h.size(); i++) f[i] = (float)(factor * h[i]);
    float* d = nullptr;
    if (hipMalloc(&d, sizeof(float) * f.size()) != hipSuccess) return nullptr;
    if (copy_sync(d, f.data(), sizeof(float) * f.size(), hipMemcpyHostToDevice) != hipSuccess) {
        hipFree(d);
        return nullptr;
    }
    cache[key] = d;
    return d;
}

// K = noise * sqrt(L^3/2) * amp[n^2] (the scaling of src/grf.c:33 and the
// phi1 table), DC = 0; noise dense N x N x (N/2+1)
template <typename T>
__global__ void k_noise_in(const cx<T>* __restrict__ noise, cx<T>* K, long hs, int N,
                           double boxlen, const double* __restrict__ amp) {
    const int H = N / 2 + 1;
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (long)N * N * H) return;
    const int z = (int)(i % H);
    const long row = i / H;
    const int x = (int)(row / N), y = (int)(row % N);
    const int nx = freq_index(x, N), ny = freq_index(y, N);
    const long n2 = (long)nx * nx + (long)ny * ny + (long)z * z;
    const double f = sqrt(boxlen * boxlen * boxlen / 2) * amp[n2];
    const cx<T> v = noise[i];
    K[row * hs + z] = n2 ? mk<T>((T)((double)v.re * f), (T)((double)v.im * f)) : mk<T>(0, 0);
}

template <typename T>
__global__ void k_fill_u64(unsigned long long* p, long n) {
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = 0;
}

inline unsigned nblk(long n, int b = 256) { return (unsigned)((n + b - 1) / b); }

// ---- FFT schedule autotuner ------------------------------------------------------------
// The plain passes of the pipeline have kFftVariants schedules each (radix
// split, tile width, rows per work-group; see fft_launch.h).  The first
// pipeline of a (device, N, precision) times every variant on its own grids
// and keeps the fastest; later pipelines of the same key reuse the choice,
// so every run in the process uses the same kernels (ensembles and unbatched
// runs give identical bits).  MITOS_FFT_SCHEDULE=default skips the timing.
enum TuneKind { TUNE_Y_FWD = 0, TUNE_X_FWD = 1, TUNE_Z_C2R = 2, TUNE_Z_R2C = 3, TUNE_KINDS = 4 };

struct FftSchedule {
    int v[TUNE_KINDS] = {0, 0, 0, 0};
    float ms[TUNE_KINDS][kFftVariants] = {};
};

inline std::mutex& schedule_mutex() {
    static std::mutex mu;
    return mu;
}
inline std::map<std::tuple<int, int, int>, FftSchedule>& schedule_table() {
    static std::map<std::tuple<int, int, int>, FftSchedule> t;
    return t;
}

// ---- the fused pipeline ------------------------------------------------------------------
template <typename T>
struct Pipe {
    int N = 0;
    long hs = 0;      // complex row stride (elements): N/2+1 rounded up to 128 bytes
    long csize = 0;   // elements of one complex grid
    cx<T>* K = nullptr;
    cx<T>* A = nullptr;  // 3 complex grids
    cx<T>* B = nullptr;  // 6 complex grids
    float *X = nullptr, *Y = nullptr, *Z = nullptr;
    long long pcap = 0;   // particles X, Y, Z hold
    long long npart = 0;  // particles of the last realization (M^3)
    double* pk_sums = nullptr;  // device [bins][2]
    long long* pk_obs = nullptr;
    double* pk_part = nullptr;  // per-work-group P(k) partials of this pipeline
    long long* pk_cnt = nullptr;
    int bins_alloc = 0;
    hipEvent_t ev[9] = {};
    double amplitude = 0;
    // optional per-kernel profile of the last run: name, algorithmic bytes,
    // start/stop events on the run's stream
    bool prof = false;
    int nprof = 0;
    const char* pname[32];
    double pbytes[32];
    hipEvent_t pev[33];
    template <typename F>
    int timed(hipStream_t s, const char* name, double bytes, F&& f) {
        if (prof && nprof < 32) {
            hipEventRecord(pev[nprof], s);
            const int rc = f();
            pname[nprof] = name;
            pbytes[nprof] = bytes;
            nprof++;
            hipEventRecord(pev[nprof], s);
            return rc;
        }
        return f();
    }

    FftSchedule sched;
    bool psi_stencilled = false;  // the displacement grids hold the stencil form
    // workspace of the two-pass lattice deposit (float weights, N >= 128);
    // null: the deposit adds its windows with atomics
    void* cic_ws = nullptr;
    // the adjoint's fixed-point scatter accumulators (two int64 grids and two
    // maxima), allocated at the first backward run
    unsigned long long* adj_ws = nullptr;
    // the FP32 displacement stages its taps in LDS (MITOS_TSC_DIRECT=1: reads
    // them from the grids, the same bits; for tests)
    bool tsc_staged = true;
    // the FP32 displacement over 8 x 8 x 16 tiles (MITOS_TSC_KERNEL=wave: the
    // one-wave row kernel)
    bool tsc_tile = true;

    // time every schedule variant of the plain passes (or reuse the choice
    // made for this device, N and precision)
    int autotune(hipStream_t s);

    // Mean time of a plain 3D r2c (real rows of prs() -> K) and c2r
    // (K -> real) over reps runs each, with the tuned schedules; uses the
    // pipeline's grids as scratch.
    int fft_timing(hipStream_t s, int reps, float* r2c_ms, float* c2r_ms);

    cx<T>* a(int i) { return A + (size_t)i * csize; }
    cx<T>* b(int i) { return B + (size_t)i * csize; }
    T* psi(int i) { return reinterpret_cast<T*>(b(3 + i)); }
    // Row stride (reals) of the displacement and delta2 grids: one complex row,
    // so every real row starts on a 128-byte boundary as the complex rows do.
    long prs() const { return 2 * hs; }
    unsigned long long* cic() { return reinterpret_cast<unsigned long long*>(b(0)); }
    // fixed-point unit of the lattice deposit (float weights in the FP32 pipeline)
    static int cic_shift() { return sizeof(T) == 4 ? MITOS_CIC_SHIFT_F32 : MITOS_CIC_SHIFT; }
    // overdensity scale of the fixed-point grid: 2^-shift * N^3 / npart
    double cic_norm() const {
        const double n3 = (double)N * N * N;
        const double f = (npart == 0 || (double)npart == n3) ? 1.0 : n3 / (double)npart;
        return ldexp(1.0, -cic_shift()) * f;
    }

    // npart_cap: the most lattice particles a realization may have (0: N^3)
    int create(int n, long long npart_cap = 0) {
        N = n;
        const long H = N / 2 + 1;
        const long q = 128 / sizeof(cx<T>);
        hs = (H + q - 1) / q * q;
        csize = (long)N * N * hs;
        // a displacement grid (rows of prs() = 2 hs reals, halo included) fits
        // in a complex grid
        if (N + MITOS_PSI_HO + 1 > 2 * hs) return MITOS_ERR_UNSUPPORTED;
        const long long ng = (long long)N * N * N;
        pcap = npart_cap > ng ? npart_cap : ng;
        MITOS_HIP_CHECK(hipMalloc(&K, sizeof(cx<T>) * csize));
        MITOS_HIP_CHECK(hipMalloc(&A, sizeof(cx<T>) * csize * 3));
        MITOS_HIP_CHECK(hipMalloc(&B, sizeof(cx<T>) * csize * 6));
        MITOS_HIP_CHECK(hipMalloc(&X, sizeof(float) * pcap));
        MITOS_HIP_CHECK(hipMalloc(&Y, sizeof(float) * pcap));
        MITOS_HIP_CHECK(hipMalloc(&Z, sizeof(float) * pcap));
        typedef typename std::conditional<sizeof(T) == 4, float, double>::type M;
        const size_t wsb = cic_stream_bytes<M>(N);
        const char* direct_env = getenv("MITOS_TSC_DIRECT");
        tsc_staged = !(direct_env && direct_env[0] == '1');
        const char* kern_env = getenv("MITOS_TSC_KERNEL");
        tsc_tile = !(kern_env && strcmp(kern_env, "wave") == 0);
        const char* atomic_env = getenv("MITOS_CIC_ATOMIC");
        const bool force_atomic = atomic_env && atomic_env[0] == '1';
        if (wsb && !force_atomic && hipMalloc(&cic_ws, wsb) != hipSuccess) {
            (void)hipGetLastError();  // no room: the atomic deposit needs none
            cic_ws = nullptr;
        }
        for (int i = 0; i < 9; i++) MITOS_HIP_CHECK(hipEventCreate(&ev[i]));
        for (int i = 0; i < 33; i++) MITOS_HIP_CHECK(hipEventCreate(&pev[i]));
        return MITOS_OK;
    }

    void destroy() {
        hipDeviceSynchronize();
        hipFree(K);
        hipFree(A);
        hipFree(B);
        hipFree(X);
        hipFree(Y);
        hipFree(Z);
        hipFree(pk_sums);
        hipFree(pk_obs);
        hipFree(pk_part);
        hipFree(pk_cnt);
        hipFree(cic_ws);
        hipFree(adj_ws);
        for (int i = 0; i < 9; i++)
            if (ev[i]) hipEventDestroy(ev[i]);
        for (int i = 0; i < 33; i++)
            if (pev[i]) hipEventDestroy(pev[i]);
    }

    int ensure_bins(int bins) {
        if (bins <= bins_alloc) return MITOS_OK;
        hipFree(pk_sums);
        hipFree(pk_obs);
        hipFree(pk_part);
        hipFree(pk_cnt);
        const int nb = pk_blocks((long)N * N * (N / 2 + 1));
        MITOS_HIP_CHECK(hipMalloc(&pk_sums, sizeof(double) * 2 * bins));
        MITOS_HIP_CHECK(hipMalloc(&pk_obs, sizeof(long long) * bins));
        MITOS_HIP_CHECK(hipMalloc(&pk_part, sizeof(double) * 4 * bins * nb));
        MITOS_HIP_CHECK(hipMalloc(&pk_cnt, sizeof(long long) * bins * nb));
        bins_alloc = bins;
        return MITOS_OK;
    }

    // One realization on stream s.  amp_tab: device phi1 amplitude table to use
    // instead of the cached one; pk_dst/obs_dst: device destinations of the
    // P(k) sums and counts instead of pk_sums/pk_obs.  No allocation and no
    // host synchronisation happen here once the tables of cfg exist, so the
    // call can be captured into a graph.
    // noise_in: unit-variance complex white noise (dense N x N x (N/2+1) of cx<T>)
    // used instead of the seed's stream.  stencil: -1 as the precision
    // (FP32 applies the lattice TSC stencils in k-space, FP64 gathers 27 taps),
    // 1 forces the stencil form (the form the adjoint differentiates).
    int enqueue(const mitos_ic_config& cfg, hipStream_t s, bool timing,
                const double* amp_tab = nullptr, double* pk_dst = nullptr,
                long long* obs_dst = nullptr, const cx<T>* noise_in = nullptr,
                int stencil = -1);
};

// instantiated in pipe_f32.hip and pipe_f64.hip
extern template struct Pipe<float>;
extern template struct Pipe<double>;

}  // namespace mitos
