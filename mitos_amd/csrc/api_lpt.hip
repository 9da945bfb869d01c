// Drop-in second-order potential solvers: solve2LPT (src/2lpt.c:38-143) and
// solveMongeAmpere (src/monge_ampere.c:50-183).
//
// The reference derives each of the six Hessian components by two k-space
// kernels and a 3D transform of its own.  Here the x pass writes three grids,
// the y pass six from those, and the z pass combines the six rows
// (multi_launch.h), so each line is read once per axis; c2r of the potential
// itself is the z pass of one of the six.  The six grids between the y and z
// passes exist as slabs of x planes, halves (2LPT) or quarters (Monge-Ampere,
// which also holds six real slabs): with the transforms' work grid eight grids
// in all, nine were held by the separate transforms.  Smaller slabs, which the
// memory-side cache would hold, are slower (2LPT at 384^3: halves 6.2 ms, slabs
// of 128 MB 8.2 ms): the launches get too short.
// solve2LPT at 256^3: 3.46 -> 1.60 ms, bound by HBM and the memory-side cache
// (6.6 GB in its passes).
#include <string.h>

#include <vector>

#include "dropin.h"
#include "kspace.h"
#include "multi_launch.h"

using namespace mitos;

namespace {

inline unsigned nblk(long n, int b = 256) { return (unsigned)((n + b - 1) / b); }

// z c2r of -k_z^2 times the values
struct OpKz2 {
    double dk;
    __device__ __forceinline__ cx<double> pre(cx<double> v, int, int, int z) const {
        return apply_mul(2, v, z * dk);
    }
    __device__ __forceinline__ cx<double> post(cx<double> v, int, int, int) const { return v; }
};

// The work of one solver call: K (the potential's modes) and three grids between
// the x and y passes, rows of hs, and six slabs of `planes` x planes
// (about N / parts).
struct HessianWork {
    int N, planes;
    long hs;
    double boxlen;  // the potential's: its wavenumbers and volume
    double hvol;    // the density's volume, of the Hessian grids
    char* mem = nullptr;
    cx<double>*K = nullptr, *A[3] = {}, *B[6] = {};

    HessianWork(int n, double L, double Ld, int parts)
        : N(n), hs(work_row<double>(n)), boxlen(L), hvol(Ld * Ld * Ld) {
        planes = n;
        for (int q = parts; q > 1 && planes % 2 == 0; q /= 2) planes /= 2;
        const size_t grid = (size_t)n * n * hs, slab = (size_t)planes * n * hs;
        mem = (char*)pool_alloc(sizeof(cx<double>) * (4 * grid + 6 * slab));
        if (!mem) return;
        K = reinterpret_cast<cx<double>*>(mem);
        for (int i = 0; i < 3; i++) A[i] = K + (i + 1) * grid;
        for (int i = 0; i < 6; i++) B[i] = K + 4 * grid + i * slab;
    }
    ~HessianWork() { pool_free(mem); }

    double dk() const { return 2 * M_PI / boxlen; }
    double vol() const { return boxlen * boxlen * boxlen; }

    // x pass: A0 = X(K), A1 = X(i kx K), A2 = X(-kx^2 K)
    int x_pass(hipStream_t s) {
        return with_size(N, [&]<int NN>() -> int {
            MultiPtrs<double, 1, 3> p;
            p.in[0] = K;
            for (int i = 0; i < 3; i++) p.out[i] = A[i];
            return MultiK<double, NN, 0, 1, 1,
                          OutCodes<MITOS_OUT(0, 0), MITOS_OUT(0, 1), MITOS_OUT(0, 2)>>::go(
                p, hs, dk(), s);
        });
    }
    // y pass of the slab from plane x0: B0 = Y(A0), B1 = Y(i ky A0),
    // B2 = Y(-ky^2 A0), B3 = Y(A1), B4 = Y(i ky A1), B5 = Y(A2)
    int y_pass(int x0, hipStream_t s) {
        return with_size(N, [&]<int NN>() -> int {
            MultiPtrs<double, 3, 6> p;
            for (int i = 0; i < 3; i++) p.in[i] = A[i] + (size_t)x0 * N * hs;
            for (int i = 0; i < 6; i++) p.out[i] = B[i];
            return MultiK<double, NN, 1, 1, 3,
                          OutCodes<MITOS_OUT(0, 0), MITOS_OUT(0, 1), MITOS_OUT(0, 2),
                                   MITOS_OUT(1, 0), MITOS_OUT(1, 1), MITOS_OUT(2, 0)>>::go(
                p, hs, dk(), s, planes);
        });
    }
    // z c2r of a slab's grid into rows of rs reals (src/fft.c:243-254)
    template <typename OP>
    int z_pass(const cx<double>* b, double* out, long rs, double vol, OP op, hipStream_t s) {
        return with_size(N, [&]<int NN>() -> int {
            return zc2r_pass_v<double, NN, 1, 0>(b, out, hs, rs, 1, 0, 0, 1.0 / vol, op, s, 0,
                                                 (long)planes * N);
        });
    }
    // delta2 rows of a slab (src/2lpt.c:84-116)
    int delta2(double* out, long rs, hipStream_t s) {
        MultiPtrs<double, 6, 1> p;
        for (int i = 0; i < 6; i++) p.in[i] = B[i];
        return with_size(N, [&]<int NN>() -> int {
            return HessZK<double, NN>::go(p, hs, dk(), 1.0 / hvol, out, rs, s,
                                          (long)planes * N);
        });
    }
};

// 2lpt.c:131-133 (f1 = f2 = 1: src/monge_ampere.c:166-170); n even
__global__ void k_combine(double* pot, const double* __restrict__ work, long n, double f1,
                          double f2) {
#pragma clang fp contract(off)
    const long k = 2 * ((long)blockIdx.x * blockDim.x + threadIdx.x);
    if (k >= n) return;
    double2 p = *reinterpret_cast<const double2*>(pot + k);
    const double2 w = *reinterpret_cast<const double2*>(work + k);
    p.x = p.x * f1 + f2 * w.x;
    p.y = p.y * f1 + f2 * w.y;
    *reinterpret_cast<double2*>(pot + k) = p;
}

struct HessPtrs {
    const double* h[6];  // xx, xy, xz, yy, yz, zz
};

// src/monge_ampere.c:124-151: residual (1 + rho) - det(I + Hessian) of every
// entry (padding included), and per-block sums of resid^2 and rho^2 (tree in
// a fixed order, so the diagnostic does not depend on scheduling)
__global__ void __launch_bounds__(256) k_ma_residual(double* out, HessPtrs p,
                                                     const double* __restrict__ rho, long n,
                                                     double* part) {
#pragma clang fp contract(off)
    __shared__ double se[256], sn[256];
    const long k = (long)blockIdx.x * blockDim.x + threadIdx.x;
    double e = 0, q = 0;
    if (k < n) {
        const double d_dxx = p.h[0][k], d_dxy = p.h[1][k], d_dxz = p.h[2][k];
        const double d_dyy = p.h[3][k], d_dyz = p.h[4][k], d_dzz = p.h[5][k];
        const double M0 = 1 + d_dxx, M1 = d_dxy, M2 = d_dxz;
        const double M3 = d_dxy, M4 = 1 + d_dyy, M5 = d_dyz;
        const double M6 = d_dxz, M7 = d_dyz, M8 = 1 + d_dzz;
        // det3 of src/monge_ampere.c:38-42
        const double det = M0 * (M4 * M8 - M5 * M7) - M1 * (M3 * M8 - M5 * M6) +
                           M2 * (M3 * M7 - M4 * M6);
        const double r = rho[k];
        const double resid = (1 + r) - det;
        out[k] = resid;
        e = resid * resid;
        q = r * r;
    }
    se[threadIdx.x] = e;
    sn[threadIdx.x] = q;
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        if ((int)threadIdx.x < w) {
            se[threadIdx.x] += se[threadIdx.x + w];
            sn[threadIdx.x] += sn[threadIdx.x + w];
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        part[2 * blockIdx.x] = se[0];
        part[2 * blockIdx.x + 1] = sn[0];
    }
}

// the argument checks both solvers share (src/2lpt.c:54-72,
// src/monge_ampere.c:68-85: asserts in the reference, and 1 for a density that
// is not in momentum space)
int check_grids(const struct distributed_grid* potential, const struct distributed_grid* density,
                const struct distributed_grid* work) {
    if (!potential || !density || !work) return MITOS_ERR_ARG;
    if (potential->NX != density->NX || density->NX != work->NX ||
        potential->X0 != density->X0 || density->X0 != work->X0 ||
        potential->N != density->N || density->N != work->N)
        return MITOS_ERR_DIMS;
    if (potential->box == density->box || work->box == density->box ||
        potential->box == work->box)
        return MITOS_ERR_ARG;
    if (density->momentum_space != 1) return 1;
    if (!potential->box || !potential->fbox || !density->box || !density->fbox || !work->box ||
        !work->fbox)
        return MITOS_ERR_ARG;
    if (!size_supported(density->N)) return MITOS_ERR_UNSUPPORTED;
    return MITOS_OK;
}

int add_second_order(struct distributed_grid* potential, const struct distributed_grid* work,
                     double f1, double f2) {
    const long padded = (long)potential->N * potential->N * (potential->N + 2);
    hipLaunchKernelGGL(k_combine, dim3(nblk(padded / 2)), dim3(256), 0, api_stream(),
                       potential->box, work->box, padded, f1, f2);
    return launch_status();
}

int solve_2lpt(struct distributed_grid* potential, struct distributed_grid* density,
               struct distributed_grid* work, double f1, double f2) {
    MITOS_TRY(check_grids(potential, density, work));
    const int N = density->N;
    const long rs = N + 2;
    HessianWork W(N, potential->boxlen, density->boxlen, 2);
    if (!W.mem) return MITOS_ERR_ALLOC;
    hipStream_t s = api_stream();
    // phi1(k) = inv_poisson * density (:75), then the density's modes anew (:78)
    KSpec ip{};
    ip.id = KID_INV_POISSON;
    MITOS_TRY(apply_padded_issue(W.K, W.hs, density, ip));
    MITOS_TRY(W.x_pass(s));
    MITOS_TRY(dg_r2c_issue(density, false));
    for (int x0 = 0; x0 < N; x0 += W.planes) {
        MITOS_TRY(W.y_pass(x0, s));
        // phi1(x) and delta2(x) rows of the slab
        MITOS_TRY(W.z_pass(W.B[0], potential->box + (size_t)x0 * N * rs, rs, W.vol(), OpNone(),
                           s));
        MITOS_TRY(W.delta2(work->box + (size_t)x0 * N * rs, rs, s));
    }
    // phi2 = Poisson solve of delta2 (:120-125), combined (:131-133), to k-space
    MITOS_TRY(dg_r2c_issue(work, true));
    MITOS_TRY(dg_c2r_issue(work));
    MITOS_TRY(add_second_order(potential, work, f1, f2));
    MITOS_TRY(dg_r2c_issue(potential, false));
    return api_sync();
}

thread_local std::vector<double> g_ma_eps;

int solve_monge_ampere(struct distributed_grid* potential, struct distributed_grid* density,
                       struct distributed_grid* work, int cycles) {
    MITOS_TRY(check_grids(potential, density, work));
    if (cycles < 0) return MITOS_ERR_ARG;
    g_ma_eps.clear();
    const int N = density->N;
    const long rs = N + 2;
    hipStream_t s = api_stream();
    KSpec ip{}, one{};
    ip.id = KID_INV_POISSON;
    one.id = KID_CONSTANT;
    one.p[0] = 1.0;
    // the Zel'dovich potential, then the density's modes anew (:91, as 2lpt.c:78)
    MITOS_TRY(apply_padded_issue(reinterpret_cast<cx<double>*>(potential->fbox), N / 2 + 1,
                                 density, ip));
    potential->momentum_space = 1;
    MITOS_TRY(dg_r2c_issue(density, false));
    if (cycles == 0) return api_sync();
    HessianWork W(N, potential->boxlen, density->boxlen, 4);
    if (!W.mem) return MITOS_ERR_ALLOC;
    const long slab = (long)W.planes * N * rs;
    const unsigned nb = nblk(slab), nslabs = (unsigned)(N / W.planes);
    struct Block {  // the six slabs of Hessian rows and the residual's partial sums
        double* p;
        explicit Block(size_t n) : p((double*)pool_alloc(sizeof(double) * n)) {}
        ~Block() { pool_free(p); }
    } h(6 * (size_t)slab + 2 * (size_t)nb * nslabs);
    if (!h.p) return MITOS_ERR_ALLOC;
    double* part = h.p + 6 * slab;
    std::vector<double> hp(2 * (size_t)nb * nslabs);
    for (int it = 0; it < cycles; it++) {
        MITOS_TRY(apply_padded_issue(W.K, W.hs, potential, one));
        MITOS_TRY(W.x_pass(s));
        for (unsigned i = 0; i < nslabs; i++) {
            const int x0 = (int)i * W.planes;
            const size_t at = (size_t)x0 * N * rs;
            MITOS_TRY(W.y_pass(x0, s));
            // the six Hessian components (:103-117), the potential itself, and the
            // residuals (:120-151)
            HessPtrs H;
            for (int j = 0; j < 6; j++) H.h[j] = h.p + j * slab;
            MITOS_TRY(W.z_pass(W.B[5], h.p + 0 * slab, rs, W.hvol, OpNone(), s));
            MITOS_TRY(W.z_pass(W.B[4], h.p + 1 * slab, rs, W.hvol, OpNone(), s));
            MITOS_TRY(W.z_pass(W.B[3], h.p + 2 * slab, rs, W.hvol, OpIkz{W.dk()}, s));
            MITOS_TRY(W.z_pass(W.B[2], h.p + 3 * slab, rs, W.hvol, OpNone(), s));
            MITOS_TRY(W.z_pass(W.B[1], h.p + 4 * slab, rs, W.hvol, OpIkz{W.dk()}, s));
            MITOS_TRY(W.z_pass(W.B[0], h.p + 5 * slab, rs, W.hvol, OpKz2{W.dk()}, s));
            MITOS_TRY(W.z_pass(W.B[0], potential->box + at, rs, W.vol(), OpNone(), s));
            hipLaunchKernelGGL(k_ma_residual, dim3(nb), dim3(256), 0, s, work->box + at, H,
                               density->box + at, slab, part + 2 * (size_t)nb * i);
            MITOS_TRY(launch_status());
        }
        MITOS_HIP_CHECK(hipMemcpyAsync(hp.data(), part, sizeof(double) * hp.size(),
                                       hipMemcpyDeviceToHost, s));
        MITOS_HIP_CHECK(hipStreamSynchronize(s));
        double eps = 0, norm = 0;
        for (size_t b = 0; b < hp.size(); b += 2) {
            eps += hp[b];
            norm += hp[b + 1];
        }
        // (:159-172) Poisson solve of the residual, added to the potential
        MITOS_TRY(dg_r2c_issue(work, true));
        MITOS_TRY(dg_c2r_issue(work));
        MITOS_TRY(add_second_order(potential, work, 1.0, 1.0));
        MITOS_TRY(dg_r2c_issue(potential, false));
        // (:183-186) root-mean-square residual relative to the source
        g_ma_eps.push_back(sqrt((eps / norm) / ((double)N * N * N)));
    }
    return api_sync();
}

}  // namespace

extern "C" int solve2LPT(struct distributed_grid* potential, struct distributed_grid* density,
                         struct distributed_grid* workspace_grid, double factor1,
                         double factor2) {
    return set_last_error(solve_2lpt(potential, density, workspace_grid, factor1, factor2));
}

extern "C" int solveMongeAmpere(struct distributed_grid* potential,
                                struct distributed_grid* density,
                                struct distributed_grid* workspace_grid, int cycles) {
    return set_last_error(solve_monge_ampere(potential, density, workspace_grid, cycles));
}

extern "C" int mitos_monge_ampere_residuals(double* rms_eps, int n) {
    const int m = (int)g_ma_eps.size();
    for (int i = 0; i < n && i < m && rms_eps; i++) rms_eps[i] = g_ma_eps[i];
    return m;
}
