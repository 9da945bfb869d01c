// Hand-written adjoint of the IC pipeline: the gradient of a P(k) or density
// loss with respect to the white noise.
//
// The forward run is the pipeline in its stencil form (the lattice TSC
// stencils applied in k-space, k_displace_lattice_s) started from a given
// noise field.  The backward pass, in the order it runs:
//   P(k) bins        -> dL/dK(k) = 2 f^2 g_b K / (obs_b L^3)      (f: window)
//   r2c of delta     -> dL/drho(x) = c2r of the half spectrum
//   CIC deposit      -> dL/dX per particle (corner differences of the grid)
//   sequential TSC   -> scatter into the adjoints of the three stencilled
//                       displacement grids, with the position derivatives of
//                       the later moves carried to the earlier ones
//   c2r of psi       -> r2c, times the multiplicity of half-spectrum modes
//   k-space combine  -> dL/dphi1 (direct) and dL/dD (2LPT source)
//   r2c of delta2    -> dL/ddelta2(x)
//   delta2 = sum of Hessian minors (src/2lpt.c:111-112): the six phi_,ij
//                       grids are recomputed from phi1, not stored
//   phi_,ij = c2r(-k_i k_j phi1) -> six r2c, accumulated into dL/dphi1
//   Hermitian planes and the spectrum amplitude -> dL/dnoise
#include "pipe.h"

using namespace mitos;

namespace mitos {

// P(k) adjoint: K <- coef[bin] f(k)^2 K with f = s w[x] w[y] w[z] (the CIC
// window and normalisation of PkCicTransform); modes outside the bins -> 0
template <typename T>
__global__ void k_adj_pk(cx<T>* K, long hs, int N, const int* __restrict__ edges, float cinv,
                         int bins, const double* __restrict__ coef, double s,
                         const double* __restrict__ win) {
    const int H = N / 2 + 1;
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (long)N * N * H) return;
    const int z = (int)(i % H);
    const long row = i / H;
    const int x = (int)(row / N), y = (int)(row % N);
    const int nx = freq_index(x, N), ny = freq_index(y, N);
    const long n2 = (long)nx * nx + (long)ny * ny + (long)z * z;
    cx<T>* p = K + row * hs + z;
    if (n2 == 0) {
        *p = mk<T>(0, 0);
        return;
    }
    const int b = pk_bin_of(n2, edges, bins, cinv);
    const double f = s * win[x] * win[y] * win[z];
    const double c = coef[b] * f * f;
    const cx<T> v = *p;
    *p = mk<T>((T)(v.re * c), (T)(v.im * c));
}

template <typename T>
__global__ void k_add_real(T* a, const T* __restrict__ b, long n) {
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) a[i] += b[i];
}

template <typename T>
__global__ void k_fill(T* p, long n, T v) {
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = v;
}

// bits of the fixed-point sums of the scatter adjoint below the largest gradient
constexpr int kAdjFixedBits = 48;

// the larger magnitude; a NaN stays
template <typename T>
__device__ __forceinline__ T adj_max(T m, T a) {
    return (a > m || a != a) ? a : m;
}

// Adjoint of the particles, in two passes over 8 x 8 x 16 lattice tiles.
// sx, sy, sz: the stencilled displacement grids (rows of rs); grho, Ax, gy, gz:
// dense N^3 grids.
//
// k_adj_gradients, per particle: the three moves recomputed in T with the
// position derivatives of their taps, the CIC adjoint at the final position,
// and from them dL/dx, dL/dy, dL/dz of the moves: Ax = -dL/dx (the x move reads
// its own site alone), gy and gz to memory.  Each work-group leaves the largest
// |gy| and |gz| in part: two atomic maxima per particle queued at one line, 6.0
// ms at 256^3 in FP32 against 0.54 ms now, bound by the 21 tap loads.
template <typename T>
__global__ void __launch_bounds__(256)
    k_adj_gradients(const T* __restrict__ sx, const T* __restrict__ sy, const T* __restrict__ sz,
                    unsigned rs, const T* __restrict__ grho, T* __restrict__ Ax,
                    T* __restrict__ gyo, T* __restrict__ gzo, double* __restrict__ part, int N,
                    double boxlen, float spacing) {
    __shared__ double red[2][4];
    int x0, y0, z0;
    adj_tile(xcd_block(blockIdx.x, gridDim.x), N, x0, y0, z0);
    const int qz = z0 + (int)(threadIdx.x & 15), qy = y0 + (int)((threadIdx.x >> 4) & 7);
    const T Lb = (T)boxlen, sN = (T)(N / boxlen);
    const float invN = 1.0f / N;
    const unsigned plane = (unsigned)N * rs, zo = MITOS_PSI_SO + qz;
    T my = 0, mz = 0;
    if (qz < N) {
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const int qx = x0 + (int)(threadIdx.x >> 7) + 2 * j;
            const unsigned yz = (unsigned)qy * rs + zo;
            // x1 = x0 - Sx(q), y1 = y0 - Fy(x1), z1 = z0 - Fz(x1, y1) as moves_s forms
            // them: the cell of a particle at a cell's edge, and so its whole
            // gradient, hangs on the last bit
            T x1, y1, z1;
            moves_s(sx, sy, sz, rs, N, sN, spacing, qx, qy, qz, x1, y1, z1);
            // dFy/dx, dFz/dx and dFz/dy from the same taps
            int cx, cy;
            T wx[3], dwx[3], wy[3], dwy[3];
            unsigned ox[3], oy[3];
            tsc_axis_near_d(x1 * sN, cx, wx, dwx);
            tsc_axis_near_d(y1 * sN, cy, wy, dwy);
            tap_rows(wrapf(cx, N, invN), N, plane, ox);
            tap_rows(wrapf(cy, N, invN), N, rs, oy);
            T Fy_x = 0, Fz_x = 0, Fz_y = 0;
#pragma unroll
            for (int a = 0; a < 3; a++) {
                Fy_x += dwx[a] * sy[ox[a] + yz];
#pragma unroll
                for (int b = 0; b < 3; b++) {
                    const T v = sz[ox[a] + oy[b] + zo];
                    Fz_x += dwx[a] * wy[b] * v;
                    Fz_y += wx[a] * dwy[b] * v;
                }
            }
            // CIC (analyse/src/mitos_read.c:285-320): d rho(corner) / d position
            int cx0, cy0, cz0;
            T dx, dy, dz;
            cic_cell_t(wrap_pos(x1, Lb), sN, N, cx0, dx);
            cic_cell_t(wrap_pos(y1, Lb), sN, N, cy0, dy);
            cic_cell_t(wrap_pos(z1, Lb), sN, N, cz0, dz);
            const int cxp = wrap1(cx0 + 1, N), cyp = wrap1(cy0 + 1, N), czp = wrap1(cz0 + 1, N);
            auto g = [&](int a, int b, int c) { return grho[((size_t)a * N + b) * N + c]; };
            const T g000 = g(cx0, cy0, cz0), g100 = g(cxp, cy0, cz0), g010 = g(cx0, cyp, cz0),
                    g001 = g(cx0, cy0, czp), g110 = g(cxp, cyp, cz0), g101 = g(cxp, cy0, czp),
                    g011 = g(cx0, cyp, czp), g111 = g(cxp, cyp, czp);
            const T tx = 1 - dx, ty = 1 - dy, tz = 1 - dz;
            const T gX = sN * (ty * tz * (g100 - g000) + dy * tz * (g110 - g010) +
                               ty * dz * (g101 - g001) + dy * dz * (g111 - g011));
            const T gY = sN * (tx * tz * (g010 - g000) + dx * tz * (g110 - g100) +
                               tx * dz * (g011 - g001) + dx * dz * (g111 - g101));
            const T gZ = sN * (tx * ty * (g001 - g000) + dx * ty * (g101 - g100) +
                               tx * dy * (g011 - g010) + dx * dy * (g111 - g110));
            const T gz = gZ;
            const T gy = gY - gz * Fz_y * sN;
            const T gx = gX - gz * Fz_x * sN - gy * Fy_x * sN;
            const size_t p = ((size_t)qx * N + qy) * N + qz;
            Ax[p] = -gx;
            gyo[p] = gy;
            gzo[p] = gz;
            my = adj_max(my, (T)fabs(gy));
            mz = adj_max(mz, (T)fabs(gz));
        }
    }
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) {
        my = adj_max(my, __shfl_xor(my, o, 64));
        mz = adj_max(mz, __shfl_xor(mz, o, 64));
    }
    if ((threadIdx.x & 63) == 0) {
        red[0][threadIdx.x >> 6] = (double)my;
        red[1][threadIdx.x >> 6] = (double)mz;
    }
    __syncthreads();
    if (threadIdx.x < 2) {
        double m = red[threadIdx.x][0];
        for (int w = 1; w < 4; w++) m = adj_max(m, red[threadIdx.x][w]);
        part[2 * blockIdx.x + threadIdx.x] = m;
    }
}

// gmax[0], gmax[1] = largest of the n pairs of part; one work-group
static __global__ void __launch_bounds__(1024)
    k_adj_max(const double* __restrict__ part, unsigned n, double* gmax) {
    __shared__ double red[2][16];
    double m[2] = {0, 0};
    for (unsigned i = threadIdx.x; i < n; i += 1024)
        for (int q = 0; q < 2; q++) m[q] = adj_max(m[q], part[2 * i + q]);
    for (int q = 0; q < 2; q++) {
        for (int o = 32; o >= 1; o >>= 1) m[q] = adj_max(m[q], __shfl_xor(m[q], o, 64));
        if ((threadIdx.x & 63) == 0) red[q][threadIdx.x >> 6] = m[q];
    }
    __syncthreads();
    if (threadIdx.x < 2) {
        double v = red[threadIdx.x][0];
        for (int w = 1; w < 16; w++) v = adj_max(v, red[threadIdx.x][w]);
        gmax[threadIdx.x] = v;
    }
}

// k_adj_scatter: the y and z move adjoints go to the x rows, and x and y rows,
// that the moves read: -g w in units of max|g| 2^-48 to 64-bit integers (at most
// 2^15 maximal contributions per cell before overflow), so the sums do not
// depend on their order and gradients are bit-reproducible;
// k_adj_fixed_to_real converts them.  Twelve global atomics per particle were
// bound by the memory-side atomic units (5.8 ms at 256^3 in FP32); here a tile
// sums in LDS windows placed at its mean displacement, four cells of margin on
// each side, and adds whole rows of 16 z to the grids (0.56 ms).  A particle past
// the margin takes the global atomics.
template <typename T>
__global__ void __launch_bounds__(512)
    k_adj_scatter(const T* __restrict__ sx, const T* __restrict__ sy, unsigned rs,
                  const T* __restrict__ gyi, const T* __restrict__ gzi, unsigned long long* AyI,
                  unsigned long long* AzI, const double* __restrict__ gmax, int N, double boxlen,
                  float spacing) {
    constexpr int MARGIN = 4, WX = kAdjTX + 2 * (MARGIN + 1), TZ = kAdjTZ;
    __shared__ unsigned long long winz[WX * WX * TZ];
    __shared__ unsigned long long winy[WX * kAdjTY * TZ];
    __shared__ int red[2][8];
    int x0, y0, z0;
    adj_tile(xcd_block(blockIdx.x, gridDim.x), N, x0, y0, z0);
    const int lz = threadIdx.x & 15, ly = (threadIdx.x >> 4) & 7;
    const int qz = z0 + lz, qy = y0 + ly;
    const bool ok = qz < N;
    for (int i = threadIdx.x; i < WX * WX * TZ; i += 512) winz[i] = 0;
    for (int i = threadIdx.x; i < WX * kAdjTY * TZ; i += 512) winy[i] = 0;
    const T sN = (T)(N / boxlen);
    const float invN = 1.0f / N;
    const unsigned plane = (unsigned)N * rs, yz = (unsigned)qy * rs + MITOS_PSI_SO + qz;
    int cx[2], cy[2], sumx = 0, sumy = 0;
    T wx[2][3], wy[2][3], gy[2], gz[2];
#pragma unroll
    for (int j = 0; j < 2; j++) {
        const int qx = x0 + (int)(threadIdx.x >> 7) + 4 * j;
        cx[j] = qx;
        cy[j] = qy;
        gy[j] = gz[j] = 0;
        if (!ok) continue;
        const size_t p = ((size_t)qx * N + qy) * N + qz;
        gy[j] = gyi[p];
        gz[j] = gzi[p];
        const T x1 = (T)(qx * spacing) - sx[(unsigned)qx * plane + yz];
        tsc_axis_near(x1 * sN, cx[j], wx[j]);
        unsigned ox[3];
        tap_rows(wrapf(cx[j], N, invN), N, plane, ox);
        T y1 = (T)(qy * spacing);
        y1 -= wx[j][0] * sy[ox[0] + yz] + wx[j][1] * sy[ox[1] + yz] + wx[j][2] * sy[ox[2] + yz];
        tsc_axis_near(y1 * sN, cy[j], wy[j]);
        sumx += cx[j] - qx;
        sumy += cy[j] - qy;
    }
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) {
        sumx += __shfl_xor(sumx, o, 64);
        sumy += __shfl_xor(sumy, o, 64);
    }
    if ((threadIdx.x & 63) == 0) {
        red[0][threadIdx.x >> 6] = sumx;
        red[1][threadIdx.x >> 6] = sumy;
    }
    __syncthreads();
    sumx = sumy = 0;
    for (int w = 0; w < 8; w++) {
        sumx += red[0][w];
        sumy += red[1][w];
    }
    const int wx0 = x0 + (int)rintf((float)sumx / 1024) - MARGIN - 1;
    const int wy0 = y0 + (int)rintf((float)sumy / 1024) - MARGIN - 1;
    const double my = gmax[0], mz = gmax[1];
    const double sy_ = my > 0 ? ldexp(1.0, kAdjFixedBits) / my : 0.0;
    const double sz_ = mz > 0 ? ldexp(1.0, kAdjFixedBits) / mz : 0.0;
#pragma unroll
    for (int j = 0; j < 2; j++) {
        if (!ok) continue;
        // unsigned: a cell anywhere in the int range falls out of the window
        const unsigned ax = (unsigned)cx[j] - 1u - (unsigned)wx0;
        const unsigned ay = (unsigned)cy[j] - 1u - (unsigned)wy0;
        const bool inx = ax < WX - 2u, in = inx && ay < WX - 2u;
#pragma unroll
        for (int a = 0; a < 3; a++) {
            const unsigned long long vy =
                (unsigned long long)llrint((double)(-gy[j] * wx[j][a]) * sy_);
            const size_t row = (size_t)wrapi(cx[j] - 1 + a, N) * N;
            if (inx)
                atomicAdd(&winy[((ax + a) * kAdjTY + ly) * TZ + lz], vy);
            else
                atomicAdd(AyI + (row + qy) * N + qz, vy);
#pragma unroll
            for (int b = 0; b < 3; b++) {
                const unsigned long long vz =
                    (unsigned long long)llrint((double)(-gz[j] * wx[j][a] * wy[j][b]) * sz_);
                if (in)
                    atomicAdd(&winz[((ax + a) * WX + ay + b) * TZ + lz], vz);
                else
                    atomicAdd(AzI + (row + wrapi(cy[j] - 1 + b, N)) * N + qz, vz);
            }
        }
    }
    __syncthreads();
    // 16 lanes a row; cells past the grid's z edge hold nothing
    for (int r = threadIdx.x >> 4; r < WX * WX; r += 32) {
        const unsigned long long v = winz[r * TZ + lz];
        if (v)
            atomicAdd(AzI + ((size_t)wrapi(wx0 + r / WX, N) * N + wrapi(wy0 + r % WX, N)) * N + qz,
                      v);
    }
    for (int r = threadIdx.x >> 4; r < WX * kAdjTY; r += 32) {
        const unsigned long long v = winy[r * TZ + lz];
        if (v)
            atomicAdd(AyI + ((size_t)wrapi(wx0 + r / kAdjTY, N) * N + y0 + r % kAdjTY) * N + qz, v);
    }
}

template <typename T>
__global__ void k_adj_fixed_to_real(const unsigned long long* __restrict__ I,
                                    const double* __restrict__ gmax, int which, T* A,
                                    long n) {
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const double m = gmax[which];
    A[i] = (T)((double)(long long)I[i] * ldexp(m, -kAdjFixedBits));
}

// k-space combine adjoint.  R_a = r2c of the displacement adjoints.  Forward:
// X_x = i kx Sx Sy Sz Phi, X_y = i ky Sy Sz Phi, X_z = i kz Sz Phi,
// Phi = W (f1 phi1 + f2 sD ip D), psi_a = c2r(X_a) / L^3.
// Writes G1 = dL/dphi1 (direct part) and GD = dL/dD / c_k (c_k = 2 inside the
// half spectrum, 1 on the z' = 0, N/2 planes), ready for the c2r that
// gives dL/ddelta2(x).
template <typename T>
__global__ void k_adj_combine(const cx<T>* __restrict__ Rx, const cx<T>* __restrict__ Ry,
                              const cx<T>* __restrict__ Rz, cx<T>* G1, cx<T>* GD, long hs, int N,
                              double dk, double boxvol, double sD, double f1, double f2,
                              const double* __restrict__ win, const double* __restrict__ S) {
    const int H = N / 2 + 1;
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (long)N * N * H) return;
    const int z = (int)(i % H);
    const long row = i / H;
    const int x = (int)(row / N), y = (int)(row % N);
    const long id = row * hs + z;
    const double kx = freq_index(x, N) * dk, ky = freq_index(y, N) * dk, kz = z * dk;
    const double k2 = kx * kx + ky * ky + kz * kz;
    const double ck = (z == 0 || z == N / 2) ? 1.0 : 2.0;
    const double Sx = S[x], Sy = S[y], Sz = S[z];
    const cx<T> rx = Rx[id], ry = Ry[id], rz = Rz[id];
    // sum_a conj(i k_a S..) R_a = -i (kx SxSySz Rx + ky SySz Ry + kz Sz Rz)
    const double ax = kx * Sx * Sy * Sz, ay = ky * Sy * Sz, az = kz * Sz;
    const double sre = ax * rx.re + ay * ry.re + az * rz.re;
    const double sim = ax * rx.im + ay * ry.im + az * rz.im;
    const double c = ck / boxvol * ((k2 > 0) ? win[x] * win[y] * win[z] : 1.0);
    const double gre = sim * c, gim = -sre * c;  // -i (sre + i sim) * c
    const double ip = (k2 > 0) ? -1.0 / k2 : 1.0;
    G1[id] = mk<T>((T)(f1 * gre), (T)(f1 * gim));
    const double d = f2 * sD * ip / ck;
    GD[id] = mk<T>((T)(d * gre), (T)(d * gim));
}

// -k_i k_j of the Hessian component q (xx, yy, zz, xy, yz, xz)
__device__ __forceinline__ double hess_factor(int q, double kx, double ky, double kz) {
    switch (q) {
        case 0: return -kx * kx;
        case 1: return -ky * ky;
        case 2: return -kz * kz;
        case 3: return -kx * ky;
        case 4: return -ky * kz;
        default: return -kx * kz;
    }
}

// x-pass operator of the Hessian c2r: phi1 -> -k_i k_j phi1
struct OpHess {
    int N, q;
    double dk;
    template <typename T>
    __device__ __forceinline__ cx<T> pre(cx<T> v, int x, int y, int z) const {
        const double f = hess_factor(q, freq_index(x, N) * dk, freq_index(y, N) * dk, z * dk);
        return mk<T>((T)(v.re * f), (T)(v.im * f));
    }
    template <typename T>
    __device__ __forceinline__ cx<T> post(cx<T> v, int, int, int) const {
        return v;
    }
};

// dL/dphi_,ij from dL/ddelta2, in place over the six recomputed phi_,ij grids
template <typename T>
__global__ void k_adj_minors(T* xx, T* yy, T* zz, T* xy, T* yz, T* xz,
                             const T* __restrict__ g, long n) {
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const T G = g[i];
    const T a = xx[i], b = yy[i], c = zz[i];
    xx[i] = G * (b + c);
    yy[i] = G * (a + c);
    zz[i] = G * (a + b);
    xy[i] = (T)-2 * G * xy[i];
    yz[i] = (T)-2 * G * yz[i];
    xz[i] = (T)-2 * G * xz[i];
}

// G1 += c_k (-k_i k_j) R / L^3
template <typename T>
__global__ void k_adj_hess_acc(cx<T>* G1, const cx<T>* __restrict__ R, long hs, int N, int q,
                               double dk, double boxvol) {
    const int H = N / 2 + 1;
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (long)N * N * H) return;
    const int z = (int)(i % H);
    const long row = i / H;
    const int x = (int)(row / N), y = (int)(row % N);
    const long id = row * hs + z;
    const double ck = (z == 0 || z == N / 2) ? 1.0 : 2.0;
    const double f = ck / boxvol * hess_factor(q, freq_index(x, N) * dk, freq_index(y, N) * dk,
                                               z * dk);
    const cx<T> r = R[id];
    cx<T> g = G1[id];
    g.re = (T)(g.re + f * r.re);
    g.im = (T)(g.im + f * r.im);
    G1[id] = g;
}

// adjoint of k_hermitian (in place): every lower-half plane point passes its
// gradient to its mirror (conjugated) and drops it; self-conjugate points
// keep the real part
template <typename T>
__global__ void k_adj_hermitian(cx<T>* f, long hs, int N) {
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    const long per = (long)(N / 2 + 1) * N;
    if (i >= 2 * per) return;
    const int z = (i < per) ? 0 : N / 2;
    const long j = i % per;
    const int x = (int)(j / N), y = (int)(j % N);
    if ((x == 0 || x == N / 2) && y > N / 2) return;
    const int invx = (x > 0) ? N - x : 0;
    const int invy = (y > 0) ? N - y : 0;
    const int invz = (z > 0) ? N - z : 0;
    const long id = ((long)x * N + y) * hs + z;
    if (invx == x && invy == y && invz == z) {
        f[id].im = 0;
    } else {
        const long mid = ((long)invx * N + invy) * hs + z;
        const cx<T> g = f[id];
        f[mid] = f[mid] + conjg(g);
        f[id] = mk<T>(0, 0);
    }
}

// dL/dnoise = sqrt(L^3/2) amp[n^2] dL/dK, into a dense N x N x (N/2+1) array
template <typename T>
__global__ void k_adj_noise(const cx<T>* __restrict__ G, long hs, cx<T>* out, int N,
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
    const cx<T> g = G[row * hs + z];
    out[i] = n2 ? mk<T>((T)(g.re * f), (T)(g.im * f)) : mk<T>(0, 0);
}

template <typename T>
static int backward(Pipe<T>* P, const mitos_ic_config& cfg, const cx<T>* noise,
                    const double* dLdP, const T* dLddelta, cx<T>* grad, hipStream_t s) {
    const int N = P->N;
    const long hs = P->hs;
    const double L = cfg.boxlen;
    const double boxvol = L * L * L;
    const double dk = 2 * M_PI / L;
    const long n3 = (long)N * N * N;
    const long nh = (long)N * N * (N / 2 + 1);
    const double sfwd = boxvol / (double)n3;
    // forward in the stencil form: K = delta(k), psi grids, positions
    MITOS_TRY(P->enqueue(cfg, s, false, nullptr, nullptr, nullptr, noise, 1));
    T* grho = reinterpret_cast<T*>(P->b(0));
    // 1. P(k) and density adjoints -> dL/drho
    if (dLdP) {
        std::vector<long long> obs(cfg.bins);
        MITOS_HIP_CHECK(hipMemcpyAsync(obs.data(), P->pk_obs, sizeof(long long) * cfg.bins,
                                       hipMemcpyDeviceToHost, s));
        MITOS_HIP_CHECK(hipStreamSynchronize(s));
        std::vector<double> coef(cfg.bins);
        for (int b = 0; b < cfg.bins; b++)
            coef[b] = obs[b] > 0 ? 2.0 * dLdP[b] / ((double)obs[b] * boxvol) : 0.0;
        double* dcoef = P->pk_sums;  // bins doubles of scratch (the sums are fetched)
        MITOS_HIP_CHECK(hipMemcpyAsync(dcoef, coef.data(), sizeof(double) * cfg.bins,
                                       hipMemcpyHostToDevice, s));
        int err = MITOS_OK;
        const int* edges = pk_bin_edges(N, L, cfg.bins, &err);
        if (!edges) return err;
        const double* w2 = window_table(N, L, 2);
        if (!w2) return MITOS_ERR_ALLOC;
        hipLaunchKernelGGL((k_adj_pk<T>), dim3(nblk(nh)), dim3(256), 0, s, P->K, hs, N, edges,
                           pk_bin_cinv(N, cfg.bins), cfg.bins, dcoef, sfwd, w2);
        MITOS_TRY(launch_status());
        MITOS_TRY((c2r_3d<T>(N, P->K, hs, P->a(0), P->a(1), hs, grho, (long)N, (T)1, OpNone(), s)));
        MITOS_HIP_CHECK(hipStreamSynchronize(s));  // dcoef is host-backed until here
    } else {
        hipLaunchKernelGGL((k_fill<T>), dim3(nblk(n3)), dim3(256), 0, s, grho, n3, (T)0);
        MITOS_TRY(launch_status());
    }
    if (dLddelta) {
        // delta = rho * N^3/npart - 1 with npart = N^3
        hipLaunchKernelGGL((k_add_real<T>), dim3(nblk(n3)), dim3(256), 0, s, grho, dLddelta, n3);
        MITOS_TRY(launch_status());
    }
    // 2. particles: CIC and TSC adjoints
    T* Ax = reinterpret_cast<T*>(P->b(1));
    T* Ay = reinterpret_cast<T*>(P->b(2));
    T* Az = reinterpret_cast<T*>(P->a(1));
    const unsigned tiles = adj_tiles(N);
    if (!P->adj_ws)
        MITOS_HIP_CHECK(hipMalloc(&P->adj_ws,
                                  sizeof(unsigned long long) * (2 * (size_t)n3 + 2 + 2 * tiles)));
    unsigned long long* AyI = P->adj_ws;
    unsigned long long* AzI = AyI + n3;
    double* gmax = reinterpret_cast<double*>(AzI + n3);
    double* part = gmax + 2;
    T* gy = reinterpret_cast<T*>(P->a(0));
    T* gz = reinterpret_cast<T*>(P->a(2));
    hipLaunchKernelGGL((k_fill<unsigned long long>), dim3(nblk(2 * n3)), dim3(256), 0, s, AyI,
                       2 * n3, 0ULL);
    hipLaunchKernelGGL((k_adj_gradients<T>), dim3(tiles), dim3(256), 0, s, P->psi(0), P->psi(1),
                       P->psi(2), (unsigned)P->prs(), grho, Ax, gy, gz, part, N, L, (float)L / N);
    hipLaunchKernelGGL(k_adj_max, dim3(1), dim3(1024), 0, s, part, tiles, gmax);
    hipLaunchKernelGGL((k_adj_scatter<T>), dim3(tiles), dim3(512), 0, s, P->psi(0), P->psi(1),
                       (unsigned)P->prs(), gy, gz, AyI, AzI, gmax, N, L, (float)L / N);
    hipLaunchKernelGGL((k_adj_fixed_to_real<T>), dim3(nblk(n3)), dim3(256), 0, s, AyI, gmax, 0,
                       Ay, n3);
    hipLaunchKernelGGL((k_adj_fixed_to_real<T>), dim3(nblk(n3)), dim3(256), 0, s, AzI, gmax, 1,
                       Az, n3);
    MITOS_TRY(launch_status());
    // 3. back to k-space: R_a = r2c(A_a)
    cx<T>* R[3] = {P->b(3), P->b(4), P->b(5)};
    T* A3[3] = {Ax, Ay, Az};
    for (int a = 0; a < 3; a++) {
        RealRowLoader<T> ld{A3[a], (long)N, 0};
        MITOS_TRY((r2c_3d<T>(N, ld, P->K, P->a(0), hs, R[a], hs, OpNone(), s)));
    }
    // 4. combine adjoint -> G1 (a1), GD (K)
    const double* win = window_table(N, L, 3);
    const double* S = smooth_table<double>(N);
    if (!win || !S) return MITOS_ERR_ALLOC;
    cx<T>* G1 = P->a(1);
    const double f2 = cfg.run2lpt ? cfg.f2 : 0.0;
    hipLaunchKernelGGL((k_adj_combine<T>), dim3(nblk(nh)), dim3(256), 0, s, R[0], R[1], R[2], G1,
                       P->K, hs, N, dk, boxvol, sfwd, cfg.f1, f2, win, S);
    MITOS_TRY(launch_status());
    if (cfg.run2lpt) {
        // 5. dL/ddelta2(x)
        T* gd2 = reinterpret_cast<T*>(P->b(0));
        MITOS_TRY((c2r_3d<T>(N, P->K, hs, P->a(0), P->a(2), hs, gd2, (long)N, (T)1, OpNone(), s)));
        // 6. recompute phi1(k) and the six phi_,ij
        const double A = amplitude_cached(cfg.n_s, cfg.gamma, cfg.sigma8);
        const double* amp = phi1_table(N, L, A, cfg.n_s, cfg.gamma);
        if (!amp) return MITOS_ERR_ALLOC;
        hipLaunchKernelGGL((k_noise_in<T>), dim3(nblk(nh)), dim3(256), 0, s, noise, P->K, hs, N,
                           L, amp);
        MITOS_TRY(launch_status());
        MITOS_TRY(launch_hermitian<T>(P->K, hs, N, s));
        T* ph[6] = {reinterpret_cast<T*>(P->b(1)), reinterpret_cast<T*>(P->b(2)),
                    reinterpret_cast<T*>(P->b(3)), reinterpret_cast<T*>(P->b(4)),
                    reinterpret_cast<T*>(P->b(5)), reinterpret_cast<T*>(P->a(2))};
        for (int q = 0; q < 6; q++)
            MITOS_TRY((c2r_3d<T>(N, P->K, hs, P->a(0), P->a(0), hs, ph[q], (long)N,
                                 (T)(1.0 / boxvol), OpHess{N, q, dk}, s)));
        // 7. Hessian-minor adjoint, then back to k-space into G1
        hipLaunchKernelGGL((k_adj_minors<T>), dim3(nblk(n3)), dim3(256), 0, s, ph[0], ph[1],
                           ph[2], ph[3], ph[4], ph[5], gd2, n3);
        MITOS_TRY(launch_status());
        for (int q = 0; q < 6; q++) {
            RealRowLoader<T> ld{ph[q], (long)N, 0};
            MITOS_TRY((r2c_3d<T>(N, ld, P->K, P->a(0), hs, P->K, hs, OpNone(), s)));
            hipLaunchKernelGGL((k_adj_hess_acc<T>), dim3(nblk(nh)), dim3(256), 0, s, G1, P->K, hs,
                               N, q, dk, boxvol);
            MITOS_TRY(launch_status());
        }
    }
    // 8. Hermitian planes and amplitude -> dL/dnoise
    hipLaunchKernelGGL((k_adj_hermitian<T>), dim3(nblk(2L * (N / 2 + 1) * N)), dim3(256), 0, s,
                       G1, hs, N);
    MITOS_TRY(launch_status());
    const double A = amplitude_cached(cfg.n_s, cfg.gamma, cfg.sigma8);
    const double* amp = phi1_table(N, L, A, cfg.n_s, cfg.gamma);
    if (!amp) return MITOS_ERR_ALLOC;
    hipLaunchKernelGGL((k_adj_noise<T>), dim3(nblk(nh)), dim3(256), 0, s, G1, hs, grad, N, L, amp);
    MITOS_TRY(launch_status());
    MITOS_HIP_CHECK(hipStreamSynchronize(s));
    return MITOS_OK;
}

}  // namespace mitos

// context internals shared with pipeline.hip
struct mitos_ic_context;
namespace mitos {
Pipe<float>* ctx_pipe_f(mitos_ic_context* c);
Pipe<double>* ctx_pipe_d(mitos_ic_context* c);
hipStream_t ctx_stream(mitos_ic_context* c);
// orders work issued next on s after the context's last realization
int ctx_order(mitos_ic_context* c, hipStream_t s);
// checks cfg against the context and records its bins and box size
int ctx_use_cfg(mitos_ic_context* c, const mitos_ic_config* cfg);
}  // namespace mitos

extern "C" int mitos_ic_noise_forward(mitos_ic_context* c, const struct mitos_ic_config* cfg,
                                      const void* noise, struct mitos_ic_result* res) {
    if (!c || !cfg || !noise) return set_last_error(MITOS_ERR_ARG);
    MITOS_TRY(set_last_error(ctx_use_cfg(c, cfg)));
    hipStream_t s = ctx_stream(c);
    MITOS_TRY(set_last_error(ctx_order(c, s)));
    int rc;
    if (ctx_pipe_f(c))
        rc = ctx_pipe_f(c)->enqueue(*cfg, s, false, nullptr, nullptr, nullptr,
                                    (const cx<float>*)noise, 1);
    else
        rc = ctx_pipe_d(c)->enqueue(*cfg, s, false, nullptr, nullptr, nullptr,
                                    (const cx<double>*)noise, 1);
    MITOS_TRY(set_last_error(rc));
    MITOS_HIP_CHECK(hipStreamSynchronize(s));
    if (res) MITOS_TRY(mitos_ic_fetch_pk(c, res));
    return MITOS_OK;
}

extern "C" int mitos_ic_noise_backward(mitos_ic_context* c, const struct mitos_ic_config* cfg,
                                       const void* noise, const double* dL_dP,
                                       const void* dL_ddelta, void* grad_noise) {
    if (!c || !cfg || !noise || !grad_noise || (!dL_dP && !dL_ddelta))
        return set_last_error(MITOS_ERR_ARG);
    MITOS_TRY(set_last_error(ctx_use_cfg(c, cfg)));
    hipStream_t s = ctx_stream(c);
    MITOS_TRY(set_last_error(ctx_order(c, s)));
    int rc;
    if (ctx_pipe_f(c))
        rc = backward<float>(ctx_pipe_f(c), *cfg, (const cx<float>*)noise, dL_dP,
                             (const float*)dL_ddelta, (cx<float>*)grad_noise, s);
    else
        rc = backward<double>(ctx_pipe_d(c), *cfg, (const cx<double>*)noise, dL_dP,
                              (const double*)dL_ddelta, (cx<double>*)grad_noise, s);
    return set_last_error(rc);
}
