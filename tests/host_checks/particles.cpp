// Host entry points to the index and weight arithmetic of
// mitos_amd/csrc/particles.h, for tests that need no GPU.
#include <math.h>

#include "../../mitos_amd/csrc/particles.h"

using namespace mitos;

namespace {

template <typename W>
void add_cloud(int N, const int i[3], const W d[3], unsigned long long* grid) {
    unsigned long long w[8];
    cic_weights(d[0], d[1], d[2], w);
    const int corner[8][3] = {{0, 0, 0}, {1, 0, 0}, {0, 1, 0}, {0, 0, 1},
                              {1, 1, 0}, {1, 0, 1}, {0, 1, 1}, {1, 1, 1}};
    for (int c = 0; c < 8; c++)
        grid[((size_t)wrapi(i[0] + corner[c][0], N) * N + wrapi(i[1] + corner[c][1], N)) * N +
             wrapi(i[2] + corner[c][2], N)] += w[c];
}

template <typename W>
void deposit(int N, double L, long n, const float* X, const float* Y, const float* Z,
             unsigned long long* grid) {
    for (long k = 0; k < n; k++) {
        int i[3];
        W d[3];
        if constexpr (sizeof(W) == 8)
            cic_cell(X[k], Y[k], Z[k], N, L, i[0], i[1], i[2], d[0], d[1], d[2]);
        else
            cic_cell_f(X[k], Y[k], Z[k], N, (float)(L / N), (float)(N / L), L, i[0], i[1], i[2],
                       d[0], d[1], d[2]);
        add_cloud(N, i, d, grid);
    }
}

}  // namespace

extern "C" {

// the fixed-point CIC sums of particles in any order, one after the other
void check_deposit_f(int N, double L, long n, const float* X, const float* Y, const float* Z,
                     unsigned long long* grid) {
    deposit<float>(N, L, n, X, Y, Z, grid);
}
void check_deposit_d(int N, double L, long n, const float* X, const float* Y, const float* Z,
                     unsigned long long* grid) {
    deposit<double>(N, L, n, X, Y, Z, grid);
}

void check_wrapf(int N, long n, const int* i, int* out) {
    for (long k = 0; k < n; k++) out[k] = wrapf(i[k], N, 1.0f / N);
}

// the deposit's base index (site + periodic offset) of positions along one axis
void check_lattice_cell_f(int N, double L, long n, int site, const float* x, int* base) {
    for (long k = 0; k < n; k++) {
        const float p = wrap_pos(x[k], (float)L);
        int rx, ry, rz;
        float fx, fy, fz;
        cic_lattice_cell<float, true>(p, p, p, N, L, 0.0f, 0.0f, site, site, site, rx, ry, rz, fx,
                                      fy, fz);
        base[k] = site + rx;
    }
}
void check_lattice_cell_d(int N, double L, long n, int site, const double* x, int* base) {
    for (long k = 0; k < n; k++) {
        const double p = wrap_pos(x[k], L);
        int rx, ry, rz;
        double fx, fy, fz;
        cic_lattice_cell<double, true>(p, p, p, N, L, 0.0f, 0.0f, site, site, site, rx, ry, rz,
                                       fx, fy, fz);
        base[k] = site + rx;
    }
}

// the same with the cells of the FP32 adjoint
void check_deposit_t(int N, double L, long n, const float* X, const float* Y, const float* Z,
                     unsigned long long* grid) {
    for (long k = 0; k < n; k++) {
        int i[3];
        float d[3];
        cic_cell_t(X[k], (float)(N / L), N, i[0], d[0]);
        cic_cell_t(Y[k], (float)(N / L), N, i[1], d[1]);
        cic_cell_t(Z[k], (float)(N / L), N, i[2], d[2]);
        add_cloud(N, i, d, grid);
    }
}

// in-cell offset of positions along one axis, and the fixed-point mass of a
// particle with that offset on all three
void check_cell_mass(int N, double L, long n, const float* x, float* d,
                     unsigned long long* mass) {
    for (long k = 0; k < n; k++) {
        int i;
        cic_cell_t(wrap_pos(x[k], (float)L), (float)(N / L), N, i, d[k]);
        unsigned long long w[8];
        cic_weights(d[k], d[k], d[k], w);
        mass[k] = 0;
        for (int c = 0; c < 8; c++) mass[k] += w[c];
    }
}

// TSC cells and weights: the reference's formulas and the kernels' short form
void check_tsc_axis(long n, const double* x, int* i, double* w) {
    for (long k = 0; k < n; k++) tsc_axis(x[k], i[k], w + 3 * k);
}
void check_tsc_axis_short(long n, const double* x, int* i, double* w) {
    for (long k = 0; k < n; k++) tsc_axis_short(x[k], i[k], w + 3 * k);
}

}  // extern "C"
