// CIC deposit of particles in any order through a counting sort by output tile
// (cic_sort.hip).
#pragma once

#include "mitos_common.h"

namespace mitos {

// Tile of 8 x 8 x 64 cells, long in z as the grid rows are: a window row of 64
// cells is 512 contiguous bytes of the grid, and particles that follow each
// other along z mostly share a tile.  The window (9 x 9 x 65 words of 64 bits,
// 42 KB) leaves three work-groups per CU.
constexpr int kCicTX = 8, kCicTY = 8, kCicTZ = 64;
// particles of one work-group of the counting pass
constexpr int kCicCountBlock = 8192;

struct CicSortDims {
    int N, nty, ntz;
    unsigned ntiles;
};
inline CicSortDims cic_sort_dims(int N) {
    const int nx = (N + kCicTX - 1) / kCicTX, ny = (N + kCicTY - 1) / kCicTY,
              nz = (N + kCicTZ - 1) / kCicTZ;
    return CicSortDims{N, ny, nz, (unsigned)nx * ny * nz};
}

// bytes per particle of a pass and bytes of the tile tables in the workspace
constexpr size_t kCicSortParticle = sizeof(float4) + sizeof(unsigned);
inline size_t cic_sort_tables(int N) {
    const size_t nt = cic_sort_dims(N).ntiles;
    return (2 * nt + 96) * sizeof(unsigned) / 64 * 64 + 64;
}
// particles of one pass: the sort's buffers stay under 1.4 GB whatever the call
constexpr long long kCicSortPass = 1LL << 26;
inline size_t cic_sort_bytes(int N, long long npart) {
    return cic_sort_tables(N) + (size_t)(npart < kCicSortPass ? npart : kCicSortPass) *
                                    kCicSortParticle;
}

// Deposit npart particles into a cleared grid, in passes of as many particles
// as ws_bytes holds.
template <typename W>
int cic_sorted(const float* X, const float* Y, const float* Z, long long npart, int N,
               double boxlen, unsigned long long* grid, void* ws, size_t ws_bytes,
               hipStream_t s);

// Whether the sort is the faster deposit.  Its five launches and the visit to
// every tile cost about 60 us; the atomics take about 0.36 us per thousand
// particles in random order and half of that in lattice order.  Measured on a
// 64^3 grid, sorted against atomics: 262144 particles 72 against 46 us (lattice
// order) and 66 against 111 us (random), 10^6 particles 101 against 214 and 94
// against 364 us.
inline bool cic_sort_pays(int N, long long npart) {
    return N <= 4096 && npart >= 524288 && npart >= (long long)cic_sort_dims(N).ntiles;
}

}  // namespace mitos
