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

// Whether the sort is the faster deposit with a workspace of ws_bytes.  A pass of up
// to its capacity is four launches (40 to 60 us on small grids), and every tile that
// holds particles clears and flushes its window (about 8 ns of the whole deposit); the
// atomics take about 0.36 us per thousand particles in random order, 0.07 to 0.2 in
// lattice order and more on grids below 64^3.  So a pass holds 524288 particles or
// more, the deposit 200 a tile, the figure at which lattice order breaks even (random
// order at about 30; the order is not known here).  mitos_cic_overdensity, atomics
// against sorted, lattice order / random:
//    64^3, 600000           134,   76 / 231,   72 us     (9375 a tile)
//   256^3, 600000           160,  177 / 290,  186 us     (146)
//   256^3, 1000000          195,  186 / 424,  219 us     (244)
//   512^3, 4000000         1130, 1243 / 2087, 1299 us    (122)
//   512^3, 16000000        2115, 1914 / 6479, 2423 us    (488)
//  1024^3, 600000          4655, 5550 / 4692, 6296 us    (2)
//  1024^3, 30000000        8977, 9640 / 16253, 10245 us  (114)
// and the FP32 realization of 128^3 particles on 16^3, where the displacement grids
// hold 4890 particles a pass: 2.6, 16.4 ms.
inline bool cic_sort_pays(int N, long long npart, size_t ws_bytes) {
    if (N > 4096 || ws_bytes < cic_sort_tables(N)) return false;
    const long long tiles = cic_sort_dims(N).ntiles;
    const long long room = (long long)((ws_bytes - cic_sort_tables(N)) / kCicSortParticle);
    const long long most = room < kCicSortPass ? room : kCicSortPass;
    const long long pass = npart < most ? npart : most;
    return pass >= 524288 && pass >= 32 * tiles && npart >= 200 * tiles;
}

}  // namespace mitos
