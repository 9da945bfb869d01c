// CIC deposit of particles in any order (the loop of
// analyse/src/mitos_read.c:281-334) through a counting sort by output tile.
//
// One thread per particle with global atomics (k_cic) is bound by the
// memory-side atomic units, at about 20 G requests/s: eight requests per
// particle.  Here the particles are first brought to the tile of grid cells
// that owns their base cell, each tile then sums its particles in an LDS
// window, and only the window's faces, which neighbouring tiles share, go to
// the grid with atomics:
//   k_cic_count    tile of every particle and its rank in the tile
//   k_cic_scan     tile offsets
//   k_cic_scatter  positions to their tile's segment, 16 bytes per particle
//   k_cic_tile     one work-group per tile: LDS window, then the grid
// Weights and cells are those of k_cic and the sums are integers, so the grid
// has the same bits.
//
// Measured, the whole deposit with the clear and the overdensity: 30 million
// particles in random order on a 512^3 grid 11.4 -> 3.4 ms (bound by the
// counting pass's atomics in random order, 1.2 ms, then by the scattered 16-byte
// stores, 0.7 ms); 134 million in lattice order 38.4 -> 4.1 ms (bound by the LDS
// atomics and the position reads); 42.9 million in lattice order on 384^3 with
// float weights 13.3 -> 1.6 ms.
#include "cic_sort.h"

#include "fft_launch.h"
#include "particles.h"

namespace mitos {

// base cell (wrapped into the grid) and in-cell offsets of k_cic
template <typename W>
__device__ __forceinline__ void cic_sort_cell(float X, float Y, float Z, int N, double boxlen,
                                              int& x, int& y, int& z, W& dx, W& dy, W& dz) {
    if constexpr (sizeof(W) == 8)
        cic_cell(X, Y, Z, N, boxlen, x, y, z, dx, dy, dz);
    else
        cic_cell_f(X, Y, Z, N, (float)(boxlen / N), (float)(N / boxlen), boxlen, x, y, z, dx, dy,
                   dz);
    x = (unsigned)x < (unsigned)N ? x : wrapi(x, N);
    y = (unsigned)y < (unsigned)N ? y : wrapi(y, N);
    z = (unsigned)z < (unsigned)N ? z : wrapi(z, N);
}

template <typename W>
__device__ __forceinline__ unsigned cic_sort_tile(float X, float Y, float Z, double boxlen,
                                                  const CicSortDims& d) {
    int x, y, z;
    W dx, dy, dz;
    cic_sort_cell<W>(X, Y, Z, d.N, boxlen, x, y, z, dx, dy, dz);
    return ((unsigned)(x / kCicTX) * d.nty + (unsigned)(y / kCicTY)) * d.ntz +
           (unsigned)(z / kCicTZ);
}

// Place of a tile's counter: neighbouring tiles, which the work-groups that run
// at one time count into, lie in 32 different stretches of the table, not in one
// line whose atomics would queue (0.98 -> 0.60 ms per 67 million lattice
// particles on a 512^3 grid).
__device__ __forceinline__ unsigned cic_slot(unsigned tile, unsigned ntiles) {
    return (tile & 31u) * ((ntiles + 31u) >> 5) + (tile >> 5);
}

// rank[i] = index of particle i among its tile's, count[tile] += 1.  A
// work-group takes 8192 consecutive particles.  Particles in lattice or any
// other spatial order lie in a small box of tiles: the work-group counts them
// in LDS over that box and takes each tile's base with one global atomic.
// Particles in random order span too many tiles for that; then every particle
// takes its own global atomic.  (One global atomic per run of equal tiles in a
// wave instead queues at the few counters that neighbouring work-groups share.)
template <typename W>
__global__ void __launch_bounds__(512)
    k_cic_count(const float* __restrict__ X, const float* __restrict__ Y,
                const float* __restrict__ Z, unsigned n, double boxlen, CicSortDims d,
                unsigned* count, unsigned* __restrict__ rank) {
    constexpr int NT = 512, K = kCicCountBlock / NT, CAP = 8192;
    __shared__ unsigned cnt[CAP];
    __shared__ int box[6];
    const unsigned i0 = blockIdx.x * (unsigned)kCicCountBlock + threadIdx.x;
    const int lane = threadIdx.x & 63;
    if (threadIdx.x < 6) box[threadIdx.x] = threadIdx.x < 3 ? 1 << 20 : -1;
    __syncthreads();
    // tile coordinates, ten bits each (at most 4096 / 8 tiles along an axis)
    unsigned tile[K];
    int lo[3] = {1 << 20, 1 << 20, 1 << 20}, hi[3] = {-1, -1, -1};
#pragma unroll
    for (int k = 0; k < K; k++) {
        const unsigned i = i0 + NT * k;
        tile[k] = 0;
        if (i >= n) continue;
        int c[3];
        W dx, dy, dz;
        cic_sort_cell<W>(X[i], Y[i], Z[i], d.N, boxlen, c[0], c[1], c[2], dx, dy, dz);
        c[0] /= kCicTX;
        c[1] /= kCicTY;
        c[2] /= kCicTZ;
        tile[k] = ((unsigned)c[0] << 20) | ((unsigned)c[1] << 10) | (unsigned)c[2];
#pragma unroll
        for (int a = 0; a < 3; a++) {
            lo[a] = c[a] < lo[a] ? c[a] : lo[a];
            hi[a] = c[a] > hi[a] ? c[a] : hi[a];
        }
    }
#pragma unroll
    for (int a = 0; a < 3; a++) {
#pragma unroll
        for (int o = 32; o >= 1; o >>= 1) {
            const int l = __shfl_xor(lo[a], o, 64), h = __shfl_xor(hi[a], o, 64);
            lo[a] = l < lo[a] ? l : lo[a];
            hi[a] = h > hi[a] ? h : hi[a];
        }
        if (lane == 0) {
            atomicMin(&box[a], lo[a]);
            atomicMax(&box[3 + a], hi[a]);
        }
    }
    __syncthreads();
    const int bx = box[0], by = box[1], bz = box[2];
    const int ny = box[4] - by + 1, nz = box[5] - bz + 1;
    const int cells = (box[3] - bx + 1) * ny * nz;
    const bool local = cells <= CAP;
    if (local) {
        for (int c = threadIdx.x; c < cells; c += NT) cnt[c] = 0;
        __syncthreads();
    }
    // index of a tile in the box (local) or in the grid
    auto index = [&](unsigned t) -> unsigned {
        const unsigned x = t >> 20, y = (t >> 10) & 1023u, z = t & 1023u;
        return local ? ((x - bx) * ny + (y - by)) * nz + (z - bz)
                     : (x * (unsigned)d.nty + y) * (unsigned)d.ntz + z;
    };
    unsigned at[K];
    if (local) {
#pragma unroll
        for (int k = 0; k < K; k++)
            if (i0 + NT * k < n) at[k] = atomicAdd(&cnt[index(tile[k])], 1u);
    } else {
#pragma unroll
        for (int k = 0; k < K; k++)
            if (i0 + NT * k < n) at[k] = atomicAdd(count + cic_slot(index(tile[k]), d.ntiles), 1u);
    }
    if (local) {
        __syncthreads();
        for (int c = threadIdx.x; c < cells; c += NT)
            if (cnt[c]) {
                const unsigned x = c / (ny * nz), y = c / nz % ny, z = c % nz;
                const unsigned t = ((bx + x) * (unsigned)d.nty + (by + y)) * (unsigned)d.ntz +
                                   (bz + z);
                cnt[c] = atomicAdd(count + cic_slot(t, d.ntiles), cnt[c]);
            }
        __syncthreads();
    }
#pragma unroll
    for (int k = 0; k < K; k++)
        if (i0 + NT * k < n) rank[i0 + NT * k] = at[k] + (local ? cnt[index(tile[k])] : 0u);
}

template <typename W, int K>
__global__ void __launch_bounds__(256)
    k_cic_scatter(const float* __restrict__ X, const float* __restrict__ Y,
                  const float* __restrict__ Z, unsigned n, double boxlen, CicSortDims d,
                  const unsigned* __restrict__ offs, const unsigned* __restrict__ rank,
                  float4* __restrict__ sorted) {
    const unsigned i0 = blockIdx.x * (256u * K) + threadIdx.x;
    float px[K], py[K], pz[K];
    unsigned r[K];
#pragma unroll
    for (int k = 0; k < K; k++) {
        const unsigned i = i0 + 256u * k;
        px[k] = i < n ? X[i] : 0.0f;
        py[k] = i < n ? Y[i] : 0.0f;
        pz[k] = i < n ? Z[i] : 0.0f;
        r[k] = i < n ? rank[i] : 0;
    }
#pragma unroll
    for (int k = 0; k < K; k++)
        r[k] += offs[cic_sort_tile<W>(px[k], py[k], pz[k], boxlen, d)];
#pragma unroll
    for (int k = 0; k < K; k++)
        if (i0 + 256u * k < n) sorted[r[k]] = make_float4(px[k], py[k], pz[k], 0.0f);
}

// One work-group per tile, or several (gridDim.y) that share a tile's particles
// where the tiles are few or full.  A window cell whose three coordinates lie
// strictly inside the tile receives mass from this tile alone: it is stored
// (`store`: one work-group per tile, first pass over a cleared grid); the
// others are added with atomics.
template <typename W>
__global__ void __launch_bounds__(512)
    k_cic_tile(const float4* __restrict__ sorted, const unsigned* __restrict__ offs,
               double boxlen, CicSortDims d, bool store, unsigned long long* grid) {
    constexpr int WY = kCicTY + 1, WZ = kCicTZ + 1, ROWS = (kCicTX + 1) * WY, R = ROWS * WZ;
    __shared__ unsigned long long win[R];
    const unsigned q0 = offs[blockIdx.x], q1 = offs[blockIdx.x + 1];
    const unsigned share = (q1 - q0 + gridDim.y - 1) / gridDim.y;
    const unsigned p0 = q0 + blockIdx.y * share, p1 = p0 + share < q1 ? p0 + share : q1;
    if (p0 >= p1) return;
    const int N = d.N;
    const int tz = (int)(blockIdx.x % (unsigned)d.ntz);
    const int ty = (int)(blockIdx.x / (unsigned)d.ntz % (unsigned)d.nty);
    const int tx = (int)(blockIdx.x / ((unsigned)d.ntz * d.nty));
    const int ox = tx * kCicTX, oy = ty * kCicTY, oz = tz * kCicTZ;
    for (int c = threadIdx.x; c < R; c += 512) win[c] = 0;
    __syncthreads();
    float4 next = make_float4(0, 0, 0, 0);
    if (p0 + threadIdx.x < p1) next = sorted[p0 + threadIdx.x];
    for (unsigned p = p0 + threadIdx.x; p < p1; p += 512) {
        const float4 q = next;
        if (p + 512 < p1) next = sorted[p + 512];
        int x, y, z;
        W dx, dy, dz;
        cic_sort_cell<W>(q.x, q.y, q.z, N, boxlen, x, y, z, dx, dy, dz);
        unsigned long long w[8];
        cic_weights(dx, dy, dz, w);
        unsigned long long* b = win + ((x - ox) * WY + (y - oy)) * WZ + (z - oz);
        constexpr int off[8] = {0,           WY * WZ,     WZ,     1,
                                WY * WZ + WZ, WY * WZ + 1, WZ + 1, WY * WZ + WZ + 1};
#pragma unroll
        for (int c = 0; c < 8; c++) atomicAdd(b + off[c], w[c]);
    }
    __syncthreads();
    // cells of the tile: fewer than its size in the last tile of an axis
    const int ex = N - ox < kCicTX ? N - ox : kCicTX, ey = N - oy < kCicTY ? N - oy : kCicTY,
              ez = N - oz < kCicTZ ? N - oz : kCicTZ;
    const int lane = threadIdx.x & 63;
    for (int r = threadIdx.x >> 6; r < ROWS; r += 8) {
        const int wx = r / WY, wy = r - wx * WY;
        if (wx > ex || wy > ey) continue;
        const int gx = ox + wx == N ? 0 : ox + wx, gy = oy + wy == N ? 0 : oy + wy;
        unsigned long long* row = grid + ((size_t)gx * N + gy) * N;
        const bool inside = store && wx > 0 && wx < ex && wy > 0 && wy < ey;
        const unsigned long long v = lane <= ez ? win[r * WZ + lane] : 0;
        const int gz = oz + lane >= N ? 0 : oz + lane;
        if (v) {
            if (inside && lane > 0 && lane < ez)
                row[gz] = v;
            else
                atomicAdd(row + gz, v);
        }
        if (lane == 0 && ez == kCicTZ) {
            const unsigned long long e = win[r * WZ + kCicTZ];
            if (e) atomicAdd(row + (oz + kCicTZ == N ? 0 : oz + kCicTZ), e);
        }
    }
}

// offs[t] = sum of count[0..t), offs[ntiles] = n; the counts return to zero.
// One work-group; the next 4096 counts load while the current ones are summed.
static __global__ void __launch_bounds__(1024)
    k_cic_scan(unsigned* count, unsigned* __restrict__ offs, unsigned ntiles) {
    __shared__ unsigned wsum[16];
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    unsigned carry = 0;
    auto load = [&](unsigned b, unsigned v[4]) {
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const unsigned i = b + threadIdx.x * 4 + k;
            v[k] = i < ntiles ? count[cic_slot(i, ntiles)] : 0;
        }
    };
    unsigned nxt[4];
    load(0, nxt);
    for (unsigned b = 0; b < ntiles; b += 4096) {
        unsigned v[4];
#pragma unroll
        for (int k = 0; k < 4; k++) v[k] = nxt[k];
        if (b + 4096 < ntiles) load(b + 4096, nxt);
        unsigned own = v[0] + v[1] + v[2] + v[3], incl = own;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const unsigned u = __shfl_up(incl, o, 64);
            if (lane >= o) incl += u;
        }
        if (lane == 63) wsum[wv] = incl;
        __syncthreads();
        unsigned before = carry, total = 0;
        for (int w = 0; w < 16; w++) {
            const unsigned u = wsum[w];
            if (w < wv) before += u;
            total += u;
        }
        unsigned at = before + incl - own;
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const unsigned i = b + threadIdx.x * 4 + k;
            if (i < ntiles) {
                offs[i] = at;
                count[cic_slot(i, ntiles)] = 0;
            }
            at += v[k];
        }
        carry += total;
        __syncthreads();  // wsum is read before the next round writes it
    }
    if (threadIdx.x == 0) offs[ntiles] = carry;
}

static __global__ void k_zero_u32(unsigned* p, unsigned n) {
    const unsigned i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = 0;
}

template <typename W>
int cic_sorted(const float* X, const float* Y, const float* Z, long long npart, int N,
               double boxlen, unsigned long long* grid, void* ws, size_t ws_bytes,
               hipStream_t s) {
    const CicSortDims d = cic_sort_dims(N);
    const size_t tables = cic_sort_tables(N);
    if (!ws || ws_bytes < tables + 1024 * kCicSortParticle) return MITOS_ERR_ARG;
    long long per = (long long)((ws_bytes - tables) / kCicSortParticle);
    if (per > kCicSortPass) per = kCicSortPass;
    unsigned* count = static_cast<unsigned*>(ws);
    unsigned* offs = count + (d.ntiles + 31) / 32 * 32;
    float4* sorted = reinterpret_cast<float4*>(static_cast<char*>(ws) + tables);
    unsigned* rank = reinterpret_cast<unsigned*>(sorted + per);
    hipLaunchKernelGGL(k_zero_u32, dim3((d.ntiles + 287) / 256), dim3(256), 0, s, count,
                       (d.ntiles + 31) / 32 * 32);
    for (long long p0 = 0; p0 < npart; p0 += per) {
        const unsigned n = (unsigned)(npart - p0 < per ? npart - p0 : per);
        constexpr int K = 4;
        const unsigned blocks = (n + 256 * K - 1) / (256 * K);
        hipLaunchKernelGGL((k_cic_count<W>), dim3((n + kCicCountBlock - 1) / kCicCountBlock),
                           dim3(512), 0, s, X + p0, Y + p0, Z + p0, n, boxlen, d, count, rank);
        hipLaunchKernelGGL(k_cic_scan, dim3(1), dim3(1024), 0, s, count, offs, d.ntiles);
        hipLaunchKernelGGL((k_cic_scatter<W, K>), dim3(blocks), dim3(256), 0, s, X + p0, Y + p0,
                           Z + p0, n, boxlen, d, offs, rank, sorted);
        // about 8192 particles per work-group
        const unsigned share = n / d.ntiles / 8192 + 1 < 64 ? n / d.ntiles / 8192 + 1 : 64;
        hipLaunchKernelGGL((k_cic_tile<W>), dim3(d.ntiles, share), dim3(512), 0, s, sorted, offs,
                           boxlen, d, p0 == 0 && share == 1, grid);
    }
    return launch_status();
}

template int cic_sorted<float>(const float*, const float*, const float*, long long, int, double,
                               unsigned long long*, void*, size_t, hipStream_t);
template int cic_sorted<double>(const float*, const float*, const float*, long long, int, double,
                                unsigned long long*, void*, size_t, hipStream_t);

}  // namespace mitos
