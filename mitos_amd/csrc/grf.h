// Gaussian random field: white noise from the xoshiro256** stream in the
// reference's draw order, with a k-dependent amplitude fused in.
#pragma once

#include "crmath.h"
#include "rng.h"

namespace mitos {

// A thread draws a segment of consecutive modes of the half grid (in the dense
// mode order): whole z-rows, or in FP64 below 256^3 pieces of 4 to 16 modes, where
// one thread per row leaves most of the chip idle (64^3 has 4096 rows, 16
// work-groups) and the correctly rounded normals make a long serial chain.  The
// shorter the segments, the more start states; each size class has the length
// that keeps about 10^5 threads.  generate_complex_grf, rows against segments: 64^3
// 128 -> 54 us, 96^3 166 -> 68 us, 128^3 206 -> 102 us, 192^3 291 -> 201 us; at
// 256^3 segments of 16 take 413 us, rows 388 us.  The FP32 draws are so short that a segment's
// start state would cost more than it (the ensemble of 96: 54.6 -> 57.8 ms).
inline int noise_segment(int N, bool fp64) {
    return !fp64 || N >= 256 ? N / 2 + 1 : N > 160 ? 16 : N > 96 ? 8 : 4;
}

// Per-grid-size jump data, resident on the device; S = noise_segment.
struct NoiseJumps {
    const uint64_t* tab;  // nbits matrices J^(2^b), J = T^(4 S), 256*4 words each
    int nbits;
    // four draws before the first: the state of the stream with the DC mode's
    // draws, which the reference does not take, so segment q starts at J^q base
    Xo base;
};

// Host: jump data for grid size N starting from state s0 (table cached).
int noise_jumps(int N, bool fp64, const Xo& s0, NoiseJumps* out);
// Host: state after the whole grid's draws, 4*(N*N*(N/2+1) - 1).
int noise_advance(int N, Xo* st);

// x * 2^s + x, written so that it stays one shift-add (v_lshl_add_u64): the
// empty asm hides that both operands are x, so the compiler cannot fold the
// sum back into a 64-bit multiply (two v_mad_u64_u32)
__device__ __forceinline__ uint64_t shl_add64(uint64_t x, int s) {
    uint64_t y = x;
    asm("" : "+v"(y));
    return (y << s) + x;
}

// 64-bit rotations and the shift by 17 on 32-bit halves with v_alignbit_b32
// (alignbit(a, b, c) = low word of ((a:b) >> c)): two instructions each
template <int K>
__device__ __forceinline__ uint64_t rotl64_dev(uint64_t x) {
    static_assert(K > 0 && K < 64 && K != 32, "rotation");
    const unsigned lo = (unsigned)x, hi = (unsigned)(x >> 32);
    unsigned nlo, nhi;
    if constexpr (K < 32) {
        nhi = __builtin_amdgcn_alignbit(hi, lo, 32 - K);
        nlo = __builtin_amdgcn_alignbit(lo, hi, 32 - K);
    } else {
        nhi = __builtin_amdgcn_alignbit(lo, hi, 64 - K);
        nlo = __builtin_amdgcn_alignbit(hi, lo, 64 - K);
    }
    return ((uint64_t)nhi << 32) | nlo;
}
template <int K>
__device__ __forceinline__ uint64_t shl64_dev(uint64_t x) {
    static_assert(K > 0 && K < 32, "shift");
    const unsigned lo = (unsigned)x, hi = (unsigned)(x >> 32);
    return ((uint64_t)__builtin_amdgcn_alignbit(hi, lo, 32 - K) << 32) | (lo << K);
}

// xo_next on the device: the same draw, with s1 * 5 and r * 9 as shift-adds
// and the rotations and shift on 32-bit halves
__device__ __forceinline__ uint64_t xo_next_dev(Xo& st) {
    const uint64_t out = shl_add64(rotl64_dev<7>(shl_add64(st.s[1], 2)), 3);
    const uint64_t t = shl64_dev<17>(st.s[1]);
    st.s[2] ^= st.s[0];
    st.s[3] ^= st.s[1];
    st.s[1] ^= st.s[2];
    st.s[0] ^= st.s[3];
    st.s[2] ^= t;
    st.s[3] = rotl64_dev<45>(st.s[3]);
    return out;
}

// Start states of the 256 segments line0 + t of a 256-thread work-group (line0
// a multiple of 256), by the whole work-group.  A product M v of a jump
// matrix and a state takes one parity per thread (output bit t = parity of
// row t of M and v) and a ballot per wave (wave w holds word w).  The
// work-group advances J.base to segment line0 (the matrices of the bits of line0,
// all above bit 7), then doubles: st[j + 2^k] = J^(2^k) st[j] for k < 8, so thread
// t reads its segment's state st[t].  That is 255 + up to 20 products shared by
// 256 segments, against up to 20 per segment when every thread jumps on its own.
// The products of a doubling are independent: four are in flight.  lds: 256 * 4 +
// 4 words.
__device__ __forceinline__ Xo block_row_start(const NoiseJumps& J, long line0, uint64_t* lds) {
    uint64_t(*st)[4] = reinterpret_cast<uint64_t(*)[4]>(lds);
    uint64_t* xw = lds + 256 * 4;
    const int t = threadIdx.x, lane = t & 63, wv = t >> 6;
    Xo v = J.base;
    for (int b = 8; b < J.nbits; b++) {
        if (!((line0 >> b) & 1)) continue;
        const uint64_t* row = J.tab + (size_t)b * 1024 + (size_t)t * 4;
        const uint64_t p = (row[0] & v.s[0]) ^ (row[1] & v.s[1]) ^ (row[2] & v.s[2]) ^
                           (row[3] & v.s[3]);
        const uint64_t w = __ballot(__builtin_popcountll(p) & 1);
        if (lane == 0) xw[wv] = w;
        __syncthreads();
        v = Xo{{xw[0], xw[1], xw[2], xw[3]}};
        __syncthreads();
    }
    if (t < 4) st[0][t] = v.s[t];
    __syncthreads();
    for (int k = 0; k < 8 && k < J.nbits; k++) {
        const int m = 1 << k;
        const uint64_t* row = J.tab + (size_t)k * 1024 + (size_t)t * 4;
        const uint64_t r0 = row[0], r1 = row[1], r2 = row[2], r3 = row[3];
        for (int j0 = 0; j0 < m; j0 += 4) {
            uint64_t p[4];
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const uint64_t* s = st[j0 + j < m ? j0 + j : 0];
                p[j] = (r0 & s[0]) ^ (r1 & s[1]) ^ (r2 & s[2]) ^ (r3 & s[3]);
            }
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const uint64_t w = __ballot(__builtin_popcountll(p[j]) & 1);
                if (lane == 0 && j0 + j < m) st[j0 + j + m][wv] = w;
            }
        }
        __syncthreads();
    }
    const Xo r = Xo{{st[t][0], st[t][1], st[t][2], st[t][3]}};
    __syncthreads();  // the table's reads precede the caller's reuse of lds
    return r;
}

// src/random.c:34-49: cosine branch of Box-Muller from two 64-bit draws.
// CR: correctly rounded log/cos (bit-exact Gaussians); else the device libm
// (within an ulp, used when the result is rounded to float anyway).
template <bool CR = true>
__device__ __forceinline__ double bm_normal(Xo& gen) {
    const uint64_t A = xo_next_dev(gen);
    const uint64_t B = xo_next_dev(gen);
    const double RMax = 18446744073709551616.0;  // (double)UINT64_MAX + 1 = 2^64
    const double u = ((double)A + 0.5) / RMax;
    const double v = ((double)B + 0.5) / RMax;
    if (CR) return sqrt(-2 * cr_log(u)) * cr_cos(2 * M_PI * v);
    return sqrt(-2 * log(u)) * cos(2 * M_PI * v);
}

// cos(2 pi v) in float for v in [0, 1): r = v - rint(v) is exact, t = |r|
// (or 1/2 - |r| past a quarter period, with the sign flipped) lies in
// [0, 1/4], and cos(2 pi t) is a degree-10 even polynomial in t fitted here
// (weighted least squares on Chebyshev nodes, iterated towards equal ripple;
// fit error 2.2e-10, float evaluation within 1.4e-7 of cos(2 pi v))
__device__ __forceinline__ float cos2pi_f(float v) {
    const float r = v - rintf(v);
    const float s = fabsf(r);
    const bool far = s > 0.25f;
    const float t = far ? 0.5f - s : s;
    const float t2 = t * t;
    float p = -24.982326173851263f;
    p = fmaf(p, t2, 60.14403025957297f);
    p = fmaf(p, t2, -85.45357257295981f);
    p = fmaf(p, t2, 64.9393466552905f);
    p = fmaf(p, t2, -19.73920854920032f);
    p = fmaf(p, t2, 0.9999999997815415f);
    return far ? -p : p;
}

// The Box-Muller pair of bm_normal in float arithmetic (FP32 pipeline): the
// same draws; the 64-bit words become floats as hi * 2^32 + lo with one
// rounding (within an ulp of the rounded word), then log, the hardware square
// root (an ulp) and cos2pi_f.
__device__ __forceinline__ float u64_to_float(uint64_t A) {
    // the empty asm keeps the high word a 32-bit value, so its conversion is
    // one v_cvt_f32_u32 rather than a 64-bit integer conversion
    unsigned hi = (unsigned)(A >> 32);
    asm("" : "+v"(hi));
    return fmaf((float)hi, 4294967296.0f, (float)(unsigned)A);
}
__device__ __forceinline__ float bm_normal_f(Xo& gen) {
    const uint64_t A = xo_next_dev(gen);
    const uint64_t B = xo_next_dev(gen);
    const float s = 5.42101086242752217e-20f;  // 2^-64
    const float u = (u64_to_float(A) + 0.5f) * s;
    const float v = (u64_to_float(B) + 0.5f) * s;
    return __builtin_amdgcn_sqrtf(-2.0f * logf(u)) * cos2pi_f(v);
}

// src/fft.c:29-35, evaluated without contraction so k matches the host bits
__host__ __device__ __forceinline__ void wavevec(int x, int y, int z, int N, double dk,
                                                 double& kx, double& ky, double& kz,
                                                 double& k) {
#pragma clang fp contract(off)
    kx = (x > N / 2) ? (x - N) * dk : x * dk;
    ky = (y > N / 2) ? (y - N) * dk : y * dk;
    kz = (z > N / 2) ? (z - N) * dk : z * dk;
    k = sqrt(kx * kx + ky * ky + kz * kz);
}

// one mode: two normals times sqrt(L^3/2) = factor and the amplitude of n^2
template <typename T, bool CR, typename AMP>
__device__ __forceinline__ cx<T> grf_mode(Xo& gen, const AMP& amp, long n2, double factor) {
    if constexpr (sizeof(T) == 4) {
        const float ga = bm_normal_f(gen);
        const float gb = bm_normal_f(gen);
        float fm;
        if constexpr (AMP::prescaled)
            fm = amp.f(n2);  // (float)(factor * amp) made on the host
        else
            fm = (float)(factor * amp(n2));
        return mk<T>(ga * fm, gb * fm);
    } else {
        const double a = bm_normal<CR>(gen) * factor;
        const double b = bm_normal<CR>(gen) * factor;
        const double m = amp(n2);
        return mk<T>((T)(a * m), (T)(b * m));
    }
}

// src/grf.c:26-69 with an amplitude amp(n2) applied to both parts (n2 =
// integer |k|^2 / dk^2).  One thread walks one z-row in stream
// order; a block's 256 rows are staged through LDS in chunks of 16 modes so
// the stores are 16-mode contiguous runs.
template <typename T, typename AMP, bool CR>
__global__ void __launch_bounds__(256)
    k_grf(cx<T>* out, long hs, int N, double boxlen, NoiseJumps J, AMP amp) {
    constexpr int ZC = 16;
    __shared__ cx<T> stage[256 * ZC];
    const long nrows = (long)N * N;
    const long line0 = (long)blockIdx.x * 256;
    const long line = line0 + threadIdx.x;
    const bool ok = line < nrows;
    const int x = (int)(line / N), y = (int)(line % N);
    Xo gen = block_row_start(J, line0, reinterpret_cast<uint64_t*>(stage));
    const double boxvol = boxlen * boxlen * boxlen;
    const double factor = sqrt(boxvol / 2);
    const int H = N / 2 + 1;
    // stored z': the modes, and the row padding up to a whole chunk (zeros),
    // so the last chunk writes whole 128-byte lines
    const long hz = (long)(H + ZC - 1) / ZC * ZC;
    const int WZ = (int)(hz < hs ? hz : hs);
    const int nx = freq_index(x, N), ny = freq_index(y, N);
    const long n2xy = (long)nx * nx + (long)ny * ny;
    for (int z0 = 0; z0 < H; z0 += ZC) {
        if (ok) {
            for (int dz = 0; dz < ZC; dz++) {
                const int z = z0 + dz;
                // past the last mode: zeros for the row padding
                if (z >= H) {
                    stage[threadIdx.x * ZC + dz] = mk<T>(0, 0);
                    continue;
                }
                // the DC mode is zero; its place in the stream lies before the
                // reference's first draw
                const long n2 = n2xy + (long)z * z;
                cx<T> val = mk<T>(0, 0);
                if (n2 > 0)
                    val = grf_mode<T, CR>(gen, amp, n2, factor);
                else
                    for (int d = 0; d < 4; d++) (void)xo_next_dev(gen);
                stage[threadIdx.x * ZC + dz] = val;
            }
        }
        __syncthreads();
        for (int i = 0; i < ZC; i++) {
            const int idx = i * 256 + threadIdx.x;
            const int r = idx / ZC, dz = idx % ZC;
            const long l = line0 + r;
            if (l < nrows && z0 + dz < WZ) st(out + l * hs + z0 + dz, stage[r * ZC + dz]);
        }
        __syncthreads();
    }
}

// k_grf with a segment of S modes per thread (grids below 256^3: the float
// quotient of a mode index is within one of its row).  The work-group's modes are
// consecutive; they are staged in LDS up to eight modes of every thread at a time
// and stored as runs of that length.
template <typename T, int S, typename AMP, bool CR>
__global__ void __launch_bounds__(256)
    k_grf_segments(cx<T>* out, long hs, int N, double boxlen, NoiseJumps J, AMP amp) {
    constexpr int ZC = S < 8 ? S : 8;
    static_assert(S % ZC == 0, "segments are whole chunks");
    __shared__ __align__(16) cx<T> stage[256 * ZC > 1028 * 8 / (int)sizeof(cx<T>)
                                             ? 256 * ZC
                                             : 1028 * 8 / (int)sizeof(cx<T>)];
    const int H = N / 2 + 1;
    const unsigned modes = (unsigned)N * N * H;
    const unsigned line0 = blockIdx.x * 256u;
    Xo gen = block_row_start(J, (long)line0, reinterpret_cast<uint64_t*>(stage));
    const double factor = sqrt(boxlen * boxlen * boxlen / 2);
    const float invH = 1.0f / H;
    // row and z' of a mode
    auto split = [&](unsigned m, int& row, int& z) {
        row = (int)((float)m * invH);
        z = (int)m - row * H;
        if (z < 0) {
            row--;
            z += H;
        } else if (z >= H) {
            row++;
            z -= H;
        }
    };
    const unsigned m0 = (line0 + threadIdx.x) * (unsigned)S;
    int row, z;
    split(m0, row, z);
    int x = row / N, y = row - x * N;
    int nx = freq_index(x, N), ny = freq_index(y, N), n2xy = nx * nx + ny * ny;
    const int hz = (H + 15) / 16 * 16 < hs ? (H + 15) / 16 * 16 : (int)hs;
    for (int c = 0; c < S; c += ZC) {
        for (int d = 0; d < ZC; d++) {
            const int n2 = n2xy + z * z;
            cx<T> val = mk<T>(0, 0);
            // the DC mode is zero; its place in the stream lies before the
            // reference's first draw
            if (m0 + c + d < modes) {
                if (n2 > 0)
                    val = grf_mode<T, CR>(gen, amp, n2, factor);
                else
                    for (int q = 0; q < 4; q++) (void)xo_next_dev(gen);
            }
            stage[threadIdx.x * ZC + d] = val;
            if (++z == H) {
                z = 0;
                if (++y == N) {
                    y = 0;
                    x++;
                }
                nx = freq_index(x, N);
                ny = freq_index(y, N);
                n2xy = nx * nx + ny * ny;
            }
        }
        __syncthreads();
#pragma unroll
        for (int i = 0; i < ZC; i++) {
            const unsigned idx = i * 256u + threadIdx.x;
            const unsigned m = (line0 + idx / ZC) * (unsigned)S + c + idx % ZC;
            if (m < modes) {
                int r, zz;
                split(m, r, zz);
                cx<T>* dst = out + (long)r * hs;
                st(dst + zz, stage[idx]);
                // zeros in the row padding, up to the lines that hold modes
                if (zz == H - 1)
                    for (int q = H; q < hz; q++) st(dst + q, mk<T>(0, 0));
            }
        }
        __syncthreads();
    }
}

// src/grf.c:78-175 on one rank.  In place: every lower-half point reads its
// mirror, which lies in the untouched upper half or is the point itself.
template <typename T>
__global__ void k_hermitian(cx<T>* f, long hs, int N) {
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
        f[id] = conjg(f[mid]);
    }
}

struct AmpOne {
    static constexpr bool prescaled = false;
    __device__ __forceinline__ double operator()(long) const { return 1.0; }
};

// amplitude looked up by the integer n^2 of the mode
struct AmpTable {
    static constexpr bool prescaled = false;
    const double* tab;
    __device__ __forceinline__ double operator()(long n2) const { return tab[n2]; }
};

// FP32 noise: the amplitude times the noise factor sqrt(L^3/2), rounded to
// float on the host, so the values are those of AmpTable in half the bytes
// (the table of a 1024^3 grid, 3.1 MB, fits one XCD's L2)
struct AmpTableF {
    static constexpr bool prescaled = true;
    const float* tabf;
    __device__ __forceinline__ float f(long n2) const { return tabf[n2]; }
    __device__ __forceinline__ double operator()(long n2) const { return tabf[n2]; }
};

template <typename T, typename AMP, bool CR = true>
int launch_grf(cx<T>* out, long hs, int N, double boxlen, const NoiseJumps& J, AMP amp,
               hipStream_t s) {
    const long rows = (long)N * N;
    if constexpr (sizeof(T) == 8) {
        const int S = noise_segment(N, true);
        if (S <= 16) {
            const long segs = (rows * (N / 2 + 1) + S - 1) / S;
            auto kern = S == 4   ? k_grf_segments<T, 4, AMP, CR>
                        : S == 8 ? k_grf_segments<T, 8, AMP, CR>
                                 : k_grf_segments<T, 16, AMP, CR>;
            hipLaunchKernelGGL(kern, dim3((unsigned)((segs + 255) / 256)), dim3(256), 0, s, out,
                               hs, N, boxlen, J, amp);
            return hipGetLastError() == hipSuccess ? MITOS_OK : MITOS_ERR_DEVICE;
        }
    }
    hipLaunchKernelGGL((k_grf<T, AMP, CR>), dim3((unsigned)((rows + 255) / 256)), dim3(256), 0, s,
                       out, hs, N, boxlen, J, amp);
    return hipGetLastError() == hipSuccess ? MITOS_OK : MITOS_ERR_DEVICE;
}

template <typename T>
int launch_hermitian(cx<T>* f, long hs, int N, hipStream_t s) {
    const long n = 2L * (N / 2 + 1) * N;
    hipLaunchKernelGGL((k_hermitian<T>), dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, f, hs,
                       N);
    return hipGetLastError() == hipSuccess ? MITOS_OK : MITOS_ERR_DEVICE;
}

}  // namespace mitos
