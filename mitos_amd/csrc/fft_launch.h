// Host-side launch layer for the FFT passes: size dispatch, twiddle tables,
// one launcher per pass kind and the composed 3D transforms.
#pragma once

#include <map>
#include <mutex>
#include <type_traits>

#include "fft_passes.h"

namespace mitos {

// Grid sizes with compiled FFT passes (line length N for the x/y passes, N/2
// for the z passes): powers of two from 8 to 1024 and 3*2^k from 24 to 1536.
template <typename F>
int with_size(int N, F&& f) {
    switch (N) {
        case 8: return f.template operator()<8>();
        case 16: return f.template operator()<16>();
        case 24: return f.template operator()<24>();
        case 32: return f.template operator()<32>();
        case 48: return f.template operator()<48>();
        case 64: return f.template operator()<64>();
        case 96: return f.template operator()<96>();
        case 128: return f.template operator()<128>();
        case 192: return f.template operator()<192>();
        case 256: return f.template operator()<256>();
        case 384: return f.template operator()<384>();
        case 512: return f.template operator()<512>();
        case 768: return f.template operator()<768>();
        case 1024: return f.template operator()<1024>();
        case 1536: return f.template operator()<1536>();
        default: return MITOS_ERR_UNSUPPORTED;
    }
}

inline bool size_supported(int N) {
    switch (N) {
        case 8: case 16: case 24: case 32: case 48: case 64: case 96: case 128: case 192:
        case 256: case 384: case 512: case 768: case 1024: case 1536:
            return true;
        default:
            return false;
    }
}

// Device twiddle table tw[k] = exp(-2 pi i k / L), k < L, one per (device, L, type).
template <typename T>
const cx<T>* twiddles(int L) {
    static std::mutex mu;
    static std::map<std::pair<int, int>, cx<T>*> cache;
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) return nullptr;
    std::lock_guard<std::mutex> lock(mu);
    auto key = std::make_pair(dev, L);
    auto it = cache.find(key);
    if (it != cache.end()) return it->second;
    cx<T>* h = new cx<T>[L];
    for (int k = 0; k < L; k++) {
        // reduce by symmetry so the quarter-period values are exact
        long n = k, d = L;
        double c, s;
        if (4 * n == d) { c = 0; s = 1; }
        else if (2 * n == d) { c = -1; s = 0; }
        else if (4 * n == 3 * d) { c = 0; s = -1; }
        else if (n == 0) { c = 1; s = 0; }
        else {
            const double a = 2.0 * M_PI * (double)n / (double)d;
            c = cos(a);
            s = sin(a);
        }
        h[k] = mk<T>((T)c, (T)(-s));
    }
    cx<T>* d = nullptr;
    if (hipMalloc(&d, sizeof(cx<T>) * L) != hipSuccess) {
        delete[] h;
        return nullptr;
    }
    if (copy_sync(d, h, sizeof(cx<T>) * L, hipMemcpyHostToDevice) != hipSuccess) {
        delete[] h;
        hipFree(d);
        return nullptr;
    }
    delete[] h;
    cache[key] = d;
    return d;
}

inline int launch_status() {
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) {
        fprintf(stderr, "mitos_hip: kernel launch failed: %s\n", hipGetErrorString(e));
        return MITOS_ERR_DEVICE;
    }
    return MITOS_OK;
}

// ---- strided pass ----------------------------------------------------------
// k_pass_strided addresses a thread's elements by a 32-bit byte offset from a
// uniform base: TPL line positions of stride pstride must span under 4 GiB
template <typename T, int L, int AXIS>
inline bool strided_offsets_fit(int tpl, long hs) {
    const long pstride = AXIS == 0 ? (long)L * hs : hs;
    return (long)tpl * pstride * (long)sizeof(cx<T>) < (1L << 32);
}

// outer indices per work-group of a strided pass: 2 consecutive y rows for the
// x lines (measured: the rows of an x pass stream faster from one work-group)
template <int L, int AXIS>
struct OuterPerBlock {
    static constexpr int value = (AXIS == 0 && L >= 64) ? 2 : 1;
};

// ---- z passes ----------------------------------------------------------------
template <int TPL>
struct RowsPerBlock {
    static constexpr int value = TPL >= 256 ? 1 : 256 / TPL;
};

// ---- tunable schedules ---------------------------------------------------------
// Variants of the plain passes that the autotuner (autotune.h) times on the
// device and picks from, per (device, N, precision):
//   strided  0: LineCfg radices, 128-byte column tile
//            1: LineCfgS radices (fewer values per thread), the widest tile
//               of at most 1024 threads
//            2: 256-byte column tile when it fits (32 values per thread for
//               1024-point float lines)
//            3: LineCfg radices, 128-byte tile, two LDS exchange buffers
//               (one exchange step fewer) when they fit in 160 KiB
//   z passes 0: LineCfg radices, RowsPerBlock rows per work-group
//            1: LineCfgS radices, RowsPerBlock rows of its thread count
//            2: LineCfg radices, twice the rows when it fits
//            3: LineCfg radices, one row per work-group when a row fills a
//               wave (no barrier waits on other rows)
constexpr int kFftVariants = 4;

// 32 values per thread for the 256-byte tile of 1024-point float lines
template <int L>
struct LineCfgW {
    static constexpr int E = LineCfg<L>::E;
    typedef typename LineCfg<L>::R R;
};
template <>
struct LineCfgW<1024> {
    static constexpr int E = 32;
    typedef Radices<16, 16, 4> R;
};

template <typename T, int L, int V>
struct StridedSched {
    typedef typename std::conditional<
        V == 1, LineCfgS<L>,
        typename std::conditional<V == 2 && sizeof(T) == 4, LineCfgW<L>, LineCfg<L>>::type>::type
        CFG;
    static constexpr int TPL = L / CFG::E;
    static constexpr int CB = (TPL * ColTile<T>::C <= 1024) ? ColTile<T>::C : 1024 / TPL;
    // the wider tile only while one exchange buffer fits in the LDS
    static constexpr int C2 = 2 * ColTile<T>::C;
    static constexpr bool WIDE = V == 2 && TPL * C2 <= 1024 &&
                                 (long)L * (C2 + 1) * (long)sizeof(T) <= 163840;
    static constexpr int C = WIDE ? C2 : CB;
};

template <typename T, int L, int C, int AXIS, int DIR, bool SPLIT, typename OP, typename CFG,
          typename RAD = typename CFG::R>
struct StridedKV;
template <typename T, int L, int C, int AXIS, int DIR, bool SPLIT, typename OP, typename CFG,
          int... Rs>
struct StridedKV<T, L, C, AXIS, DIR, SPLIT, OP, CFG, Radices<Rs...>> {
    static void go(dim3 g, dim3 b, hipStream_t s, const cx<T>* in, cx<T>* out, long hs,
                   long ohs, int ncols, const cx<T>* tw, OP op, int o0) {
        hipLaunchKernelGGL((k_pass_strided<T, L, CFG::E, C, AXIS, DIR, SPLIT,
                                           OuterPerBlock<L, AXIS>::value, OP, Rs...>),
                           g, b, 0, s, in, out, hs, ohs, ncols, tw, op, o0);
    }
};

// in: rows of hs, out: rows of ohs; outer indices o0 .. o0+no-1 only when no > 0
template <typename T, int L, int AXIS, int DIR, int V, typename OP>
int strided_pass_v(const cx<T>* in, long hs, cx<T>* out, long ohs, OP op, hipStream_t s,
                   int o0 = 0, int no = 0) {
    if (no <= 0) {
        o0 = 0;
        no = L;
    }
    constexpr int KO = OuterPerBlock<L, AXIS>::value;
    if (o0 < 0 || o0 + no > L || o0 % KO || no % KO) return MITOS_ERR_ARG;
    if (in == out && hs != ohs) return MITOS_ERR_ARG;
    typedef StridedSched<T, L, V> S;
    constexpr int C = S::C;
    constexpr long LDS2 = 2 * (long)LdsMap<T, L, C, true>::SIZE * (long)sizeof(T);
    constexpr bool SPLIT = V == 3 ? LDS2 > 163840 : LDS2 > 81920;
    const int ncols = L / 2 + 1;
    if (!strided_offsets_fit<T, L, AXIS>(S::TPL, hs)) return MITOS_ERR_UNSUPPORTED;
    const cx<T>* tw = twiddles<T>(L);
    if (!tw) return MITOS_ERR_ALLOC;
    dim3 grid((stored_cols<T, C>(ncols, ohs) + C - 1) / C, no / KO);
    StridedKV<T, L, C, AXIS, DIR, SPLIT, OP, typename S::CFG>::go(
        grid, dim3(S::TPL * C), s, in, out, hs, ohs, ncols, tw, op, o0);
    return launch_status();
}

// strided pass with a run-time schedule variant
template <typename T, int L, int AXIS, int DIR, typename OP>
int strided_pass_tuned(int variant, const cx<T>* in, cx<T>* out, long hs, OP op, hipStream_t s) {
    switch (variant) {
        case 1: return strided_pass_v<T, L, AXIS, DIR, 1>(in, hs, out, hs, op, s);
        case 2: return strided_pass_v<T, L, AXIS, DIR, 2>(in, hs, out, hs, op, s);
        case 3: return strided_pass_v<T, L, AXIS, DIR, 3>(in, hs, out, hs, op, s);
        default: return strided_pass_v<T, L, AXIS, DIR, 0>(in, hs, out, hs, op, s);
    }
}

// work-groups of a z pass: each walks several row groups (about 8192 waves
// in all, enough to fill the device), at most one per group
inline unsigned z_groups(long nrows, int rw, int tpl) {
    const long ngroups = (nrows + rw - 1) / rw;
    const long waves = ((long)tpl * rw + 63) / 64;
    const long cap = 8192 / waves > 0 ? 8192 / waves : 1;
    return (unsigned)(ngroups < cap ? ngroups : cap);
}

template <typename T, int L, int V>
struct ZSched {
    typedef typename std::conditional<V == 1, LineCfgS<L>, LineCfg<L>>::type CFG;
    static constexpr int TPL = L / CFG::E;
    static constexpr int RW0 = V == 3 ? (TPL >= 64 ? 1 : RowsPerBlock<TPL>::value)
                                      : RowsPerBlock<TPL>::value * (V == 2 ? 2 : 1);
    static constexpr int RW = (TPL * RW0 <= 1024) ? RW0 : RowsPerBlock<TPL>::value;
};

template <typename T, int L, int RW, int HO, typename OP, typename CFG,
          typename RAD = typename CFG::R>
struct ZC2RKV;
template <typename T, int L, int RW, int HO, typename OP, typename CFG, int... Rs>
struct ZC2RKV<T, L, RW, HO, OP, CFG, Radices<Rs...>> {
    template <typename... A>
    static void go(dim3 g, dim3 b, hipStream_t s, A... a) {
        hipLaunchKernelGGL((k_zc2r<T, L, CFG::E, RW, HO, OP, Rs...>), g, b, 0, s, a...);
    }
};

// rows r0 .. r1-1 only when r1 > 0
template <typename T, int N, int V, int HO, typename OP>
int zc2r_pass_v(const cx<T>* in, T* out, long hs, long rs, int nbatch, long inb, long outb,
                T scale, OP op, hipStream_t s, long r0 = 0, long r1 = 0) {
    if (rs < N + (HO > 0 ? HO + 1 : 0)) return MITOS_ERR_ARG;
    constexpr int L = N / 2;
    typedef ZSched<T, L, V> S;
    if (r1 <= 0) {
        r0 = 0;
        r1 = (long)N * N;
    }
    if (r0 < 0 || r1 > (long)N * N || r0 >= r1) return MITOS_ERR_ARG;
    const cx<T>* tw = twiddles<T>(L);
    const cx<T>* twN = twiddles<T>(N);
    if (!tw || !twN) return MITOS_ERR_ALLOC;
    dim3 grid(z_groups(r1 - r0, S::RW, S::TPL), nbatch);
    ZC2RKV<T, L, S::RW, HO, OP, typename S::CFG>::go(grid, dim3(S::TPL * S::RW), s, in, out, r0,
                                                     r1, N, hs, rs, inb, outb, tw, twN, scale,
                                                     op);
    return launch_status();
}

template <typename T, int N, int HO, typename OP>
int zc2r_pass_tuned(int variant, const cx<T>* in, T* out, long hs, long rs, int nbatch, long inb,
                    long outb, T scale, OP op, hipStream_t s, long r0 = 0, long r1 = 0) {
    switch (variant) {
        case 1:
            return zc2r_pass_v<T, N, 1, HO>(in, out, hs, rs, nbatch, inb, outb, scale, op, s, r0,
                                            r1);
        case 2:
            return zc2r_pass_v<T, N, 2, HO>(in, out, hs, rs, nbatch, inb, outb, scale, op, s, r0,
                                            r1);
        case 3:
            return zc2r_pass_v<T, N, 3, HO>(in, out, hs, rs, nbatch, inb, outb, scale, op, s, r0,
                                            r1);
        default:
            return zc2r_pass_v<T, N, 0, HO>(in, out, hs, rs, nbatch, inb, outb, scale, op, s, r0,
                                            r1);
    }
}

template <typename T, int L, int RW, typename LOADER, typename OP, typename CFG,
          typename RAD = typename CFG::R>
struct ZR2CKV;
template <typename T, int L, int RW, typename LOADER, typename OP, typename CFG, int... Rs>
struct ZR2CKV<T, L, RW, LOADER, OP, CFG, Radices<Rs...>> {
    template <typename... A>
    static void go(dim3 g, dim3 b, hipStream_t s, A... a) {
        hipLaunchKernelGGL((k_zr2c<T, L, CFG::E, RW, LOADER, OP, Rs...>), g, b, 0, s, a...);
    }
};

// rows r0 .. r1-1 only when r1 > 0
template <typename T, int N, int V, typename LOADER, typename OP>
int zr2c_pass_v(LOADER loader, cx<T>* out, long hs, int nbatch, long outb, OP op,
                hipStream_t s, long r0 = 0, long r1 = 0) {
    constexpr int L = N / 2;
    typedef ZSched<T, L, V> S;
    if (r1 <= 0) {
        r0 = 0;
        r1 = (long)N * N;
    }
    if (r0 < 0 || r1 > (long)N * N || r0 >= r1) return MITOS_ERR_ARG;
    const cx<T>* tw = twiddles<T>(L);
    const cx<T>* twN = twiddles<T>(N);
    if (!tw || !twN) return MITOS_ERR_ALLOC;
    dim3 grid(z_groups(r1 - r0, S::RW, S::TPL), nbatch);
    ZR2CKV<T, L, S::RW, LOADER, OP, typename S::CFG>::go(grid, dim3(S::TPL * S::RW), s, loader,
                                                         out, r0, r1, N, hs, outb, tw, twN, op);
    return launch_status();
}

template <typename T, int N, typename LOADER, typename OP>
int zr2c_pass_tuned(int variant, LOADER loader, cx<T>* out, long hs, int nbatch, long outb,
                    OP op, hipStream_t s, long r0 = 0, long r1 = 0) {
    switch (variant) {
        case 1: return zr2c_pass_v<T, N, 1>(loader, out, hs, nbatch, outb, op, s, r0, r1);
        case 2: return zr2c_pass_v<T, N, 2>(loader, out, hs, nbatch, outb, op, s, r0, r1);
        case 3: return zr2c_pass_v<T, N, 3>(loader, out, hs, nbatch, outb, op, s, r0, r1);
        default: return zr2c_pass_v<T, N, 0>(loader, out, hs, nbatch, outb, op, s, r0, r1);
    }
}

// ---- composed 3D transforms ---------------------------------------------------
// The passes between the caller's arrays run through work grids w1, w2 of rows of
// whs, whole 128-byte lines (work_row elements) where there is room: a pass over the
// dense rows of N/2+1 values splits every tile row over two lines.  w2 == w1 passes
// x in place, which the drop-in calls do above 128^3: a second grid gains 4 to 11% at
// 128^3 and 5% of an r2c at 512^3 (1.40 against 1.48 ms in FP64), but loses 21% at
// 256^3 (206 against 163 us), where the arrays then leave the memory-side cache.  The
// pass at the caller's dense grid is the y pass, whose tiles of one plane meet in L2
// (512^3 FP64: 0.44 ms reading and 0.49 ms writing it, an x pass 0.54 and 0.64 ms).
// Whole transforms in FP64 against passes over dense rows: 512^3 c2r 1.55 -> 1.31 ms,
// r2c 1.57 -> 1.48 ms; 256^3 211 -> 164 us, 199 -> 164 us; bound by HBM (512^3: three
// passes of 2.15 GB at 4.8 TB/s).  Schedules: variant 0 of the strided passes, variant
// 1 of the z passes (the 16 values per thread of variant 0 take twice as long in FP64
// at 256^3 and 512^3: z r2c 907 against 424 us).
template <typename T>
inline long work_row(int N) {
    const long q = 128 / (long)sizeof(cx<T>);
    return (N / 2 + 1 + q - 1) / q * q;
}
template <typename T>
inline size_t work_grid_bytes(int N) {
    return sizeof(cx<T>) * (size_t)N * N * (size_t)work_row<T>(N);
}

// c2r: y (in -> w1, values through op.pre), x (w1 -> w2), z (w2 -> out).  The
// input is left unchanged (unless it is w1).
template <typename T, typename OP>
int c2r_3d(int N, const cx<T>* in, long ihs, cx<T>* w1, cx<T>* w2, long whs, T* out, long rs,
           T scale, OP op, hipStream_t s) {
    return with_size(N, [&]<int NN>() -> int {
        MITOS_TRY((strided_pass_v<T, NN, 1, 1, 0>(in, ihs, w1, whs, op, s)));
        MITOS_TRY((strided_pass_v<T, NN, 0, 1, 0>(w1, whs, w2, whs, OpNone(), s)));
        return zc2r_pass_v<T, NN, 1, 0>(w2, out, whs, rs, 1, 0, 0, scale, OpNone(), s);
    });
}

// r2c: z (loader -> w1), x (w1 -> w2), y (w2 -> out, values through op.post).
template <typename T, typename LOADER, typename OP>
int r2c_3d(int N, LOADER loader, cx<T>* w1, cx<T>* w2, long whs, cx<T>* out, long ohs, OP op,
           hipStream_t s) {
    return with_size(N, [&]<int NN>() -> int {
        MITOS_TRY((zr2c_pass_v<T, NN, 1>(loader, w1, whs, 1, 0, OpNone(), s)));
        MITOS_TRY((strided_pass_v<T, NN, 0, -1, 0>(w1, whs, w2, whs, OpNone(), s)));
        return strided_pass_v<T, NN, 1, -1, 0>(w2, whs, out, ohs, op, s);
    });
}

}  // namespace mitos
