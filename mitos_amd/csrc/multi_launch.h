// Launches of the multi-output passes of pipeline_kernels.h, shared by the fused
// pipeline and the drop-in 2LPT and Monge-Ampere solvers.
#pragma once

#include "pipeline_kernels.h"

namespace mitos {

// ---- launch helpers for the fused kernels ---------------------------------------------
// Line configuration and tile width of the register-heavy multi-transform
// kernels: 8 (or 12) values per thread and 64-byte tile rows, so that the
// input tile, the transformed copy and the radix temporaries stay in VGPRs.
// Multi-output passes on float lines of 1024: 16 values per thread, so a
// line is one wave (fewer exchange steps), and 128-byte tile rows (whole
// lines; work-groups of 1024 threads, one per CU); the combine pass keeps the
// smaller line configuration (MULTI = false).
template <typename T, int L, bool MULTI = true>
struct HeavyCfg {
    static constexpr bool WIDE = MULTI && sizeof(T) == 4 && L == 1024;
    typedef typename std::conditional<WIDE, LineCfg<L>, LineCfgS<L>>::type CFG;
    static constexpr int E = CFG::E;
    static constexpr int TPL = L / E;
    static constexpr int C0 = (WIDE ? 128 : 64) / (2 * (int)sizeof(T));
    static constexpr int C = (TPL * C0 <= 1024) ? C0 : 1024 / TPL;
};
template <typename T, int L, int AXIS, int DIR, int NIN, typename CODES,
          typename RAD = typename HeavyCfg<T, L>::CFG::R>
struct MultiK;
template <typename T, int L, int AXIS, int DIR, int NIN, typename CODES, int... Rs>
struct MultiK<T, L, AXIS, DIR, NIN, CODES, Radices<Rs...>> {
    // no: outer indices of the launch (a slab of x planes of a y pass; the
    // pointers start at the slab)
    static int go(const MultiPtrs<T, NIN, CODES::n>& P, long hs, double dk, hipStream_t s,
                  int no = L) {
        constexpr int C = HeavyCfg<T, L>::C;
        constexpr int E = HeavyCfg<T, L>::E;
        // one exchange buffer per component unless that leaves less than two
        // work-groups per CU; the wide form runs one per CU by its registers
        // anyway (1024 threads at about 124), so it takes both (139 KB)
        constexpr bool SPLIT = !HeavyCfg<T, L>::WIDE &&
                               2 * LdsMap<T, L, C, true>::SIZE * sizeof(T) > 81920;
        const int ncols = L / 2 + 1;
        const cx<T>* tw = twiddles<T>(L);
        if (!tw) return MITOS_ERR_ALLOC;
        constexpr int KO = (AXIS == 0 && L >= 64) ? 2 : 1;
        hipLaunchKernelGGL((k_multi_strided<T, L, E, C, AXIS, DIR, SPLIT, NIN, CODES, KO, Rs...>),
                           dim3((ncols + C - 1) / C, no / KO), dim3(L / E * C), 0, s, P, hs, ncols,
                           dk, tw);
        return launch_status();
    }
};

// Lines of k_hess_z: in FP64 four values a thread for powers of two, so the four
// arrays of a thread's row leave room for its addresses and twiddles, and a row of
// 256 is one wave, whose barriers wait on nobody (rows of fewer threads share a
// wave).  Against eight a thread, by the realization's own stage times: 128^3 48 -> 37
// us, 256^3 341 -> 247 us, 512^3 2.61 -> 1.65 ms, 1024^3 16.2 -> 15.0 ms (lines of 64 to
// 512); the drop-in 2LPT at 256^3 1.80 -> 1.66 ms.  Bound by latency at two waves a
// SIMD: four waves (addresses and twiddles formed anew per row) were slower (512^3 2.33
// against 2.14 ms under the profiler).
template <typename T, int L>
struct HessCfg : LineCfgS<L> {};
template <>
struct HessCfg<double, 64> {
    static constexpr int E = 4;
    typedef Radices<4, 4, 4> R;
};
template <>
struct HessCfg<double, 128> {
    static constexpr int E = 4;
    typedef Radices<4, 4, 4, 2> R;
};
template <>
struct HessCfg<double, 256> {
    static constexpr int E = 4;
    typedef Radices<4, 4, 4, 4> R;
};
template <>
struct HessCfg<double, 512> {
    static constexpr int E = 4;
    typedef Radices<4, 4, 4, 4, 2> R;
};

template <typename T, int N, typename RAD = typename HessCfg<T, N / 2>::R>
struct HessZK;
template <typename T, int N, int... Rs>
struct HessZK<T, N, Radices<Rs...>> {
    // delta2 rows written as reals (row stride rs) for a separate z pass; nrows
    // rows from the pointers on
    static int go(const MultiPtrs<T, 6, 1>& P, long hs, double dk, T scale, T* real, long rs,
                  hipStream_t s, long nrows = (long)N * N) {
        constexpr int L = N / 2;
        constexpr int E = HessCfg<T, L>::E;
        constexpr int TPL = L / E;
        // a row of a wave or more: one row per work-group (no barrier waits
        // on other rows' waves)
        constexpr int RW = TPL >= 64                            ? 1
                           : sizeof(T) == 8 && E == 4 && TPL >= 16 ? 64 / TPL
                                                   : RowsPerBlock<TPL>::value;
        const cx<T>* tw = twiddles<T>(L);
        const cx<T>* twN = twiddles<T>(N);
        if (!tw || !twN) return MITOS_ERR_ALLOC;
        hipLaunchKernelGGL((k_hess_z<T, L, E, RW, Rs...>), dim3((unsigned)((nrows + RW - 1) / RW)),
                           dim3(TPL * RW), 0, s, P, nrows, hs, dk, scale, tw, twN, real, rs);
        return launch_status();
    }
};

}  // namespace mitos
