// Members of Pipe that launch the fused kernels (pipe.h declares them), compiled
// once per precision by pipe_f32.hip and pipe_f64.hip.
#pragma once

#include "multi_launch.h"
#include "pipe.h"

namespace mitos {

template <typename T, int N, typename RAD = typename HeavyCfg<T, N, false>::CFG::R>
struct CombineK;
template <typename T, int N, int... Rs>
struct CombineK<T, N, Radices<Rs...>> {
    static int go(const cx<T>* D, const cx<T>* K, cx<T>* C0, cx<T>* C1, long hs,
                  const CombineParams& cp, hipStream_t s) {
        constexpr int L = N;
        constexpr int C = HeavyCfg<T, L, false>::C;
        constexpr int E = HeavyCfg<T, L, false>::E;
        constexpr bool SPLIT = 2 * LdsMap<T, L, C, true>::SIZE * sizeof(T) > 81920;
        const int ncols = L / 2 + 1;
        const cx<T>* tw = twiddles<T>(L);
        if (!tw) return MITOS_ERR_ALLOC;
        hipLaunchKernelGGL((k_x_combine<T, L, E, C, SPLIT, Rs...>),
                           dim3((ncols + C - 1) / C, L), dim3(L / E * C), 0, s, D, K, C0, C1, hs,
                           ncols, cp, tw);
        return launch_status();
    }
};

template <typename T>
int Pipe<T>::autotune(hipStream_t s) {
    int dev = 0;
    MITOS_HIP_CHECK(hipGetDevice(&dev));
    const auto key = std::make_tuple(dev, N, (int)sizeof(T));
    std::lock_guard<std::mutex> lock(schedule_mutex());
    auto& table = schedule_table();
    auto it = table.find(key);
    if (it != table.end()) {
        sched = it->second;
        return MITOS_OK;
    }
    FftSchedule sc;
    const char* env = getenv("MITOS_FFT_SCHEDULE");
    if (!(env && strcmp(env, "default") == 0)) {
        hipEvent_t e0, e1;
        MITOS_HIP_CHECK(hipEventCreate(&e0));
        MITOS_HIP_CHECK(hipEventCreate(&e1));
        int rc = with_size(N, [&]<int NN>() -> int {
            auto time_it = [&](auto&& launch, float* ms) -> int {
                MITOS_TRY(launch());  // warm-up
                MITOS_HIP_CHECK(hipEventRecord(e0, s));
                for (int r = 0; r < 3; r++) MITOS_TRY(launch());
                MITOS_HIP_CHECK(hipEventRecord(e1, s));
                MITOS_HIP_CHECK(hipEventSynchronize(e1));
                MITOS_HIP_CHECK(hipEventElapsedTime(ms, e0, e1));
                *ms /= 3;
                return MITOS_OK;
            };
            CicLoader<T> ld{cic(), (long)NN, 1.0};
            for (int v = 0; v < kFftVariants; v++) {
                // out of place, as the runs use them
                MITOS_TRY(time_it([&] {
                    return strided_pass_tuned<T, NN, 1, -1>(v, K, a(0), hs, OpNone(), s);
                }, &sc.ms[TUNE_Y_FWD][v]));
                MITOS_TRY(time_it([&] {
                    return strided_pass_tuned<T, NN, 0, -1>(v, a(0), K, hs, OpNone(), s);
                }, &sc.ms[TUNE_X_FWD][v]));
                MITOS_TRY(time_it([&] {
                    // the displacement grids' layout of the default form
                    constexpr int HO = sizeof(T) == 4 ? MITOS_PSI_SO : MITOS_PSI_HO;
                    return zc2r_pass_tuned<T, NN, HO>(v, b(0), psi(0), hs, prs(), 1, 0, 0,
                                                      (T)1, OpNone(), s);
                }, &sc.ms[TUNE_Z_C2R][v]));
                MITOS_TRY(time_it([&] {
                    return zr2c_pass_tuned<T, NN>(v, ld, K, hs, 1, 0, OpNone(), s);
                }, &sc.ms[TUNE_Z_R2C][v]));
            }
            return MITOS_OK;
        });
        hipEventDestroy(e0);
        hipEventDestroy(e1);
        MITOS_TRY(rc);
        for (int k = 0; k < TUNE_KINDS; k++)
            for (int v = 1; v < kFftVariants; v++)
                if (sc.ms[k][v] < sc.ms[k][sc.v[k]]) sc.v[k] = v;
    }
    table[key] = sc;
    sched = sc;
    return MITOS_OK;
}

template <typename T>
int Pipe<T>::fft_timing(hipStream_t s, int reps, float* r2c_ms, float* c2r_ms) {
    hipEvent_t e0, e1, e2;
    MITOS_HIP_CHECK(hipEventCreate(&e0));
    MITOS_HIP_CHECK(hipEventCreate(&e1));
    MITOS_HIP_CHECK(hipEventCreate(&e2));
    T* real = psi(0);
    const long rs = prs();
    const int rc = with_size(N, [&]<int NN>() -> int {
        RealRowLoader<T> ld{real, rs, 0};
        auto r2c = [&]() -> int {
            MITOS_TRY((zr2c_pass_tuned<T, NN>(sched.v[TUNE_Z_R2C], ld, K, hs, 1, 0, OpNone(), s)));
            // out of place (an in-place strided pass streams slower)
            MITOS_TRY((strided_pass_tuned<T, NN, 1, -1>(sched.v[TUNE_Y_FWD], K, a(0), hs, OpNone(),
                                                        s)));
            return strided_pass_tuned<T, NN, 0, -1>(sched.v[TUNE_X_FWD], a(0), K, hs, OpNone(), s);
        };
        auto c2r = [&]() -> int {
            MITOS_TRY((strided_pass_tuned<T, NN, 0, 1>(sched.v[TUNE_X_FWD], K, a(0), hs, OpNone(), s)));
            MITOS_TRY((strided_pass_tuned<T, NN, 1, 1>(sched.v[TUNE_Y_FWD], a(0), a(1), hs, OpNone(),
                                                       s)));
            return zc2r_pass_tuned<T, NN, 0>(sched.v[TUNE_Z_C2R], a(1), real, hs, rs, 1, 0, 0,
                                             (T)1, OpNone(), s);
        };
        MITOS_TRY(r2c());
        MITOS_TRY(c2r());
        MITOS_HIP_CHECK(hipEventRecord(e0, s));
        for (int r = 0; r < reps; r++) MITOS_TRY(r2c());
        MITOS_HIP_CHECK(hipEventRecord(e1, s));
        for (int r = 0; r < reps; r++) MITOS_TRY(c2r());
        MITOS_HIP_CHECK(hipEventRecord(e2, s));
        MITOS_HIP_CHECK(hipEventSynchronize(e2));
        MITOS_HIP_CHECK(hipEventElapsedTime(r2c_ms, e0, e1));
        MITOS_HIP_CHECK(hipEventElapsedTime(c2r_ms, e1, e2));
        *r2c_ms /= reps;
        *c2r_ms /= reps;
        return MITOS_OK;
    });
    hipEventDestroy(e0);
    hipEventDestroy(e1);
    hipEventDestroy(e2);
    return rc;
}

template <typename T>
int Pipe<T>::enqueue(const mitos_ic_config& cfg, hipStream_t s, bool timing,
            const double* amp_tab, double* pk_dst,
            long long* obs_dst, const cx<T>* noise_in,
            int stencil) {
    // particle lattice M^3 (src/particle.c:87-129); the lattice-tile
    // kernels (stencil form, tiled moves and deposits) need M = N
    const int Ml = cfg.M > 0 ? cfg.M : N;
    const long long nl = (long long)Ml * Ml * Ml;
    if (nl > pcap) return MITOS_ERR_DIMS;
    if (Ml != N && (noise_in || stencil > 0)) return MITOS_ERR_UNSUPPORTED;
    npart = nl;
    // the stencil form is exact only for particles on grid nodes
    const bool STENCIL =
        Ml == N && (stencil < 0 ? (sizeof(T) == 4 && lattice_on_nodes(N, cfg.boxlen))
                                : stencil != 0);
    psi_stencilled = STENCIL;
    const double L = cfg.boxlen;
    const double dk = 2 * M_PI / L;
    const double boxvol = L * L * L;
    const double sfwd = boxvol / ((long long)N * N * N);
    const long long np = (long long)N * N * N;
    // algorithmic bytes: one half-complex grid, one real grid
    const double G = (double)N * N * (N / 2 + 1) * sizeof(cx<T>);
    const double Rg = (double)np * sizeof(T);
    MITOS_TRY(ensure_bins(cfg.bins));
    amplitude = amplitude_cached(cfg.n_s, cfg.gamma, cfg.sigma8);
    nprof = 0;
    auto mark = [&](int i) {
        if (timing) hipEventRecord(ev[i], s);
    };
    mark(0);
    // 1. noise -> phi1(k), Hermitian planes (src/grf.c, src/2lpt.c:75)
    Xo s0 = xo_seed(cfg.seed);
    NoiseJumps J;
    MITOS_TRY(noise_jumps(N, sizeof(T) == 8, s0, &J));
    const double* amp = amp_tab ? amp_tab : phi1_table(N, L, amplitude, cfg.n_s, cfg.gamma);
    if (!amp) return MITOS_ERR_ALLOC;
    // FP64 keeps correctly rounded Box-Muller; FP32 rounds every value to float
    MITOS_TRY(timed(s, "grf_noise", G, [&] {
        if (noise_in) {
            hipLaunchKernelGGL((k_noise_in<T>), dim3(nblk((long)N * N * (N / 2 + 1))),
                               dim3(256), 0, s, noise_in, K, hs, N, L, amp);
            return launch_status();
        }
        if constexpr (sizeof(T) == 4) {
            if (!amp_tab) {
                // an unbatched FP32 run: the prescaled float table (the
                // same values as the double table's product)
                const float* ampf = phi1_table_f(N, L, amplitude, cfg.n_s, cfg.gamma);
                if (!ampf) return MITOS_ERR_ALLOC;
                return launch_grf<T, AmpTableF, false>(K, hs, N, L, J, AmpTableF{ampf}, s);
            }
        }
        return launch_grf<T, AmpTable, sizeof(T) == 8>(K, hs, N, L, J, AmpTable{amp}, s);
    }));
    MITOS_TRY(timed(s, "hermitian_planes", 0.0,
                    [&] { return launch_hermitian<T>(K, hs, N, s); }));
    mark(1);
    return with_size(N, [&]<int NN>() -> int {
        cx<T>* D = a(0);
        if (cfg.run2lpt) {
            // 2. x pass: A0 = X(phi1), A1 = X(i kx phi1), A2 = X(-kx^2 phi1)
            MultiPtrs<T, 1, 3> p2;
            p2.in[0] = K;
            p2.out[0] = a(0);
            p2.out[1] = a(1);
            p2.out[2] = a(2);
            MITOS_TRY(timed(s, "hessian_x_1to3", 4 * G, [&] {
                return MultiK<T, NN, 0, 1, 1,
                              OutCodes<MITOS_OUT(0, 0), MITOS_OUT(0, 1), MITOS_OUT(0, 2)>>::go(
                    p2, hs, dk, s);
            }));
            // 3. y pass: six Hessian factors
            MultiPtrs<T, 3, 6> p3;
            p3.in[0] = a(0);
            p3.in[1] = a(1);
            p3.in[2] = a(2);
            for (int i = 0; i < 6; i++) p3.out[i] = b(i);
            MITOS_TRY(timed(s, "hessian_y_3to6", 9 * G, [&] {
                return MultiK<T, NN, 1, 1, 3,
                              OutCodes<MITOS_OUT(0, 0), MITOS_OUT(0, 1), MITOS_OUT(0, 2),
                                       MITOS_OUT(1, 0), MITOS_OUT(1, 1), MITOS_OUT(2, 0)>>::go(
                    p3, hs, dk, s);
            }));
            mark(2);
            // 4. z pass: delta2 and its r2c row (src/2lpt.c:84-116, poisson.c:61)
            MultiPtrs<T, 6, 1> p4;
            for (int i = 0; i < 6; i++) p4.in[i] = b(i);
            p4.out[0] = D;
            // delta2(x) rows into a(1) as reals, then their r2c into D
            T* d2 = reinterpret_cast<T*>(a(1));
            const long rs2 = prs();
            MITOS_TRY(timed(s, "hessian_z_delta2", 6 * G + Rg, [&] {
                return HessZK<T, NN>::go(p4, hs, dk, (T)(1.0 / boxvol), d2, rs2, s);
            }));
            MITOS_TRY(timed(s, "delta2_z_r2c", Rg + G, [&] {
                RealRowLoader<T> ld{d2, rs2, 0};
                return zr2c_pass_tuned<T, NN>(sched.v[TUNE_Z_R2C], ld, D, hs, 1, 0, OpNone(), s);
            }));
            // 5. y pass forward of delta2, out of place into a(2)
            MITOS_TRY(timed(s, "delta2_y_fwd", 2 * G, [&] {
                return strided_pass_tuned<T, NN, 1, -1>(sched.v[TUNE_Y_FWD], D, a(2), hs,
                                                        OpNone(), s);
            }));
            D = a(2);
        } else {
            D = K;  // Zel'dovich: the second-order term is multiplied by zero
            mark(2);
        }
        mark(3);
        // 6. x pass: Poisson + combine + TSC window + first inverse pass
        CombineParams cp;
        cp.dk = dk;
        cp.sD = sfwd;
        cp.f1 = cfg.f1;
        cp.f2 = cfg.run2lpt ? cfg.f2 : 0.0;
        cp.win = window_table(NN, L, 3);
        if (!cp.win) return MITOS_ERR_ALLOC;
        // the stencil form applies the lattice TSC stencils in k-space
        // (k_displace_lattice_s)
        cp.smooth = nullptr;
        if (STENCIL) {
            cp.smooth = smooth_table<double>(NN);
            if (!cp.smooth) return MITOS_ERR_ALLOC;
        }
        // C0, C1 into a(0), a(1) (D is a(2) or K)
        MITOS_TRY(timed(s, "combine_x", 4 * G, [&] {
            return CombineK<T, NN>::go(D, K, a(0), a(1), hs, cp, s);
        }));
        // 7. y pass: E1 = Y(i ky C0) (FP32: i ky S(ky) C0), E2 = Y(C0), E0 = Y(C1)
        MultiPtrs<T, 2, 3> p7;
        p7.in[0] = a(0);
        p7.in[1] = a(1);
        p7.out[0] = b(1);
        p7.out[1] = b(2);
        p7.out[2] = b(0);
        if (STENCIL) {
            p7.smooth = smooth_table<T>(NN);
            if (!p7.smooth) return MITOS_ERR_ALLOC;
        }
        MITOS_TRY(timed(s, "displacement_y_2to3", 5 * G, [&] {
            if (STENCIL)
                return MultiK<T, NN, 1, 1, 2,
                              OutCodes<MITOS_OUT(0, 3), MITOS_OUT(0, 0),
                                       MITOS_OUT(1, 0)>>::go(p7, hs, dk, s);
            return MultiK<T, NN, 1, 1, 2,
                          OutCodes<MITOS_OUT(0, 1), MITOS_OUT(0, 0), MITOS_OUT(1, 0)>>::go(
                p7, hs, dk, s);
        }));
        // 8. z c2r: displacement grids (src/mitos.c:404-416); the
        // stencil form without the z halo (its moves read no z taps)
        const T cs = (T)(1.0 / boxvol);
        auto psi_c2r = [&](const cx<T>* in, T* out, auto op) -> int {
            if (STENCIL)
                return zc2r_pass_tuned<T, NN, MITOS_PSI_SO>(sched.v[TUNE_Z_C2R], in, out, hs,
                                                            prs(), 1, 0, 0, cs, op, s);
            return zc2r_pass_tuned<T, NN, MITOS_PSI_HO>(sched.v[TUNE_Z_C2R], in, out, hs,
                                                        prs(), 1, 0, 0, cs, op, s);
        };
        MITOS_TRY(timed(s, "displacement_z_c2r", G + Rg,
                        [&] { return psi_c2r(b(0), psi(0), OpNone()); }));
        MITOS_TRY(timed(s, "displacement_z_c2r", G + Rg,
                        [&] { return psi_c2r(b(1), psi(1), OpNone()); }));
        MITOS_TRY(timed(s, "displacement_z_c2r", G + Rg,
                        [&] { return psi_c2r(b(2), psi(2), OpIkz{dk}); }));
        mark(4);
        // 9-10. lattice + sequential TSC displacement + wrap + CIC deposit
        const float spacing = (float)L / Ml;  // src/particle.c:102-103
        // the two-pass deposit of the lattice particles stores every
        // grid cell, the one-pass and the adjoint-mode deposits add to a
        // cleared grid (far-particle lists use K, free after combine_x)
        typedef typename std::conditional<sizeof(T) == 4, float, double>::type M;
        const bool two_pass = cic_ws && NN % 32 == 0 && Ml == NN &&
                              cic_list_bytes<M>(NN) <= sizeof(cx<T>) * (size_t)csize;
        if (!two_pass)
            MITOS_TRY(timed(s, "cic_clear", 8.0 * np, [&] {
                hipLaunchKernelGGL((k_fill_u64<T>), dim3(nblk(np)), dim3(256), 0, s, cic(),
                                   (long)np);
                return launch_status();
            }));
        mark(5);
        // FP32 moves the particles in float arithmetic, FP64 in double
        if (noise_in) {
            // the forward of the adjoint: the moves and cells that its backward
            // differentiates, positions in T up to the deposit.  FP64 positions lie
            // in the A grids (free once the displacement grids are made).
            MITOS_TRY(timed(s, "move_deposit", 3 * Rg + 12.0 * np + 8.0 * np, [&] {
                if constexpr (NN % 32 == 0 && NN > 32) {
                    // moves, then the tiled LDS deposit of the pipeline: 0.06 ms at
                    // 96^3 in FP64, a global atomic per corner and particle 0.30 ms
                    // (at 32^3 one launch is the faster: 164 against 175 us the forward)
                    T* xt = reinterpret_cast<T*>(a(0));
                    T* yt = reinterpret_cast<T*>(a(1));
                    T* zt = reinterpret_cast<T*>(a(2));
                    hipLaunchKernelGGL((k_moves_s<T>), dim3(adj_tiles(NN)), dim3(256), 0, s,
                                       psi(0), psi(1), psi(2), (unsigned)(prs()), NN, L, spacing,
                                       X, Y, Z, xt, yt, zt);
                    if constexpr (sizeof(T) == 8) {
                        MITOS_TRY((cic_lattice_launch<M, false, T, true>(
                            xt, yt, zt, NN, L, cic(), nullptr, nullptr, s)));
                    } else if (two_pass) {
                        MITOS_TRY((cic_lattice_launch<M, true, float, true>(
                            X, Y, Z, NN, L, cic(), cic_ws, K, s)));
                        MITOS_TRY(cic_gather_launch<M>(NN, cic(), cic_ws, s));
                        MITOS_TRY((cic_far_launch<M, true>(X, Y, Z, NN, L, cic(), cic_ws, K, s)));
                    } else {
                        MITOS_TRY((cic_lattice_launch<M, false, float, true>(
                            X, Y, Z, NN, L, cic(), nullptr, nullptr, s)));
                    }
                    return launch_status();
                }
                hipLaunchKernelGGL((k_move_deposit_s<T>), dim3(nblk(np)), dim3(256), 0, s,
                                   psi(0), psi(1), psi(2), (unsigned)(prs()),
                                   NN, L, spacing, X, Y, Z, cic(), cic_shift());
                return launch_status();
            }));
        } else {
            // reads 3 displacement grids, writes 3 float coordinates
            MITOS_TRY(timed(s, "displace_tsc", 3 * Rg + 12.0 * nl, [&] {
                constexpr int NT = NN >= 256 ? 256 : 64;
                const int nch = (NN + NT - 1) / NT;
                const unsigned rs = (unsigned)(prs());
                if (Ml != NN) {
                    // an M^3 lattice off the grid nodes: the 27-tap moves
                    // at each particle's position
                    hipLaunchKernelGGL((k_displace_lattice<T, M>),
                                       dim3(displace_lattice_blocks(Ml)), dim3(256), 0, s,
                                       psi(0), psi(1), psi(2), rs, NN, Ml,
                                       displace_lattice_planes(Ml), L, spacing, X, Y, Z);
                } else if (STENCIL && NN % 16 == 0 && tsc_tile) {
                    auto tile = [&](auto kern, int txn, int ty, int tz, int pp) {
                        const dim3 gridt(
                            (unsigned)((long)(NN / txn) * (NN / ty) * (NN / tz)));
                        hipLaunchKernelGGL(kern, gridt, dim3(txn / pp * ty * tz), 0, s,
                                           psi(0), psi(1), psi(2), rs, NN, (T)L, spacing, L,
                                           X, Y, Z, tsc_staged ? 1 : 0);
                    };
                    // 8 x 8 x 16 tiles, four particles per thread; windows of at
                    // most 40 x rows and 576 rows of 16 z (a limit of 608 left
                    // 0.2% of the tiles of a 1.95 Mpc/h cell at z = 0 amplitude
                    // to the direct reads), four work-groups per CU
                    tile(k_displace_tile<T, 8, 8, 16, 4, 40, 576, 12, 0>, 8, 8, 16, 4);
                } else if (STENCIL && NN % 64 == 0) {
                    constexpr int TX = 16, PPT = 8;
                    const dim3 gridw((unsigned)((long)NN * NN / PPT * (NN / 64)));
                    hipLaunchKernelGGL((k_displace_lattice_w<T, TX, PPT, 16, 6>), gridw,
                                       dim3(64), 0, s, psi(0), psi(1), psi(2), rs, NN,
                                       (T)L, spacing, L, X, Y, Z, tsc_staged ? 1 : 0);
                } else if (STENCIL) {
                    constexpr int TX = NN % 16 == 0 ? 16 : 8;
                    constexpr int PPT = 4;
                    const dim3 gridp((unsigned)((long)NN * NN / PPT * nch));
                    hipLaunchKernelGGL((k_displace_lattice_s<T, NT, TX, PPT>), gridp,
                                       dim3(NT), 0, s, psi(0), psi(1), psi(2), rs, NN, nch,
                                       (T)L, spacing, L, X, Y, Z);
                } else if (sizeof(T) == 8 && NN % 16 == 0 && tsc_tile) {
                  if constexpr (sizeof(T) == 8) {
                    // the reference's 27-tap moves over 8 x 8 x 16 tiles with the
                    // taps staged in LDS (same positions as the per-particle
                    // kernel, which MITOS_TSC_KERNEL=wave selects)
                    auto tile = [&](auto kern, int txn, int ty, int tz, int pp) {
                        const dim3 gridt(
                            (unsigned)((long)(NN / txn) * (NN / ty) * (NN / tz)));
                        hipLaunchKernelGGL(kern, gridt, dim3(txn / pp * ty * tz), 0, s,
                                           psi(0), psi(1), psi(2), rs, NN, spacing, L, X,
                                           Y, Z);
                    };
                    // 256 window rows (37 KB of LDS) and eight rows in flight per
                    // 32 lanes; four work-groups per CU (128 registers)
                    tile(k_displace_tile_ref<8, 8, 16, 4, 256, 8>, 8, 8, 16, 4);
                  }
                } else {
                    hipLaunchKernelGGL((k_displace_lattice<T, M>),
                                       dim3(displace_lattice_blocks(NN)), dim3(256), 0, s,
                                       psi(0), psi(1), psi(2), rs, NN, NN,
                                       displace_lattice_planes(NN), L, spacing, X, Y, Z);
                }
                return launch_status();
            }));
            // reads 3 float coordinates, writes the grid (two passes: the
            // windows through the workspace, then summed into the grid)
            MITOS_TRY(timed(s, "cic_deposit", two_pass ? 12.0 * np : 12.0 * nl + 8.0 * np, [&] {
                if constexpr (sizeof(M) == 4) {
                    if (two_pass) {
                        MITOS_TRY((cic_lattice_launch<M, true>(X, Y, Z, NN, L, cic(), cic_ws,
                                                               K, s)));
                        return launch_status();
                    }
                }
                if (NN % 32 == 0 && Ml == NN) {
                    MITOS_TRY((cic_lattice_launch<M, false>(X, Y, Z, NN, L, cic(), nullptr,
                                                            nullptr, s)));
                    return launch_status();
                }
                // another lattice than the grid's: sorted by tile, in the A grids
                // (free once the displacement grids are made)
                const size_t room = sizeof(cx<T>) * (size_t)csize * 3;
                if (cic_sort_pays(NN, nl, room))
                    return cic_sorted<M>(X, Y, Z, nl, NN, L, cic(), A, room, s);
                hipLaunchKernelGGL(k_cic<M>, dim3(nblk(nl)), dim3(256), 0, s, X, Y, Z, nl, NN, L,
                                   cic());
                return launch_status();
            }));
            if constexpr (sizeof(M) == 4) {
                if (two_pass) {
                    MITOS_TRY(timed(s, "cic_gather", 8.0 * np, [&] {
                        MITOS_TRY(cic_gather_launch<M>(NN, cic(), cic_ws, s));
                        return launch_status();
                    }));
                    MITOS_TRY(timed(s, "cic_far", 0.0, [&] {
                        MITOS_TRY(cic_far_launch<M>(X, Y, Z, NN, L, cic(), cic_ws, K, s));
                        return launch_status();
                    }));
                }
            }
        }
        mark(6);
        // 11. density r2c (overdensity on load), 12. P(k) with CIC window
        // delta = sum_w * N^3 / npart - 1 (analyse/src/mitos_read.c:363-376)
        CicLoader<T> ld{cic(), (long)NN, cic_norm()};
        MITOS_TRY(timed(s, "density_z_r2c", 8.0 * np + G, [&] {
            return zr2c_pass_tuned<T, NN>(sched.v[TUNE_Z_R2C], ld, K, hs, 1, 0, OpNone(), s);
        }));
        // y and x out of place through a(0) (free once the displacement
        // grids are made)
        MITOS_TRY(timed(s, "density_y_fwd", 2 * G, [&] {
            return strided_pass_tuned<T, NN, 1, -1>(sched.v[TUNE_Y_FWD], K, a(0), hs, OpNone(), s);
        }));
        MITOS_TRY(timed(s, "density_x_fwd", 2 * G, [&] {
            return strided_pass_tuned<T, NN, 0, -1>(sched.v[TUNE_X_FWD], a(0), K, hs, OpNone(), s);
        }));
        const double* w2 = window_table(NN, L, 2);
        if (!w2) return MITOS_ERR_ALLOC;
        PkCicTransform xf{sfwd, w2, NN};
        MITOS_TRY(timed(s, "pk_bins", G, [&] {
            return pk_run<T, PkCicTransform>(K, K, NN, hs, L, cfg.bins, xf, nullptr, nullptr,
                                             s, pk_dst ? pk_dst : pk_sums,
                                             obs_dst ? obs_dst : pk_obs, pk_part, pk_cnt);
        }));
        mark(7);
        return MITOS_OK;
    });
}

}  // namespace mitos
