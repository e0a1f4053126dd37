// Bodies of the per-length launchers declared in mesh.hpp.
#pragma once

#include "mesh.hpp"
#include "density.hpp"
#include "spin_plane.hpp"

namespace cpwgpu {

template <typename R, int N>
int launch_col_fast(cpwgpu_plan_s *p, const LocalArgs &a, cplx<R> *colbuf, int stage, hipStream_t s) {
    const FftGeom &g = p->g;
    constexpr int CT = col_tile<N>();
    const int ntiles = (g.ncol + CT - 1) / CT;
    const dim3 grid(8 * ((a.nb + 7) / 8) * ntiles);
    if (stage == ST_COL_BWD) {
        launch_batchable<ColBwdFast<R, N>>(CPWGPU_K_COL_BWD, (k_col_bwd_fast<R, N>), grid, dim3(FT), 0, s, a.psi, a.ldp, colbuf,
                           (const int *)p->col_ptr.p, (const int *)p->ent_i.p,
                           (const int *)p->ent_cz.p, (const double2 *)p->tw[2].p, g, ntiles, a.nb);
    } else {
        launch_batchable<ColFwdFast<R, N>>(CPWGPU_K_COL_FWD, (k_col_fwd_fast<R, N>), grid, dim3(FT), 0, s, a.psi, a.ldp, a.hpsi, a.ldh,
                           (const cplx<R> *)colbuf, (const int *)p->col_ptr.p,
                           (const int *)p->ent_i.p, (const int *)p->ent_cz.p,
                           (const double *)p->ekpg.p, (const double2 *)p->tw[2].p, g, ntiles, a.nb,
                           p->inv_n, a.mode);
    }
    HIPCHK(hipGetLastError());
    return CPWGPU_OK;
}

template <typename R, int N>
int launch_plane_fast(cpwgpu_plan_s *p, const LocalArgs &a, cplx<R> *colbuf, const R *vr, hipStream_t s) {
    const FftGeom &g = p->g;
    const size_t dyn =
        sizeof(cplx<R>) * ((size_t)N * plane_sub_stride(g.nx) + (size_t)plane_rows_fast<N>() * row_stride<N>());
    const size_t stat = sizeof(cplx<R>) * 2 * N;
    if (dyn + stat > 160 * 1024)
        return fail(CPWGPU_ERR_SIZE, "plane of %d x %d does not fit in LDS", N, N);
    static bool attr = false;
    if (!attr) {
        HIPCHK(hipFuncSetAttribute((const void *)k_plane_fast<R, N, N>,
                                   hipFuncAttributeMaxDynamicSharedMemorySize,
                                   (int)(160 * 1024 - stat)));
        attr = true;
    }
    launch_timed(CPWGPU_K_PLANE, (k_plane_fast<R, N, N>), dim3(g.n[2] * a.nb), dim3(FT), dyn, s, colbuf,
                       (const int *)p->col_uy.p, vr, (const double2 *)p->tw[0].p,
                       (const double2 *)p->tw[1].p, g);
    HIPCHK(hipGetLastError());
    return CPWGPU_OK;
}

template <typename R, int N, int V>
int launch_plane_reg(cpwgpu_plan_s *p, const LocalArgs &a, cplx<R> *colbuf, const R *vr,
                     hipStream_t s) {
    constexpr RegShapeT SH = reg_shape<R, N>(V);
    constexpr int GX = SH.GX, GY = SH.GY, P = SH.P, T = SH.T, W = SH.W;
    constexpr bool YW = SH.YW, PR = SH.PR;
    if constexpr (!reg_var_ok<R, N>(V)) {
        return fail(CPWGPU_ERR_MODE, "plane variant %d is not built for N = %d", V, N);
    } else {
        const FftGeom &g = p->g;
        if (PR && !prune_fits(g))
            return fail(CPWGPU_ERR_MODE, "plane variant %d needs the sphere box inside N/4", V);
        const auto go = [&](auto kernel, auto body, int S, bool &attr) -> int {
            const size_t dyn = plane_reg_lds<R, N, P>(S);
            if (dyn > 160 * 1024)
                return fail(CPWGPU_ERR_SIZE, "plane variant %d: %zu bytes of LDS", V, dyn);
            if (!attr) {
                HIPCHK(hipFuncSetAttribute((const void *)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024));
                attr = true;
            }
            const dim3 grid(((a.nb + P - 1) / P) * g.n[2]);
            const int *uy = (const int *)p->col_uy.p;
            const double2 *tw = (const double2 *)p->tw[0].p;
            if constexpr (std::is_void<typename decltype(body)::type>::value)
                launch_timed(CPWGPU_K_PLANE, kernel, grid, dim3(T), dyn, s, colbuf, uy, vr, tw, g, a.nb, S);
            else
                launch_batchable<typename decltype(body)::type>(CPWGPU_K_PLANE, kernel, grid, dim3(T), dyn, s, colbuf, uy,
                                                                vr, tw, g, a.nb, S);
            HIPCHK(hipGetLastError());
            return CPWGPU_OK;
        };
        // body: the default shape of the length can be batched
        struct None { using type = void; };
        const int S = reg_stride(g.nx);
        static bool attr_rt = false;
        if constexpr (PR) {
            constexpr int SC = pr_stride<R, N, V>();
            static bool attr_ct = false;
            struct Body { using type = PlaneReg<R, N, GX, GY, P, T, W, YW, PR, SC>; };
            using B = typename std::conditional<V == plane_var_default<R, N>(), Body, None>::type;
            if (S <= SC) return go(k_plane_reg<R, N, GX, GY, P, T, W, YW, PR, SC>, B{}, SC, attr_ct);
            // kd = N/4 exactly where the stride is N/2 + 1
            if constexpr (SC >= N / 2 + 3 || N % 4 != 0)
                return fail(CPWGPU_ERR_MODE, "plane variant %d: %d box columns exceed its row stride", V, g.nx);
            else
                return go(k_plane_reg<R, N, GX, GY, P, T, W, YW, PR, 0>, None{}, S, attr_rt);
        } else {
            return go(k_plane_reg<R, N, GX, GY, P, T, W, YW, PR, 0>, None{}, S, attr_rt);
        }
    }
}

template <typename R, int N, int T>
int launch_plane_wave(cpwgpu_plan_s *p, const LocalArgs &a, cplx<R> *colbuf, const R *vr, hipStream_t s) {
    const FftGeom &g = p->g;
    const size_t dyn = plane_wave_lds<R, N, T>(g.nx);
    const size_t stat = sizeof(cplx<R>) * 2 * N;
    if (dyn + stat > 160 * 1024)
        return fail(CPWGPU_ERR_SIZE, "plane of %d x %d does not fit in LDS with %d threads", N, N, T);
    static bool attr = false;
    if (!attr) {
        HIPCHK(hipFuncSetAttribute((const void *)k_plane_wave<R, N, N, T, 2>,
                                   hipFuncAttributeMaxDynamicSharedMemorySize, (int)(160 * 1024 - stat)));
        attr = true;
    }
    launch_timed(CPWGPU_K_PLANE, (k_plane_wave<R, N, N, T, 2>), dim3(g.n[2] * a.nb), dim3(T), dyn, s, colbuf,
                       (const int *)p->col_uy.p, vr, (const double2 *)p->tw[0].p, (const double2 *)p->tw[1].p, g);
    HIPCHK(hipGetLastError());
    return CPWGPU_OK;
}

template <typename R, int N>
int launch_col_reg(cpwgpu_plan_s *p, const LocalArgs &a, cplx<R> *colbuf, int stage, hipStream_t s) {
    constexpr int G = col_reg_g<R, N>();
    if constexpr (G == 0) {
        return fail(CPWGPU_ERR_MODE, "register column kernels are not built for N = %d", N);
    } else {
        const FftGeom &g = p->g;
        constexpr int CPB = COLR_T / G;
        const int ntiles = (g.ncol + CPB - 1) / CPB;
        const dim3 grid(8 * ((a.nb + 7) / 8) * ntiles);
        const bool pr = col_prune_fits(g);
        const double2 *tw3 = (const double2 *)p->tw[2].p;
        const int *zm = (const int *)p->zmap.p;
        if (stage == ST_COL_BWD) {
            if constexpr (col_reg_inverse<R, N>()) {
                if (pr)
                    launch_batchable<ColBwdReg<R, N, G, true>>(CPWGPU_K_COL_BWD, (k_col_bwd_reg<R, N, G, true>), grid, dim3(COLR_T), 0, s, a.psi, a.ldp, colbuf,
                                       zm, tw3, g, ntiles, a.nb);
                else
                    launch_timed(CPWGPU_K_COL_BWD, (k_col_bwd_reg<R, N, G, false>), grid, dim3(COLR_T), 0, s, a.psi, a.ldp, colbuf,
                                       zm, tw3, g, ntiles, a.nb);
            } else {
                return fail(CPWGPU_ERR_MODE, "register inverse column kernels are not built for N = %d", N);
            }
        } else {
            if (pr)
                launch_batchable<ColFwdReg<R, N, G, true>>(CPWGPU_K_COL_FWD, (k_col_fwd_reg<R, N, G, true>), grid, dim3(COLR_T), 0, s, a.psi, a.ldp, a.hpsi,
                                   a.ldh, (const cplx<R> *)colbuf, zm, (const double *)p->ekpg.p, tw3, g, ntiles,
                                   a.nb, p->inv_n, a.mode);
            else
                launch_timed(CPWGPU_K_COL_FWD, (k_col_fwd_reg<R, N, G, false>), grid, dim3(COLR_T), 0, s, a.psi, a.ldp, a.hpsi,
                                   a.ldh, (const cplx<R> *)colbuf, zm, (const double *)p->ekpg.p, tw3, g, ntiles,
                                   a.nb, p->inv_n, a.mode);
        }
        HIPCHK(hipGetLastError());
        return CPWGPU_OK;
    }
}

template <typename R, int N>
int launch_plane(cpwgpu_plan_s *p, const LocalArgs &a, cplx<R> *colbuf, const R *vr, int v, hipStream_t s) {
#define CPW_LR(V) if (v == V) return launch_plane_reg<R, N, V>(p, a, colbuf, vr, s);
    CPW_LR(1) CPW_LR(2) CPW_LR(3) CPW_LR(7) CPW_LR(8) CPW_LR(9) CPW_LR(10) CPW_LR(11)
#undef CPW_LR
    if constexpr (full_length(N)) {
        if (v == 4) return launch_plane_wave<R, N, WAVE_T[0]>(p, a, colbuf, vr, s);
        if (v == 5) return launch_plane_wave<R, N, WAVE_T[1]>(p, a, colbuf, vr, s);
        if (v == 6) return launch_plane_wave<R, N, WAVE_T[2]>(p, a, colbuf, vr, s);
        return launch_plane_fast<R, N>(p, a, colbuf, vr, s);
    } else {
        return fail(CPWGPU_ERR_MODE, "plane variant %d is not built for N = %d", v, N);
    }
}

template <typename R, int N>
int launch_plane_spin_reg(cpwgpu_plan_s *p, cplx<R> *colbuf, const R *vr, long vstride, int npair,
                          hipStream_t s) {
    if constexpr (!spin_reg_ok<R, N>()) {
        return fail(CPWGPU_ERR_MODE, "register two-component plane kernel is not built for N = %d", N);
    } else {
        const FftGeom &g = p->g;
        const auto go = [&](auto kernel, int S, int T, bool &attr) -> int {
            const size_t dyn = sizeof(cplx<R>) * ((size_t)N + 2 * (size_t)N * S);
            if (dyn > 160 * 1024)
                return fail(CPWGPU_ERR_SIZE, "two-component plane of %d x %d does not fit in LDS", N, N);
            if (!attr) {
                HIPCHK(hipFuncSetAttribute((const void *)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024));
                attr = true;
            }
            launch_timed(CPWGPU_K_PLANE, kernel, dim3(g.n[2] * npair), dim3(T), dyn, s, colbuf,
                         (const int *)p->col_uy.p, vr, vstride, (const double2 *)p->tw[0].p, g, npair, S);
            HIPCHK(hipGetLastError());
            return CPWGPU_OK;
        };
        static bool attr_p = false, attr_u = false;
        using P = SpinShape<R, N, true>;
        using U = SpinShape<R, N, false>;
        // a box inside N/4: the pruned shape.  Its row stride holds every such box: where
        // two planes of it do not fit (128 in FP64), those of a wider box do not either
        if constexpr (sizeof(cplx<R>) * ((size_t)N + 2 * (size_t)N * pr_sub_stride<N>()) > 160 * 1024)
            return fail(CPWGPU_ERR_SIZE, "two-component plane of %d x %d does not fit in LDS", N, N);
        else if (prune_fits(g))
            return go(k_plane_spin_reg<R, N, P::GX, P::GY, P::T, P::W, true>, pr_sub_stride<N>(), P::T, attr_p);
        else
            return go(k_plane_spin_reg<R, N, U::GX, U::GY, U::T, U::W, false>, reg_stride(g.nx), U::T, attr_u);
    }
}

template <typename R, int N>
int launch_plane_spin(cpwgpu_plan_s *p, cplx<R> *colbuf, const R *vr, long vstride, int npair, int var,
                      hipStream_t s) {
    if (var == 1) return launch_plane_spin_reg<R, N>(p, colbuf, vr, vstride, npair, s);
    const FftGeom &g = p->g;
    const size_t dyn = sizeof(cplx<R>) * (2 * (size_t)N * plane_sub_stride(g.nx) +
                                          (size_t)plane_rows_fast<N>() * row_stride<N>());
    const size_t stat = sizeof(cplx<R>) * 2 * N;
    if (dyn + stat > 160 * 1024)
        return fail(CPWGPU_ERR_SIZE, "two-component plane of %d x %d does not fit in LDS", N, N);
    static bool attr = false;
    if (!attr) {
        HIPCHK(hipFuncSetAttribute((const void *)k_plane_spin<R, N, N>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                   (int)(160 * 1024 - stat)));
        attr = true;
    }
    launch_timed(CPWGPU_K_PLANE, (k_plane_spin<R, N, N>), dim3(g.n[2] * npair), dim3(FT), dyn, s, colbuf,
                       (const int *)p->col_uy.p, vr, vstride, (const double2 *)p->tw[0].p,
                       (const double2 *)p->tw[1].p, g, npair);
    HIPCHK(hipGetLastError());
    return CPWGPU_OK;
}

template <int N>
int launch_density(cpwgpu_plan_s *p, const cplx<double> *colbuf, const double *occ, int nb, int bpg, hipStream_t s,
                   double *rhor) {
    const FftGeom &g = p->g;
    const bool pr = den_prune_fits<N>(g);
    const int ngrp = (nb + bpg - 1) / bpg;
    const int *uy = (const int *)p->col_uy.p;
    const double2 *tw = (const double2 *)p->tw[0].p;
    const auto go = [&](auto kernel, int S, int T, bool &attr) -> int {
        const size_t dyn = 16 * ((size_t)N + (size_t)N * S);
        if (dyn > 160 * 1024) return fail(CPWGPU_ERR_SIZE, "density plane %d does not fit in LDS", N);
        if (!attr) {
            HIPCHK(hipFuncSetAttribute((const void *)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024));
            attr = true;
        }
        hipLaunchKernelGGL(kernel, dim3(g.n[2] * ngrp), dim3(T), dyn, s, colbuf, uy, occ, tw, g, nb, bpg, S, rhor);
        HIPCHK(hipGetLastError());
        return CPWGPU_OK;
    };
    constexpr int G = DEN_G;
    if constexpr (den_reg_ok<N>(true)) {
        static bool attr_p = false;
        constexpr int T = den_threads<N>(true), SC = den_stride<N>();
        if (pr) return go(k_density_reg<N, G, G, T, den_waves<N>(), true, true, SC>, SC, T, attr_p);
    }
    if constexpr (den_reg_ok<N>(false)) {
        static bool attr_u = false;
        constexpr int T = den_threads<N>(false);
        return go(k_density_reg<N, G, G, T, den_waves<N>(), false, false, 0>, reg_stride(g.nx), T, attr_u);
    }
    constexpr int RB = plane_rows_fast<N>();
    const size_t dyn = 16 * ((size_t)N * (g.nx | 1) + (size_t)RB * row_stride<N>()) + 8 * (size_t)N * N;
    const size_t stat = 16 * 2 * (size_t)N;
    if (dyn + stat > 160 * 1024) return fail(CPWGPU_ERR_SIZE, "density plane %d does not fit in LDS", N);
    static bool attr = false;
    if (!attr) {
        HIPCHK(hipFuncSetAttribute((const void *)k_density_fast<N, N>,
                                   hipFuncAttributeMaxDynamicSharedMemorySize, (int)(160 * 1024 - stat)));
        attr = true;
    }
    hipLaunchKernelGGL((k_density_fast<N, N>), dim3(g.n[2] * ngrp), dim3(FT), dyn, s, colbuf, uy, occ, tw,
                       (const double2 *)p->tw[1].p, g, nb, bpg, rhor);
    HIPCHK(hipGetLastError());
    return CPWGPU_OK;
}

}  // namespace cpwgpu
