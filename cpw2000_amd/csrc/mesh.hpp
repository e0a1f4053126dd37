// Specialised mesh lengths: which kernels exist for a length, and the launchers
// of one length (bodies in mesh_launch.hpp, instantiated per length in
// mesh.hip so that the lengths compile side by side).
#pragma once

#include "host.hpp"
#include "fft_fast.hpp"
#include "fft_reg.hpp"
#include "fft_wave.hpp"
#include "fft_col_reg.hpp"

namespace cpwgpu {

// ---- specialised kernels: mesh lengths with a two-pass split ---------------
#define CPW_FAST_SIZES(X) X(24) X(48) X(64) X(72) X(80) X(96) X(108) X(128)

enum LocalStage { ST_COL_BWD, ST_PLANE, ST_COL_FWD };

struct LocalArgs {
    const double2 *psi;
    long ldp;
    double2 *hpsi;
    long ldh;
    int nb;
    int mode;  // COLF_ACC / COLF_KIN: what the gather adds to local/N
};

// ---- plane stage variants ---------------------------------------------------
// 0: k_plane_fast (LDS two-pass lines); 4..6: k_plane_wave (LDS two-pass
// lines, wave-local exchanges) with 256, 192 and 128 threads per block; the
// others: k_plane_reg shapes (x lanes GX, y lanes GY, planes per block P,
// threads T, waves per SIMD W, y lines through the LDS wave transform YW,
// box pruning PR) per precision.
struct RegShapeT {
    int GX, GY, P, T, W;
    bool YW, PR;
};
template <typename R> constexpr RegShapeT reg_shape(int v);
template <> constexpr RegShapeT reg_shape<float>(int v) {
    // 1-3 spill-free at 72: 67, 74 and 127 VGPRs
    return v == 1 ? RegShapeT{8, 8, 1, 256, 5, false, false}
         : v == 2 ? RegShapeT{8, 8, 2, 256, 4, false, false}
         : v == 3 ? RegShapeT{4, 4, 1, 256, 3, false, false}
         : v == 7 ? RegShapeT{8, 8, 1, 256, 5, true, false}
         : v == 8 ? RegShapeT{2, 2, 1, 256, 3, true, true}
         : v == 9 ? RegShapeT{4, 4, 1, 256, 4, true, true}
         : v == 10 ? RegShapeT{8, 8, 1, 256, 5, true, true}
         : v == 11 ? RegShapeT{2, 4, 1, 256, 3, false, true}
                   : RegShapeT{0, 0, 0, 0, 0, false, false};
}
template <> constexpr RegShapeT reg_shape<double>(int v) {
    return v == 1 ? RegShapeT{8, 8, 1, 256, 3, false, false}
         : v == 2 ? RegShapeT{8, 8, 1, 320, 4, false, false}
         : v == 3 ? RegShapeT{4, 8, 1, 256, 3, false, false}
         : v == 7 ? RegShapeT{8, 8, 1, 256, 3, true, false}
         : v == 8 ? RegShapeT{4, 4, 1, 256, 3, true, true}
         : v == 9 ? RegShapeT{8, 8, 1, 256, 3, true, true}
         : v == 10 ? RegShapeT{4, 4, 1, 256, 3, false, true}
         : v == 11 ? RegShapeT{8, 8, 1, 256, 3, false, true}
                   : RegShapeT{0, 0, 0, 0, 0, false, false};
}
constexpr int NPLANE_VAR = 12;
constexpr int WAVE_T[3] = {256, 192, 128};
constexpr bool is_reg_variant(int v) { return (v >= 1 && v <= 3) || (v >= 7 && v < NPLANE_VAR); }

// a register shape is built for a mesh length when both splits divide N and a
// lane holds at most 288 bytes of one line
template <typename R, int N, int GX, int GY> constexpr bool reg_ok() {
    return GX > 0 && GY > 0 && N % GX == 0 && N % GY == 0 && first_factor(N / GX) <= 5 &&
           first_factor(N / GY) <= 5 && 2 * sizeof(R) * (N / GX) <= 288 && 2 * sizeof(R) * (N / GY) <= 288 &&
           N / GX <= 64 && N / GY <= 64;
}
template <typename R, int N> constexpr bool reg_var_ok(int v) {
#define CPW_RV(V) (v == V && reg_ok<R, N, reg_shape<R>(V).GX, reg_shape<R>(V).GY>())
    return CPW_RV(1) || CPW_RV(2) || CPW_RV(3) || CPW_RV(7) || CPW_RV(8) || CPW_RV(9) || CPW_RV(10) ||
           CPW_RV(11);
#undef CPW_RV
}
// a pruned shape needs the sphere box inside |x|, |y| <= N/4 (true on the
// meshes size_fft chooses for the density, n >= 4 kd + 1)
inline bool prune_fits(const FftGeom &g) { return 4 * g.kd[0] <= g.n[0] && 4 * g.kd[1] <= g.n[1]; }

// LDS row stride of the register variant's sub-plane for nx box columns
inline int reg_stride(int nx) { return plane_sub_stride(nx); }

// ---- register column kernels -------------------------------------------------
// lanes per z column: 8 where the column fits in registers, else 4
template <typename R, int N> constexpr int col_reg_g() {
    return reg_ok<R, N, 8, 8>() ? 8 : reg_ok<R, N, 4, 4>() ? 4 : 0;
}
template <typename R, int N> constexpr bool col_reg_built() { return col_reg_g<R, N>() > 0; }
// the sphere box inside |z| <= N3/4: the pruned register column kernels
inline bool col_prune_fits(const FftGeom &g) { return 4 * g.kd[2] <= g.n[2]; }

// whether the wave-exchange variant v (4..6) fits in LDS for nx box columns
template <typename R, int N> bool plane_wave_fits(int v, int nx) {
    const size_t stat = sizeof(cplx<R>) * 2 * N;
    const size_t dyn = v == 4 ? plane_wave_lds<R, N, WAVE_T[0]>(nx)
                       : v == 5 ? plane_wave_lds<R, N, WAVE_T[1]>(nx) : plane_wave_lds<R, N, WAVE_T[2]>(nx);
    return dyn + stat <= 160 * 1024;
}

template <typename R, int N> constexpr bool plane_var_ok(int v) {
    return v == 0 || (v >= 4 && v <= 6) || reg_var_ok<R, N>(v);
}

// default plane variant of a mesh length
template <typename R, int N> constexpr int plane_var_default() { return 0; }

// register shape of the coupled two-component plane kernel: (x lanes, y
// lanes, threads, waves per SIMD); both components' rows live in registers.
// FP64: the two sub-planes (about 86 KB at 72) allow one block per CU, so the
// block has 512 threads for 2 waves per SIMD (184 VGPRs fit that budget).
template <typename R> struct SpinShape;
template <> struct SpinShape<float> { static constexpr int GX = 8, GY = 8, T = 256, W = 3; };
template <> struct SpinShape<double> { static constexpr int GX = 8, GY = 8, T = 512, W = 2; };
template <typename R, int N> constexpr bool spin_reg_ok() {
    return reg_ok<R, N, SpinShape<R>::GX, SpinShape<R>::GY>();
}

// register shape of the density pass: x lanes, y lanes, waves per SIMD
constexpr int DEN_GX = 8, DEN_GY = 8, DEN_W = 3;
// threads of the register density pass for line length N: the smallest of 256,
// 320 and 384 that keeps a lane's row accumulators (rows per x task x N / GX
// doubles) within 27, for lines of at most 10 values per lane: spill-free at 3
// waves per SIMD (24-72: 256, 80: 320); 0 = not built (96 and 128 spill, 108 has
// no 8-lane split: k_density_fast)
template <int N> constexpr int den_threads() {
    if (!reg_ok<double, N, DEN_GX, DEN_GY>() || N / DEN_GX > 10) return 0;
    for (int t : {256, 320, 384})
        if (((N + t / DEN_GX - 1) / (t / DEN_GX)) * (N / DEN_GX) <= 27) return t;
    return 0;
}
template <int N> constexpr bool den_reg_ok() { return den_threads<N>() > 0; }

// launchers (mesh_launch.hpp)
template <typename R, int N>
int launch_col_fast(cpwgpu_plan_s *p, const LocalArgs &a, cplx<R> *colbuf, int stage, hipStream_t s);
template <typename R, int N>
int launch_col_reg(cpwgpu_plan_s *p, const LocalArgs &a, cplx<R> *colbuf, int stage, hipStream_t s);
template <typename R, int N>
int launch_plane(cpwgpu_plan_s *p, const LocalArgs &a, cplx<R> *colbuf, const R *vr, hipStream_t s);
// var: the plan's resolved two-component plane kernel
template <typename R, int N>
int launch_plane_spin(cpwgpu_plan_s *p, cplx<R> *colbuf, const R *vr, long vstride, int npair, int var, hipStream_t s);
template <int N>
int launch_density(cpwgpu_plan_s *p, const cplx<double> *colbuf, const double *occ, int nb, int bpg,
                   int ngrp, int Q1, int Q2, double2 *t2, hipStream_t s, double *rhor = nullptr);

}  // namespace cpwgpu
