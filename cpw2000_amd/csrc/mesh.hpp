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
// CPW_FULL_SIZES: every kernel family (all plane variants, density, coupled
// two-component plane).  CPW_FAST_SIZES adds the lengths of the size table that
// small and elongated cells take: column kernels and one pruned register plane
// shape each (with the generic kernels a 36^3 plane stage of 20 bands took 70 us
// against 10, a 32x32x128 one of 72 bands 442 against 41).
#define CPW_FULL_SIZES(X) X(24) X(48) X(64) X(72) X(80) X(96) X(108) X(128)
#define CPW_FAST_SIZES(X) X(18) X(20) X(24) X(32) X(36) X(40) X(48) X(50) X(54) X(64) X(72) X(80) X(96) X(100) X(108) X(128)
constexpr bool full_length(int n) {
#define CPW_IS(N) || n == N
    return false CPW_FULL_SIZES(CPW_IS);
#undef CPW_IS
}

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
constexpr RegShapeT NO_SHAPE{0, 0, 0, 0, 0, false, false};
// Lengths that 8 does not divide go by 4 or 2 lanes with up to 27 values each:
// FP64 gives them the registers of 2 waves per SIMD, as many as their LDS lets
// run (108: one block of 512 threads per CU).
template <typename R, int N> constexpr RegShapeT reg_shape(int v) {
    if constexpr (!full_length(N)) {
        // one pruned shape: 9 in FP64, 10 in FP32
        if (v != (sizeof(R) == 8 ? 9 : 10)) return NO_SHAPE;
        const int w = sizeof(R) == 8 ? 3 : N % 8 == 0 ? 5 : 4;
        // FP64: as many threads as one round of rows takes, by 4 lanes (us per H|psi>
        // call against 256 threads by 8 (36: by 4) lanes: 32, 72 bands on 32 x 32 x 128
        // 106 / 102; 36, 60 bands on 36 x 36 x 72 71 / 70; 40, 60 bands on 40^3 56 / 53)
        if (sizeof(R) == 8 && N == 32) return RegShapeT{4, 4, 1, 128, 4, false, true};
        if (sizeof(R) == 8 && (N == 36 || N == 40)) return RegShapeT{4, 4, 1, 192, w, true, true};
        return N == 18 ? RegShapeT{2, 2, 1, 64, 2, false, true}
             : N == 20 ? RegShapeT{4, 4, 1, 128, w, false, true}
             : N == 36 ? RegShapeT{4, 4, 1, 256, w, true, true}
             : N == 50 || N == 54 ? RegShapeT{2, 2, 1, 128, sizeof(R) == 8 ? 2 : 3, false, true}
             : N == 100 ? (sizeof(R) == 8 ? RegShapeT{4, 4, 1, 512, 2, false, true} : RegShapeT{4, 4, 1, 256, 4, true, true})
                        : RegShapeT{8, 8, 1, 256, w, true, true};
    } else if constexpr (sizeof(R) == 4) {
        // 1-3 spill-free at 72: 67, 74 and 127 VGPRs
        return v == 1 ? RegShapeT{8, 8, 1, 256, 5, false, false}
             : v == 2 ? RegShapeT{8, 8, 2, 256, 4, false, false}
             : v == 3 ? RegShapeT{4, 4, 1, 256, 3, false, false}
             : v == 7 ? RegShapeT{8, 8, 1, 256, 5, true, false}
             : v == 8 ? RegShapeT{2, 2, 1, 256, 3, true, true}
             : v == 9 ? RegShapeT{4, 4, 1, 256, 4, true, true}
             : v == 10 ? RegShapeT{8, 8, 1, 256, 5, true, true}
             : v == 11 ? RegShapeT{2, 4, 1, 256, 3, false, true}
                       : NO_SHAPE;
    } else {
        if (N == 108 && v == 9) return RegShapeT{4, 4, 1, 512, 2, false, true};
        if (N == 128 && v == 10) return RegShapeT{8, 8, 1, 768, 3, false, true};
        return v == 1 ? RegShapeT{8, 8, 1, 256, 3, false, false}
             : v == 2 ? RegShapeT{8, 8, 1, 320, 4, false, false}
             : v == 3 ? RegShapeT{4, 8, 1, 256, 3, false, false}
             : v == 7 ? RegShapeT{8, 8, 1, 256, 3, true, false}
             : v == 8 ? RegShapeT{4, 4, 1, 256, 3, true, true}
             : v == 9 ? RegShapeT{8, 8, 1, 256, 3, true, true}
             : v == 10 ? RegShapeT{4, 4, 1, 256, 3, false, true}
             : v == 11 ? RegShapeT{8, 8, 1, 256, 3, false, true}
                       : NO_SHAPE;
    }
}
constexpr int NPLANE_VAR = 12;
constexpr int WAVE_T[3] = {256, 192, 128};
constexpr bool is_reg_variant(int v) { return (v >= 1 && v <= 3) || (v >= 7 && v < NPLANE_VAR); }

// a register shape is built for a mesh length when both splits divide N and a
// lane holds at most MAXB bytes of one line: 288, or 432 with the registers of
// 2 waves per SIMD
template <typename R, int N, int GX, int GY, int MAXB = 288> constexpr bool reg_ok() {
    return GX > 0 && GY > 0 && N % GX == 0 && N % GY == 0 && first_factor(N / GX) <= 5 &&
           first_factor(N / GY) <= 5 && 2 * sizeof(R) * (N / GX) <= MAXB && 2 * sizeof(R) * (N / GY) <= MAXB &&
           N / GX <= 64 && N / GY <= 64;
}
template <typename R, int N> constexpr int reg_bytes(int v) { return reg_shape<R, N>(v).W <= 2 ? 432 : 288; }
template <typename R, int N> constexpr bool reg_var_ok(int v) {
#define CPW_RV(V) (v == V && reg_ok<R, N, reg_shape<R, N>(V).GX, reg_shape<R, N>(V).GY, reg_bytes<R, N>(V)>())
    return CPW_RV(1) || CPW_RV(2) || CPW_RV(3) || CPW_RV(7) || CPW_RV(8) || CPW_RV(9) || CPW_RV(10) ||
           CPW_RV(11);
#undef CPW_RV
}
// a pruned shape needs the sphere box inside |x|, |y| <= N/4 (true on the
// meshes size_fft chooses for the density, n >= 4 kd + 1)
inline bool prune_fits(const FftGeom &g) { return 4 * g.kd[0] <= g.n[0] && 4 * g.kd[1] <= g.n[1]; }

// LDS row stride of the register variant's sub-plane for nx box columns
inline int reg_stride(int nx) { return plane_sub_stride(nx); }
// Compile-time row stride of a pruned shape.  N/2 + 3 holds every box inside
// N/4; N/2 + 1 (odd) all but the one with kd = N/4 exactly, and is taken where it
// lets one more block run per CU (80: three FP64 blocks instead of two, 181 ->
// 150 us for 64 bands; 72, 96 and 128 gain no block and measured up to 10%
// slower) or where N/2 + 3 is even (18, 50, 54: their box never has kd = N/4).
template <typename R, int N, int V> constexpr int pr_stride() {
    constexpr RegShapeT SH = reg_shape<R, N>(V);
    constexpr int wide = N / 2 + 3, tight = (N / 2 + 1) | 1;
    if (wide % 2 == 0) return tight;
    const int cap = sizeof(R) == 8 ? SH.W * 256 / SH.T : 8;
    const int bw = 160 * 1024 / (2 * (int)sizeof(R) * (N + N * wide));
    const int bt = 160 * 1024 / (2 * (int)sizeof(R) * (N + N * tight));
    return (bt < cap ? bt : cap) > (bw < cap ? bw : cap) ? tight : wide;
}

// ---- register column kernels -------------------------------------------------
// lanes per z column: 8 where the column fits in registers, else 4
template <typename R, int N> constexpr int col_reg_g() {
    return reg_ok<R, N, 8, 8>() ? 8 : reg_ok<R, N, 4, 4>() ? 4 : 0;
}
template <typename R, int N> constexpr bool col_reg_built() { return col_reg_g<R, N>() > 0; }
// whether the register lines serve the inverse columns too
template <typename R, int N> constexpr bool col_reg_inverse() {
    return col_reg_built<R, N>() && (sizeof(R) == 4 || N <= 40);
}
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
    return v == 0 || (full_length(N) && v >= 4 && v <= 6) || reg_var_ok<R, N>(v);
}

// Default plane variant of a mesh length for a box inside N/4: the pruned
// register shape that measured fastest (64-128 bands, us, LDS two-pass kernel
// in brackets; FP64 64: 57 [98], 72: 181 [323], 80: 150 [349], 96: 280 [596],
// 108: 1060 [1757], 128: 704 [1484]; FP32 64: 34 [50], 72: 97 [154], 80: 85 [122],
// 96: 148 [284], 108: 489 [735], 128: 473 [607]).
template <typename R, int N> constexpr int plane_var_default() {
    if (sizeof(R) == 4) return N == 96 || N == 108 ? 9 : 10;
    return N == 96 ? 11 : N == 128 ? 10 : 9;
}

// register shape of the coupled two-component plane kernel: (x lanes, y
// lanes, threads, waves per SIMD); both components' rows live in registers.
// FP64: the two sub-planes (about 90 KB at 72) allow one block per CU, whose rows
// are one round of tasks (8 N threads; with 512, 72 rows left 8 of them to a second
// round); a box beyond N/4 needs the registers of 2 waves per SIMD.
template <typename R, int N, bool CS> struct SpinShape {
    static constexpr int GX = 8, GY = 8;
    static constexpr int T = sizeof(R) == 4 ? 256 : CS ? 8 * N : 512, W = sizeof(R) == 4 || CS ? 3 : 2;
};
template <typename R, int N> constexpr bool spin_reg_ok() {
    return reg_ok<R, N, 8, 8>();
}

// Register shapes of the density pass: 8 lanes per line, den_threads() threads,
// den_waves() waves per SIMD, row stride den_stride() for a box inside N/4 (0:
// any box, the stride an argument).  Threads: the smallest of 256, 320 and 384
// that keeps a lane's row accumulators (rows per x task x N / 8 doubles) within
// 27, for lines of at most 10 values per lane (24-72: 256, 80: 320).  For a box
// inside N/4 also 96, at 2 waves per SIMD, and 80 takes 256 threads and the
// tighter stride: three blocks per CU instead of two (128 bands 306 -> 220 us).
// 72, 128 bands: 158 us before the pruning and the whole rounds, 128 with them.
// 108 has no 8-lane split and 128 no room for its accumulators: k_density_fast.
constexpr int DEN_G = 8;
template <int N> constexpr int den_threads(bool pr) {
    if (!reg_ok<double, N, DEN_G, DEN_G>()) return 0;
    if (pr && (N == 80 || N == 96)) return 256;
    if (N / DEN_G > 10) return 0;
    for (int t : {256, 320, 384})
        if (((N + t / DEN_G - 1) / (t / DEN_G)) * (N / DEN_G) <= 27) return t;
    return 0;
}
template <int N> constexpr int den_waves() { return N / DEN_G > 10 ? 2 : 3; }
template <int N> constexpr int den_stride() { return N == 80 ? N / 2 + 1 : pr_sub_stride<N>(); }
template <int N> bool den_prune_fits(const FftGeom &g) { return prune_fits(g) && reg_stride(g.nx) <= den_stride<N>(); }
template <int N> constexpr bool den_reg_ok(bool pr) { return den_threads<N>(pr) > 0; }
// Bands per group of the density pass: a block takes one plane of a group, so
// the groups are chosen to fill whole rounds of the blocks that fit on the GPU at
// once (half a band more per round for its start and its plane of output).  72,
// 128 bands: 10 groups of 13 in one round; groups of 8 took two.
template <int N> int den_bands_per_group(const FftGeom &g, int nb) {
    const bool pr = den_prune_fits<N>(g);
    if (!den_reg_ok<N>(pr)) return 8;
    const long lds = 16 * ((long)N + (long)N * (pr ? den_stride<N>() : reg_stride(g.nx)));
    const int wpb = den_threads<N>(pr) / 64;
    const long slots = 256 * std::max(1L, std::min<long>(160 * 1024 / lds, 4 * den_waves<N>() / wpb));
    int best = 1;
    double cost = HUGE_VAL;
    for (int bpg = std::max(1, nb / 64); bpg <= nb; bpg++) {
        const long ngrp = (nb + bpg - 1) / bpg;
        const double c = (double)((g.n[2] * ngrp + slots - 1) / slots) * (bpg + 0.5);
        if (c < cost) {
            cost = c;
            best = bpg;
        }
    }
    return best;
}

// launchers (mesh_launch.hpp); v: the plane variant, resolved for the mesh
template <typename R, int N>
int launch_col_fast(cpwgpu_plan_s *p, const LocalArgs &a, cplx<R> *colbuf, int stage, hipStream_t s);
template <typename R, int N>
int launch_col_reg(cpwgpu_plan_s *p, const LocalArgs &a, cplx<R> *colbuf, int stage, hipStream_t s);
template <typename R, int N>
int launch_plane(cpwgpu_plan_s *p, const LocalArgs &a, cplx<R> *colbuf, const R *vr, int v, hipStream_t s);
// var: the plan's resolved two-component plane kernel
template <typename R, int N>
int launch_plane_spin(cpwgpu_plan_s *p, cplx<R> *colbuf, const R *vr, long vstride, int npair, int var, hipStream_t s);
template <int N>
int launch_density(cpwgpu_plan_s *p, const cplx<double> *colbuf, const double *occ, int nb, int bpg, hipStream_t s,
                   double *rhor);

}  // namespace cpwgpu
