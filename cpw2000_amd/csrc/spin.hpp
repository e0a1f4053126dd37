// Two-component (spinor) H|psi>, Src/hk_psi/reference/hk_psi_spin_c16.f90.
// psi_sp(2 mxddim, neig): row 2i is the spin-up (s = +1/2) coefficient of
// plane wave i, row 2i+1 the spin-down one.  The components are split into
// scalar bands [up 0..nb) | [down 0..nb) so the scalar column kernels apply;
// the potential acts per plane (k_plane_spin couples the two components for
// the non-collinear case); the results are merged back into the interleaved
// rows.
#pragma once

#include "fft_fast.hpp"

namespace cpwgpu {

constexpr int SP_THREADS = 256;

// s(:, n) = up component of band n, s(:, nb + n) = down component (ld = mtxd)
__global__ __launch_bounds__(SP_THREADS) void k_spin_split(const double2 *__restrict__ psi, long ldp, int mtxd,
                                                           int nb, double2 *__restrict__ s) {
    const int i = blockIdx.x * SP_THREADS + threadIdx.x, n = blockIdx.y;
    if (i >= mtxd || n >= nb) return;
    const double2 *c = psi + (long)n * ldp + 2 * (long)i;
    s[(long)n * mtxd + i] = c[0];
    s[(long)(nb + n) * mtxd + i] = c[1];
}

// hpsi rows 2i / 2i+1 of band n (+)= h(:, n) / h(:, nb + n); add != 0 keeps
// what hpsi holds (the non-local term)
__global__ __launch_bounds__(SP_THREADS) void k_spin_merge(const double2 *__restrict__ h, int mtxd, int nb,
                                                           double2 *__restrict__ hpsi, long ldh, int add) {
    const int i = blockIdx.x * SP_THREADS + threadIdx.x, n = blockIdx.y;
    if (i >= mtxd || n >= nb) return;
    double2 *c = hpsi + (long)n * ldh + 2 * (long)i;
    double2 u = h[(long)n * mtxd + i], d = h[(long)(nb + n) * mtxd + i];
    if (add) {
        const double2 u0 = c[0], d0 = c[1];
        u = make_double2(u.x + u0.x, u.y + u0.y);
        d = make_double2(d.x + d0.x, d.y + d0.y);
    }
    c[0] = u;
    c[1] = d;
}

// Potential components in the layout the plane kernels read (per component
// the vscr layout, ntot values each), from vscr_sp(mxdscr, nsp):
//   nsp = 1: [V1]        nsp = 2: [V1 + V2, V1 - V2]
//   nsp = 4: [V1 + V2, V1 - V2, V3, V4]   (up-up, down-down, sigma_x, sigma_y parts)
template <typename R>
__global__ __launch_bounds__(SP_THREADS) void k_spin_potential(const double *__restrict__ vsp, long ldv, int nsp,
                                                               long ntot, R *__restrict__ out) {
    const long k = (long)blockIdx.x * SP_THREADS + threadIdx.x;
    if (k >= ntot) return;
    const double v1 = vsp[k];
    if (nsp == 1) {
        out[k] = (R)v1;
        return;
    }
    const double v2 = vsp[ldv + k];
    out[k] = (R)(v1 + v2);
    out[ntot + k] = (R)(v1 - v2);
    if (nsp == 4) {
        out[2 * ntot + k] = (R)vsp[2 * ldv + k];
        out[3 * ntot + k] = (R)vsp[3 * ldv + k];
    }
}

}  // namespace cpwgpu
