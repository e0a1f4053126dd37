// Atomic forces of E = sum_n occ_n <psi_n| V_loc + V_NL |psi_n> at fixed psi
// (FP64), the adjoint of the local and non-local parts of H|psi> with respect
// to the atomic positions.
//
// Local (Src/ALFA/for_str_local_force.f90:102-145):
//   f_j(atom) = 2 pi sum_q q_j Re[i exp(-2 pi i q.rat) f_s(q) conj(rho(q))]
// with rho(q) = (1/N) sum_r rho(r) exp(-i q.r), rho(r) = sum_n occ_n |psi_n(r)|^2
// (Src/omp/charge_by_fft.f90:191-214).  rho(r) is formed per z-plane from the
// z-column buffer of k_col_bwd (same inverse transforms as H|psi>), and only
// its Fourier components on the box of the local potential's q vectors are
// kept: per plane a partial transform along x then y, then along z per q.
//
// Non-local (Src/ALFA/for_str_nl_kb.f90:286-362, :392-398; d beta/d rat_j =
// -2 pi i g_j beta, Src/omp/proj_nl_kb_drat.f90:218-220):
//   f_j(atom) = -sum_n occ_n sum_{a in atom} xnlkb_a 2 Re[conj(P0) 2 pi i Pj]
// with P0 = <beta|psi> and Pj = sum_G g_j conj(beta) psi from the split-K
// projection GEMM with a per-plane-wave weight g_j.
// All f are covariant (per unit fractional coordinate); the host converts to
// Cartesian with inv(avec)^T.
#pragma once

#include "fft_fast.hpp"

namespace cpwgpu {

// rho[(z n2 + y) id + x] = sum over band groups of part[grp][z][y][x] in
// group order (x < n1; the padding x >= n1 of the id-wide layout is zero)
__global__ __launch_bounds__(256) void k_rho_r_reduce(const double *__restrict__ part, int ngrp, int n1,
                                                      int n2, int n3, int id, double *__restrict__ rho) {
    const long q = (long)blockIdx.x * 256 + threadIdx.x;
    const long tot = (long)id * n2 * n3;
    if (q >= tot) return;
    const int x = (int)(q % id);
    const long yz = q / id;
    double s = 0.0;
    if (x < n1) {
        const long nmesh = (long)n1 * n2 * n3;
        const long src = yz * n1 + x;
        for (int gq = 0; gq < ngrp; gq++) s += part[gq * nmesh + src];
    }
    rho[q] = s;
}

// Per z-plane (one block each): rho(x, y) = sum over band groups of
// rhor[grp][z][y][x] in group order, then the partial transforms of
// k_density_fast: T2[z][q2][q1] = sum_y e^{-2 pi i q2 y/n2} sum_x
// e^{-2 pi i q1 x/n1} rho(x, y), |q1| <= Q1, |q2| <= Q2.  Dynamic LDS:
// tw1[n1], tw2[n2] (exp(+2 pi i e/n)), T1[n2][2 Q1 + 1], rho[n2][n1].
__global__ __launch_bounds__(256) void k_rho_partial(const double *__restrict__ rhor, int ngrp, int n1, int n2,
                                                     int n3, int Q1, int Q2, const double2 *__restrict__ tw1g,
                                                     const double2 *__restrict__ tw2g, double2 *__restrict__ t2) {
    extern __shared__ __align__(16) unsigned char smem_raw[];
    const int W1 = 2 * Q1 + 1, W2 = 2 * Q2 + 1;
    double2 *tw1 = reinterpret_cast<double2 *>(smem_raw);
    double2 *tw2 = tw1 + n1;
    double2 *t1 = tw2 + n2;                                  // [n2][W1]
    double *acc = reinterpret_cast<double *>(t1 + n2 * W1);  // [n2][n1]
    const int z = blockIdx.x;
    const long plane = (long)n1 * n2;
    for (int i = threadIdx.x; i < n1; i += blockDim.x) tw1[i] = tw1g[i];
    for (int i = threadIdx.x; i < n2; i += blockDim.x) tw2[i] = tw2g[i];
    for (long i = threadIdx.x; i < plane; i += blockDim.x) {
        double v = 0.0;
        for (int grp = 0; grp < ngrp; grp++) v += rhor[((long)grp * n3 + z) * plane + i];
        acc[i] = v;
    }
    __syncthreads();
    // along x: T1[y][q1 + Q1] = sum_x rho(x, y) conj(tw1[q1 x mod n1])
    for (int idx = threadIdx.x; idx < n2 * W1; idx += blockDim.x) {
        const int y = idx / W1, q1 = idx - y * W1 - Q1;
        const int de = ((q1 % n1) + n1) % n1;
        int e = 0;
        double sr = 0.0, si = 0.0;
        for (int x = 0; x < n1; x++) {
            const double a = acc[y * n1 + x];
            sr += a * tw1[e].x;
            si -= a * tw1[e].y;
            e += de;
            if (e >= n1) e -= n1;
        }
        t1[idx] = make_double2(sr, si);
    }
    __syncthreads();
    // along y: T2[z][q2 + Q2][q1 + Q1] = sum_y T1[y][q1] conj(tw2[q2 y mod n2])
    double2 *out = t2 + (long)z * W2 * W1;
    for (int idx = threadIdx.x; idx < W2 * W1; idx += blockDim.x) {
        const int q2 = idx / W1 - Q2, q1i = idx - (idx / W1) * W1;
        const int de = ((q2 % n2) + n2) % n2;
        int e = 0;
        double sr = 0.0, si = 0.0;
        for (int y = 0; y < n2; y++) {
            const double2 a = t1[y * W1 + q1i], w = tw2[e];
            sr += a.x * w.x + a.y * w.y;
            si += a.y * w.x - a.x * w.y;
            e += de;
            if (e >= n2) e -= n2;
        }
        out[idx] = make_double2(sr, si);
    }
}

// T2s[z][q2][q1] = sum over band groups of T2[grp][z][q2][q1], in group order
__global__ void k_t2_sum(const double2 *__restrict__ t2, long nplane, int ngrp, double2 *__restrict__ t2s) {
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= nplane) return;
    double sr = 0.0, si = 0.0;
    for (int grp = 0; grp < ngrp; grp++) {
        const double2 a = t2[grp * nplane + i];
        sr += a.x;
        si += a.y;
    }
    t2s[i] = make_double2(sr, si);
}

// rho(q) for each listed q: (1/N) sum_z T2s exp(-2 pi i q3 z / N3)
__global__ void k_rho_q(const double2 *__restrict__ t2s, const int *__restrict__ qv, int nq,
                        const double2 *__restrict__ tw3, int n3, int Q1, int Q2, double inv_n,
                        double2 *__restrict__ rho) {
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= nq) return;
    const int q1 = qv[3 * k], q2 = qv[3 * k + 1], q3 = qv[3 * k + 2];
    const int W1 = 2 * Q1 + 1, W2 = 2 * Q2 + 1;
    const long off = (long)(q2 + Q2) * W1 + (q1 + Q1);
    // twiddle index e = q3 z mod n3, advanced by de per plane
    const int de = ((q3 % n3) + n3) % n3;
    int e = 0;
    double sr = 0.0, si = 0.0;
    for (int z = 0; z < n3; z++) {
        const double2 a = t2s[(long)z * W2 * W1 + off];
        const double2 w = tw3[e];
        sr += a.x * w.x + a.y * w.y;
        si += a.y * w.x - a.x * w.y;
        e += de;
        if (e >= n3) e -= n3;
    }
    rho[k] = make_double2(sr * inv_n, si * inv_n);
}

__device__ __forceinline__ void block_sum3(double *red, double v0, double v1, double v2, double *out) {
    red[threadIdx.x] = v0;
    red[blockDim.x + threadIdx.x] = v1;
    red[2 * blockDim.x + threadIdx.x] = v2;
    __syncthreads();
    for (int s = blockDim.x / 2; s > 0; s >>= 1) {
        if (threadIdx.x < s) {
            red[threadIdx.x] += red[threadIdx.x + s];
            red[blockDim.x + threadIdx.x] += red[blockDim.x + threadIdx.x + s];
            red[2 * blockDim.x + threadIdx.x] += red[2 * blockDim.x + threadIdx.x + s];
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        out[0] = red[0];
        out[1] = red[blockDim.x];
        out[2] = red[2 * blockDim.x];
    }
}

// covariant local force of one atom per block (256 threads, fixed-order sums)
__global__ __launch_bounds__(256) void k_force_local(const double2 *__restrict__ rho,
                                                     const int *__restrict__ qv,
                                                     const double *__restrict__ fq, int nq,
                                                     const double *__restrict__ rat,
                                                     const int *__restrict__ species,
                                                     double *__restrict__ fout) {
    __shared__ double red[3 * 256];
    const int atom = blockIdx.x;
    const int sp = species[atom];
    const double r1 = rat[3 * atom], r2 = rat[3 * atom + 1], r3 = rat[3 * atom + 2];
    double s0 = 0.0, s1 = 0.0, s2 = 0.0;
    for (int k = threadIdx.x; k < nq; k += blockDim.x) {
        const int q1 = qv[3 * k], q2 = qv[3 * k + 1], q3 = qv[3 * k + 2];
        double sn, cs;
        sincospi(2.0 * (q1 * r1 + q2 * r2 + q3 * r3), &sn, &cs);
        // i * exp(-i phi) * f * conj(rho): real part
        const double f = fq[(long)sp * nq + k];
        const double2 rh = rho[k];
        // exp(-i phi) conj(rho) = (cs - i sn)(rx - i ry) = (cs rx - sn ry) - i (cs ry + sn rx)
        const double im = -(cs * rh.y + sn * rh.x);
        const double e1 = -f * im;  // Re[i z] = -Im z
        s0 += q1 * e1;
        s1 += q2 * e1;
        s2 += q3 * e1;
    }
    block_sum3(red, s0, s1, s2, fout + 3 * atom);
    if (threadIdx.x == 0) {
        const double tp = 6.283185307179586477;
        fout[3 * atom] *= tp;
        fout[3 * atom + 1] *= tp;
        fout[3 * atom + 2] *= tp;
    }
}

// covariant non-local force and non-local energy of one atom per block.
// p holds 4 matrices (P0, P1, P2, P3), each [band][proj] (nanl fastest).
__global__ __launch_bounds__(256) void k_force_nl(const double2 *__restrict__ p, int nanl, int nb,
                                                  const double *__restrict__ xnl,
                                                  const double *__restrict__ occ,
                                                  const int *__restrict__ proj_atom,
                                                  double *__restrict__ fout,
                                                  double *__restrict__ eout) {
    __shared__ double red[3 * 256];
    const int atom = blockIdx.x;
    const long mat = (long)nanl * nb;
    double s0 = 0.0, s1 = 0.0, s2 = 0.0, en = 0.0;
    for (long idx = threadIdx.x; idx < mat; idx += blockDim.x) {
        const int a = (int)(idx % nanl), n = (int)(idx / nanl);
        if (proj_atom[a] != atom) continue;
        const double w = 2.0 * (occ ? occ[n] : 1.0) * xnl[a];
        const double2 p0 = p[idx];
        en += 0.5 * w * (p0.x * p0.x + p0.y * p0.y);
        double s[3];
#pragma unroll
        for (int j = 0; j < 3; j++) {
            const double2 pj = p[(j + 1) * mat + idx];
            // Re[(-i pj) conj(p0)] = Re[-i (pj conj(p0))] = Im(pj conj(p0))
            s[j] = w * (pj.y * p0.x - pj.x * p0.y);
        }
        s0 += s[0];
        s1 += s[1];
        s2 += s[2];
    }
    block_sum3(red, s0, s1, s2, fout + 3 * atom);
    __syncthreads();
    red[threadIdx.x] = en;
    __syncthreads();
    for (int k = blockDim.x / 2; k > 0; k >>= 1) {
        if (threadIdx.x < k) red[threadIdx.x] += red[threadIdx.x + k];
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        const double tp = 6.283185307179586477;
        fout[3 * atom] *= tp;
        fout[3 * atom + 1] *= tp;
        fout[3 * atom + 2] *= tp;
        eout[atom] = red[0];
    }
}

}  // namespace cpwgpu
