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
// kept: partial transforms along x, y and, per q, z.
//
// Non-local (Src/ALFA/for_str_nl_kb.f90:286-362, :392-398; d beta/d rat_j =
// -2 pi i g_j beta, Src/omp/proj_nl_kb_drat.f90:218-220):
//   f_j(atom) = -sum_n occ_n sum_{a in atom} xnlkb_a 2 Re[conj(P0) 2 pi i Pj]
// with P0 = <beta|psi> and Pj = sum_G g_j conj(beta) psi.  The band sum is taken
// before the plane-wave sum:
//   sum_n occ_n Im[Pj conj(P0)] = sum_G g_j Im[conj(beta_a(G)) Phi_a(G)],
//   Phi_a(G) = sum_n psi_n(G) occ_n conj(P0_an),
// so one product of the back-projection's shape serves all three directions
// where three weighted projections were needed.
// All f are covariant (per unit fractional coordinate); the host converts to
// Cartesian with inv(avec)^T.
#pragma once

#include "fft_fast.hpp"
#include "nl_gemm.hpp"

namespace cpwgpu {

// Occupations travel as kernel arguments, OCC_ARGS at a time: in the order of the
// caller's stream, so that a call does not overwrite those that the call before it
// still reads, and with no wait for a copy from the caller's array.
constexpr int OCC_ARGS = 256;
struct OccArgs {
    double v[OCC_ARGS];
};
__global__ __launch_bounds__(OCC_ARGS) void k_put_occ(const OccArgs a, int n, double *__restrict__ out) {
    if ((int)threadIdx.x < n) out[threadIdx.x] = a.v[threadIdx.x];
}

// sum over band groups of p[grp * step] in group order, eight loads in flight
// (clamped; one after the other they cost a memory round trip each)
__device__ __forceinline__ double sum_groups(const double *__restrict__ p, long step, int ngrp) {
    double s = 0.0;
    for (int g0 = 0; g0 < ngrp; g0 += 8) {
        double v[8];
#pragma unroll
        for (int u = 0; u < 8; u++) v[u] = p[min(g0 + u, ngrp - 1) * step];
#pragma unroll
        for (int u = 0; u < 8; u++)
            if (g0 + u < ngrp) s += v[u];
    }
    return s;
}

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
        s = sum_groups(part + yz * n1 + x, nmesh, ngrp);
    }
    rho[q] = s;
}

// Partial transform along x of RHO_RY rows of one z-plane (grid n3 x
// ceil(n2 / RHO_RY)): rho(x, y) = sum over band groups of rhor[grp][z][y][x] in
// group order, T1[z][y][q1 + Q1] = sum_x e^{-2 pi i q1 x/n1} rho(x, y), |q1| <= Q1.
// Few rows per block, so that the group sums, a read of ngrp planes, come
// from all of the GPU (one block per plane took 140 us at 80^3, 128 bands, for
// the x and y transforms; these two kernels 21 + 7).  Dynamic LDS: tw1[n1]
// (exp(+2 pi i e/n1)), rho[RHO_RY][n1].
constexpr int RHO_RY = 8;
__global__ __launch_bounds__(256) void k_rho_x(const double *__restrict__ rhor, int ngrp, int n1, int n2, int n3,
                                               int Q1, const double2 *__restrict__ tw1g, double2 *__restrict__ t1) {
    extern __shared__ __align__(16) unsigned char smem_raw[];
    const int W1 = 2 * Q1 + 1;
    double2 *tw1 = reinterpret_cast<double2 *>(smem_raw);
    double *acc = reinterpret_cast<double *>(tw1 + n1);
    const int z = blockIdx.x, y0 = blockIdx.y * RHO_RY, ny = min(RHO_RY, n2 - y0);
    const long plane = (long)n1 * n2;
    for (int i = threadIdx.x; i < n1; i += blockDim.x) tw1[i] = tw1g[i];
    for (int i = threadIdx.x; i < ny * n1; i += blockDim.x) {
        acc[i] = sum_groups(rhor + (long)z * plane + (long)y0 * n1 + i, n3 * plane, ngrp);
    }
    __syncthreads();
    for (int idx = threadIdx.x; idx < ny * W1; idx += blockDim.x) {
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
        t1[((long)z * n2 + y0) * W1 + idx] = make_double2(sr, si);
    }
}

// Along y: T2[z][q2 + Q2][q1 + Q1] = sum_y e^{-2 pi i q2 y/n2} T1[z][y][q1].  Grid
// n3 x ceil(W2 W1 / 256).  Dynamic LDS: tw2[n2].
__global__ __launch_bounds__(256) void k_rho_y(const double2 *__restrict__ t1, int n2, int Q1, int Q2,
                                               const double2 *__restrict__ tw2g, double2 *__restrict__ t2) {
    extern __shared__ __align__(16) unsigned char smem_raw[];
    double2 *tw2 = reinterpret_cast<double2 *>(smem_raw);
    for (int i = threadIdx.x; i < n2; i += blockDim.x) tw2[i] = tw2g[i];
    __syncthreads();
    const int W1 = 2 * Q1 + 1, W2 = 2 * Q2 + 1;
    const int z = blockIdx.x, idx = blockIdx.y * 256 + threadIdx.x;
    if (idx >= W2 * W1) return;
    const int q2 = idx / W1 - Q2, q1i = idx - (idx / W1) * W1;
    const int de = ((q2 % n2) + n2) % n2;
    const double2 *src = t1 + (long)z * n2 * W1 + q1i;
    int e = 0;
    double sr = 0.0, si = 0.0;
#pragma unroll 8
    for (int y = 0; y < n2; y++) {
        const double2 a = src[(long)y * W1], w = tw2[e];
        sr += a.x * w.x + a.y * w.y;
        si += a.y * w.x - a.x * w.y;
        e += de;
        if (e >= n2) e -= n2;
    }
    t2[(long)z * W2 * W1 + idx] = make_double2(sr, si);
}

// rho(q) for each listed q: (1/N) sum_z T2 exp(-2 pi i q3 z / N3).  RHO_L lanes
// per q take every RHO_L-th plane each and are added up in lane order: one thread
// per q leaves most of the GPU idle (4,169 q of the 64-atom cell: 28 us, 5 with 8).
constexpr int RHO_L = 8;
__global__ __launch_bounds__(256) void k_rho_q(const double2 *__restrict__ t2, const int *__restrict__ qv, int nq,
                                               const double2 *__restrict__ tw3, int n3, int Q1, int Q2, double inv_n,
                                               double2 *__restrict__ rho) {
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    const int k = min(t / RHO_L, nq - 1), l = t % RHO_L;
    const int q1 = qv[3 * k], q2 = qv[3 * k + 1], q3 = qv[3 * k + 2];
    const int W1 = 2 * Q1 + 1, W2 = 2 * Q2 + 1;
    const long off = (long)(q2 + Q2) * W1 + (q1 + Q1);
    // twiddle index e = q3 z mod n3
    const int d1 = ((q3 % n3) + n3) % n3, de = (d1 * RHO_L) % n3;
    int e = (d1 * l) % n3;
    double sr = 0.0, si = 0.0;
#pragma unroll 4
    for (int z = l; z < n3; z += RHO_L) {
        const double2 a = t2[(long)z * W2 * W1 + off];
        const double2 w = tw3[e];
        sr += a.x * w.x + a.y * w.y;
        si += a.y * w.x - a.x * w.y;
        e += de;
        if (e >= n3) e -= n3;
    }
    for (int h = 1; h < RHO_L; h <<= 1) {
        sr += __shfl_xor(sr, h);
        si += __shfl_xor(si, h);
    }
    if (l == 0 && t / RHO_L < nq) rho[k] = make_double2(sr * inv_n, si * inv_n);
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

// c[a][n] = occ_n conj(P0[n][a]): the small operand of k_force_phi, n fastest
__global__ __launch_bounds__(256) void k_force_coef(const double2 *__restrict__ p0, int nanl, int nb,
                                                    const double *__restrict__ occ, cplx<double> *__restrict__ c) {
    const long t = (long)blockIdx.x * 256 + threadIdx.x;
    if (t >= (long)nanl * nb) return;
    const int n = (int)(t % nb), a = (int)(t / nb);
    const double2 v = p0[(long)n * nanl + a];
    const double w = occ ? occ[n] : 1.0;
    c[t] = mk<double>(w * v.x, -w * v.y);
}

// part[blk][a][j] = sum over this block's plane waves of g_j Im[conj(beta_a) Phi_a],
// Phi = psi c^T.  The product of k_back_direct (its shape 2: 128 plane waves x 32
// rows of the small operand per block, register fragments one chunk of bands
// ahead of the MFMAs), whose tile stays in registers: the epilogue multiplies it by
// the projectors and sums over the plane waves, so Phi (as large as the
// projectors) is never stored.  FP64 MFMA bound: 25.6k plane waves x 256
// projectors x 128 bands 114 us (59 TFLOP/s of the plain complex product), where
// the three weighted projections took 450.
// grid (ceil(mtxd / 128), ceil(nanl / 32)).
constexpr int PHI_NT = 2, PHI_IT = 2, PHI_KPL = 2, PHI_BI = 4 * 16 * PHI_IT, PHI_BA = 16 * PHI_NT;
__global__ __launch_bounds__(GEMM_THREADS, 2) void k_force_phi(
    const cplx<double> *__restrict__ psi, long ldp, const cplx<double> *__restrict__ c,
    const cplx<double> *__restrict__ anl, long lda, const double *__restrict__ gw, int mtxd, int nanl, int nb,
    double *__restrict__ part) {
    typedef MF<double>::v4 v4;
    constexpr int NT = PHI_NT, IT = PHI_IT, KPL = PHI_KPL, KC = 4 * KPL;
    __shared__ double red[4][PHI_BA][3];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int lr = lane & 15, lg = lane >> 4;
    const Tile3 tl = gemm_tile_yfirst(Blk::here());
    const int i0 = tl.x * PHI_BI + wave * 16 * IT;
    const int a0 = tl.y * PHI_BA;
    const cplx<double> *pcol[IT];
#pragma unroll
    for (int q = 0; q < IT; q++) pcol[q] = psi + min(i0 + q * 16 + lr, mtxd - 1);
    const cplx<double> *crow[NT];
#pragma unroll
    for (int t = 0; t < NT; t++) crow[t] = c + (long)min(a0 + t * 16 + lr, nanl - 1) * nb;
    v4 P1[NT][IT], P2[NT][IT], P3[NT][IT];
#pragma unroll
    for (int t = 0; t < NT; t++)
#pragma unroll
        for (int q = 0; q < IT; q++) {
            P1[t][q] = v4{0, 0, 0, 0};
            P2[t][q] = v4{0, 0, 0, 0};
            P3[t][q] = v4{0, 0, 0, 0};
        }
    cplx<double> cv[2][NT][KPL], pv[2][IT][KPL];
    // the tail of the band sum is read at clamped addresses with c masked to zero
    const auto load = [&](cplx<double>(&cc)[NT][KPL], cplx<double>(&pp)[IT][KPL], int k0, bool tail) {
#pragma unroll
        for (int u = 0; u < KPL; u++) {
            const int n = k0 + lg * KPL + u, nc = tail ? min(n, nb - 1) : n;
#pragma unroll
            for (int t = 0; t < NT; t++) {
                const cplx<double> v = crow[t][nc];
                cc[t][u] = tail && n >= nb ? mk<double>(0.0, 0.0) : v;
            }
#pragma unroll
            for (int q = 0; q < IT; q++) pp[q][u] = pcol[q][(long)nc * ldp];
        }
    };
    const auto compute = [&](const cplx<double>(&cc)[NT][KPL], const cplx<double>(&pp)[IT][KPL]) {
#pragma unroll
        for (int u = 0; u < KPL; u++) {
            double ps[IT];
#pragma unroll
            for (int q = 0; q < IT; q++) ps[q] = pp[q][u].x + pp[q][u].y;
#pragma unroll
            for (int t = 0; t < NT; t++) {
                const double cs = cc[t][u].x + cc[t][u].y;
#pragma unroll
                for (int q = 0; q < IT; q++) {
                    P1[t][q] = MF<double>::mma(cc[t][u].x, pp[q][u].x, P1[t][q]);
                    P2[t][q] = MF<double>::mma(cc[t][u].y, pp[q][u].y, P2[t][q]);
                    P3[t][q] = MF<double>::mma(cs, ps[q], P3[t][q]);
                }
            }
        }
    };
    const int nfull = nb / KC;
    if (nfull > 0) {
        load(cv[0], pv[0], 0, false);
        int k = 0;
        for (; k + 2 <= nfull; k += 2) {
            load(cv[1], pv[1], (k + 1) * KC, false);
            __builtin_amdgcn_sched_barrier(0);  // the loads stay above the MFMAs
            compute(cv[0], pv[0]);
            load(cv[0], pv[0], min(k + 2, nfull - 1) * KC, false);
            __builtin_amdgcn_sched_barrier(0);
            compute(cv[1], pv[1]);
        }
        if (k < nfull) compute(cv[0], pv[0]);
    }
    if (nfull * KC < nb) {
        load(cv[0], pv[0], nfull * KC, true);
        compute(cv[0], pv[0]);
    }
    double s[NT][4][3] = {};
#pragma unroll
    for (int q = 0; q < IT; q++) {
        const int i = i0 + q * 16 + lr;
        const bool ok = i < mtxd;
        const int ic = ok ? i : mtxd - 1;
        const double g0 = ok ? gw[ic] : 0.0, g1 = ok ? gw[(long)mtxd + ic] : 0.0, g2 = ok ? gw[2L * mtxd + ic] : 0.0;
#pragma unroll
        for (int t = 0; t < NT; t++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const cplx<double> b = anl[(long)min(a0 + t * 16 + MF<double>::row(lg, r), nanl - 1) * lda + ic];
                const double p1 = P1[t][q][r], p2 = P2[t][q][r], p3 = P3[t][q][r];
                const double im = b.x * (p3 - p1 - p2) - b.y * (p1 - p2);
                s[t][r][0] += g0 * im;
                s[t][r][1] += g1 * im;
                s[t][r][2] += g2 * im;
            }
    }
    // the 16 plane waves of a row are the 16 lanes of a group
#pragma unroll
    for (int t = 0; t < NT; t++)
#pragma unroll
        for (int r = 0; r < 4; r++)
#pragma unroll
            for (int j = 0; j < 3; j++) {
                double v = s[t][r][j];
                for (int h = 1; h < 16; h <<= 1) v += __shfl_xor(v, h);
                if (lr == 0) red[wave][t * 16 + MF<double>::row(lg, r)][j] = v;
            }
    __syncthreads();
    for (int x = threadIdx.x; x < PHI_BA * 3; x += GEMM_THREADS) {
        const int a = x / 3, j = x - 3 * a;
        if (a0 + a < nanl)
            part[((long)tl.x * nanl + a0 + a) * 3 + j] = ((red[0][a][j] + red[1][a][j]) + red[2][a][j]) + red[3][a][j];
    }
}

// Covariant non-local force and non-local energy of one atom per block: its
// projectors are listed in LDS, FNL_CHUNK at a time (in order), and the block
// sums their k_force_phi partials (nblk of them) and occ |P0|^2 in a fixed order.
constexpr int FNL_CHUNK = 256;
__global__ __launch_bounds__(FNL_CHUNK) void k_force_nl(const double *__restrict__ part, int nblk,
                                                        const double2 *__restrict__ p0, int nanl, int nb,
                                                        const double *__restrict__ xnl,
                                                        const double *__restrict__ occ,
                                                        const int *__restrict__ proj_atom,
                                                        double *__restrict__ fout, double *__restrict__ eout) {
    __shared__ double red[3 * FNL_CHUNK];
    __shared__ int list[FNL_CHUNK];
    __shared__ int count[FNL_CHUNK / 64];
    const int atom = blockIdx.x, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    double s0 = 0.0, s1 = 0.0, s2 = 0.0, en = 0.0;
    for (int c0 = 0; c0 < nanl; c0 += FNL_CHUNK) {
        const int a = c0 + (int)threadIdx.x;
        const bool mine = a < nanl && proj_atom[a] == atom;
        const unsigned long long bal = __ballot(mine);
        if (lane == 0) count[wave] = __popcll(bal);
        __syncthreads();
        int at = __popcll(bal & ((1ull << lane) - 1)), m = 0;
        for (int w = 0; w < FNL_CHUNK / 64; w++) {
            if (w < wave) at += count[w];
            m += count[w];
        }
        if (mine) list[at] = a;
        __syncthreads();
        for (int t = threadIdx.x; t < m * nblk; t += FNL_CHUNK) {
            const int al = list[t % m];
            const double w = 2.0 * xnl[al];
            const double *p = part + ((long)(t / m) * nanl + al) * 3;
            s0 += w * p[0];
            s1 += w * p[1];
            s2 += w * p[2];
        }
        for (int t = threadIdx.x; t < m * nb; t += FNL_CHUNK) {
            const int al = list[t % m], n = t / m;
            const double2 v = p0[(long)n * nanl + al];
            en += xnl[al] * (occ ? occ[n] : 1.0) * (v.x * v.x + v.y * v.y);
        }
        __syncthreads();  // the list is read before the next chunk's
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
