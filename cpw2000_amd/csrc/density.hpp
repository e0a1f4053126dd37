// Band density per z-plane (FP64): occ |psi(r)|^2 summed over groups of bands,
// from the z-column buffer of the inverse column kernels.  Used by the density
// (Src/omp/charge_by_fft.f90:170-197) and by the local part of the forces.
#pragma once

#include "fft_fast.hpp"
#include "fft_reg.hpp"

namespace cpwgpu {

// per (z, band group): rho(x,y) = sum_{bands in group} occ |psi(x,y,z)|^2 into
// rhor[grp][z][y][x], for lengths and boxes without a register shape.  LDS:
// tw1[N1] tw2[N2] static; dynamic sub[N2][nxp], rows[RB][row_stride], acc[N2][N1].
template <int N1, int N2>
__global__ __launch_bounds__(FT) void k_density_fast(const cplx<double> *__restrict__ colbuf,
                                                     const int *__restrict__ col_uy,
                                                     const double *__restrict__ occ,
                                                     const double2 *__restrict__ tw1g,
                                                     const double2 *__restrict__ tw2g, FftGeom g,
                                                     int nb, int bpg, double *__restrict__ rhor) {
    typedef double R;
    constexpr int A1 = split_a(N1), B1 = N1 / A1;
    constexpr int RB = FT / B1;
    constexpr int RS = row_stride<N1>();
    __shared__ cplx<R> tw1[N1];
    __shared__ cplx<R> tw2[N2];
    extern __shared__ __align__(16) unsigned char smem_raw[];
    const int nx = g.nx, kd1 = g.kd[0];
    const int nxp = nx | 1;
    cplx<R> *sub = reinterpret_cast<cplx<R> *>(smem_raw);  // [N2][nxp]
    cplx<R> *rows = sub + N2 * nxp;                        // [RB][RS]
    R *acc = reinterpret_cast<R *>(rows + RB * RS);        // [N2][N1]
    const int n3 = g.n[2];
    const int z = blockIdx.x % n3, grp = blockIdx.x / n3;
    const int b0 = grp * bpg, b1 = min(nb, b0 + bpg);
    load_twiddles(tw1, tw1g, N1);
    load_twiddles(tw2, tw2g, N2);
    for (int t = threadIdx.x; t < N2 * N1; t += FT) acc[t] = 0.0;
    const int xhi = N1 - kd1, ushift = N1 - nx;
    const int r = threadIdx.x / B1, t = threadIdx.x - (threadIdx.x / B1) * B1;
    cplx<R> *row = rows + r * RS;
    for (int b = b0; b < b1; b++) {
        for (int q = threadIdx.x; q < N2 * nxp; q += FT) sub[q] = mk<R>(0, 0);
        __syncthreads();
        const cplx<R> *cb = colbuf + ((long)b * n3 + z) * g.ncolp;
        for (int c = threadIdx.x; c < g.ncol; c += FT) {
            const int uy = col_uy[c];
            sub[(uy >> 16) * nxp + (uy & 0xffff)] = cb[c];
        }
        __syncthreads();
        line_fft<R, N2, +1>(sub, nx, 1, nxp, tw2);
        const R w = occ ? occ[b] : 1.0;
        for (int y0 = 0; y0 < N2; y0 += RB) {
            const int y = y0 + r;
            const bool act = r < RB && y < N2;
            cplx<R> v[B1 > A1 ? B1 : A1];
            if (act && t < A1) {
#pragma unroll
                for (int j = 0; j < B1; j++) {
                    const int x = t + A1 * j;
                    v[j] = mk<R>(0, 0);
                    if (x <= kd1) v[j] = sub[y * nxp + x];
                    else if (x >= xhi) v[j] = sub[y * nxp + x - ushift];
                }
                dft<B1, +1, R>(v);
#pragma unroll
                for (int k = 0; k < B1; k++) row[rpos<N1>(t + A1 * k)] = k == 0 ? v[0] : cmul(v[k], tw1[t * k]);
            }
            __syncthreads();
            if (act) {
#pragma unroll
                for (int s = 0; s < A1; s++) v[s] = row[rpos<N1>(s + A1 * t)];
                dft<A1, +1, R>(v);
                // each (y, x = t + B1 q) belongs to this thread alone
#pragma unroll
                for (int q = 0; q < A1; q++) acc[y * N1 + t + B1 * q] += w * (v[q].x * v[q].x + v[q].y * v[q].y);
            }
            __syncthreads();
        }
    }
    __syncthreads();
    double *o = rhor + ((long)grp * n3 + z) * (N2 * N1);
    for (int q = threadIdx.x; q < N2 * N1; q += FT) o[q] = acc[q];
}

// Register-line variant of the density pass (the line layout of k_plane_reg):
// per (z, band group) each band's y/x-box sub-plane (LDS, with a zero column)
// goes through the inverse y and x transforms.  An x-row task keeps the same
// rows for every band of the group, so occ |psi(x, y)|^2 accumulates in the
// registers of the lane that holds (x, y) (x = MX k2 + k after the
// decimation-in-frequency transform), and each block writes its rho(x, y) plane
// once: rhor[grp][z][y][x], summed over groups in a fixed order afterwards.
// Grid: n3 * ceil(nb / bpg) blocks of T threads.
// PR: the sphere box lies inside N/4 (checked by the caller): row stride at
// compile time (SC), and the register slots that hold only x (y) outside the box
// are known zeros (as in k_plane_reg).  YW: y lines by the wave-exchanged LDS
// transform (GY unused).
// Bound by FP64 issue of the transforms, so the work of a band is what counts:
// the z-column map is read once per block and the columns of the next band are
// loaded while this one is transformed, where the registers allow it.
template <int N, int GX, int GY, int T, int W, bool YW, bool PR, int SC>
__global__ __launch_bounds__(T, W) void k_density_reg(const cplx<double> *__restrict__ colbuf,
                                                   const int *__restrict__ col_uy,
                                                   const double *__restrict__ occ,
                                                   const double2 *__restrict__ twg, FftGeom g, int nb,
                                                   int bpg, int S_arg, double *__restrict__ rhor) {
    typedef double R;
    static_assert(N % GX == 0 && N % GY == 0 && T % 64 == 0, "bad plane shape");
    const int S = SC ? SC : S_arg;
    constexpr int MX = N / GX, MY = N / GY;
    constexpr u64mask XB = PR ? box_slots(N, GX, MX, N / 4) : full_mask(MX);
    constexpr u64mask YB = PR ? box_slots(N, GY, MY, N / 4) : full_mask(MY);
    constexpr int TX = T / GX;                 // x-row tasks per round
    constexpr int RPT = (N + TX - 1) / TX;     // rows per x task
    extern __shared__ __align__(16) unsigned char smem_raw[];
    cplx<R> *twN = reinterpret_cast<cplx<R> *>(smem_raw);  // [N]
    cplx<R> *sub = twN + N;                                 // [N][S]
    const int n3 = g.n[2];
    const int z = blockIdx.x % n3, grp = blockIdx.x / n3;
    const int b0 = grp * bpg, b1 = min(nb, b0 + bpg);
    const int nx = g.nx, kd1 = g.kd[0], ushift = N - nx, xhi = N - kd1;
    const int tid = threadIdx.x;
    // NPRE columns per thread go through registers (clamped: ncol >= 1), the others
    // through gather_plane; p0..p3: their places in the sub-plane
    // (named values of a vector type: arrays and structures go to scratch memory)
    typedef double V2 __attribute__((ext_vector_type(2)));
    constexpr int NPRE = 4;
    const long bstep = (long)n3 * g.ncolp;
    const cplx<R> *cb = colbuf + ((long)b0 * n3 + z) * g.ncolp;
    const int c0 = min(tid, g.ncol - 1), c1 = min(tid + T, g.ncol - 1), c2 = min(tid + 2 * T, g.ncol - 1),
              c3 = min(tid + 3 * T, g.ncol - 1);
    const auto place = [&](int c) {
        const int uy = col_uy[c];
        return (uy >> 16) * S + (uy & 0xffff);
    };
    const int p0 = place(c0), p1 = place(c1), p2 = place(c2), p3 = place(c3);
    const auto col = [](const cplx<R> *p) { return *reinterpret_cast<const V2 *>(p); };
    V2 q0, q1, q2, q3;
    const auto fetch = [&](const cplx<R> *p) {
        q0 = col(p + c0);
        q1 = col(p + c1);
        q2 = col(p + c2);
        q3 = col(p + c3);
    };
    // one band ahead where the registers last (with 9 and more values per lane
    // at 3 waves per SIMD they spill: there before the sub-plane is cleared)
    constexpr bool AHEAD = MX <= 8 || W <= 2;
    if (AHEAD) fetch(cb);
    load_twiddles(twN, twg, N);
    const Lanes<R, GX> LX;
    R racc[RPT][MX];
#pragma unroll
    for (int r = 0; r < RPT; r++)
#pragma unroll
        for (int k = 0; k < MX; k++) racc[r][k] = 0.0;
    for (int b = b0; b < b1; b++, cb += bstep) {
        if (!AHEAD) fetch(cb);
        for (int q = tid; q < N * S; q += T) sub[q] = mk<R>(0, 0);
        __syncthreads();
        // (a clamped column is stored again by its own thread with the same value)
        sub[p0] = mk<R>(q0.x, q0.y);
        sub[p1] = mk<R>(q1.x, q1.y);
        sub[p2] = mk<R>(q2.x, q2.y);
        sub[p3] = mk<R>(q3.x, q3.y);
        gather_plane<R, T>(sub, cb, col_uy, g.ncol, S, NPRE * T);
        __syncthreads();
        if (AHEAD) fetch(b + 1 < b1 ? cb + bstep : cb);  // the last band: its own again, unused
        // inverse y on the nx box lines
        if constexpr (YW) {
            line_fft_wave<R, N, +1, T>(sub, nx, 1, S, twN);
        } else {
            const Lanes<R, GY> LY;
            for (int u = tid / GY; u < nx; u += T / GY) {
                cplx<R> *col = sub + u;
                cplx<R> v[MY];
#pragma unroll
                for (int j = 0; j < MY; j++)
                    if (has_bit(YB, j)) v[j] = col[(LY.g + GY * j) * S];
                line_dif<+1, GY, MY, R, YB>(v, LY, twN);
#pragma unroll
                for (int k = 0; k < MY; k++) col[(k + MY * LY.k2) * S] = v[k];
            }
        }
        __syncthreads();
        // inverse x per row, occ |psi|^2 into the row's registers
        const R w = occ ? occ[b] : 1.0;
#pragma unroll
        for (int r = 0; r < RPT; r++) {
            const int y = tid / GX + r * TX;
            if (y < N) {
                const cplx<R> *row = sub + y * S;
                cplx<R> v[MX];
#pragma unroll
                for (int j = 0; j < MX; j++) {
                    const int x = LX.g + GX * j;
                    if (has_bit(XB, j)) v[j] = row[x <= kd1 ? x : x >= xhi ? x - ushift : nx];
                }
                line_dif<+1, GX, MX, R, XB>(v, LX, twN);
#pragma unroll
                for (int k = 0; k < MX; k++) racc[r][k] += w * (v[k].x * v[k].x + v[k].y * v[k].y);
            }
        }
        __syncthreads();  // the rows are read before the next band clears sub
    }
    double *o = rhor + ((long)grp * n3 + z) * (N * N);
#pragma unroll
    for (int r = 0; r < RPT; r++) {
        const int y = tid / GX + r * TX;
        if (y < N) {
#pragma unroll
            for (int k = 0; k < MX; k++) o[y * N + MX * LX.k2 + k] = racc[r][k];
        }
    }
}

}  // namespace cpwgpu
