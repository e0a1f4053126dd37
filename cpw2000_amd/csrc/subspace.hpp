// FP64 subspace step on the GPU: Rayleigh-Ritz with Cholesky
// orthonormalisation, a Hermitian eigensolver, the rotation of psi / H psi and
// the residual norms.
//
// Reference semantics (the FP64 steps of the diagonaliser that calls hk_psi):
//   Src/ditsp/ditsp_c16_ritz.f90:195-200  H_sub = hbas^H bas, diagonalised
//   Src/ditsp/diag_c16.f90:65-86           zheevd of the subspace matrix
//   Src/ditsp/ditsp_c16_ritz.f90:284-287  rotation of the basis
//   Src/ditsp/grsch_loop_c16.f90:100-130  orthonormalisation (Gram-Schmidt;
//                                          here Cholesky of the overlap)
//   Src/ditsp/ditsp_error.f90:70-76        residual ||H psi - eps psi||^2
//
// The nb x nb matrices are column-major complex128 (element (i,j) at i + j*n).
// The dense steps here run in one workgroup of SS_THREADS threads each, for any
// nb; small_eig.hpp holds the Jacobi eigensolver and the faster forms for nb up
// to a few hundred.
#pragma once

#include <hip/hip_runtime.h>

namespace cpwgpu {

constexpr int SS_THREADS = 1024;

__device__ __forceinline__ double2 zmul(double2 a, double2 b) {
    return make_double2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}
__device__ __forceinline__ double2 zmulc(double2 a, double2 b) {  // conj(a) * b
    return make_double2(a.x * b.x + a.y * b.y, a.x * b.y - a.y * b.x);
}
__device__ __forceinline__ double2 zconj(double2 a) { return make_double2(a.x, -a.y); }

// In place: lower Cholesky factor of the Hermitian positive definite a.
// info = 0, or j+1 if the j-th pivot is not positive.
__global__ __launch_bounds__(SS_THREADS) void k_cholesky(double2 *a, int n, int *info) {
    __shared__ double piv;
    __shared__ int bad;
    if (threadIdx.x == 0) bad = 0;
    __syncthreads();
    for (int j = 0; j < n; j++) {
        if (threadIdx.x == 0) {
            const double d = a[j + (long)j * n].x;
            if (!(d > 0.0) && !bad) bad = j + 1;
            piv = d > 0.0 ? sqrt(d) : 1.0;
            a[j + (long)j * n] = make_double2(piv, 0.0);
        }
        __syncthreads();
        const double inv = 1.0 / piv;
        for (int i = j + 1 + threadIdx.x; i < n; i += blockDim.x) {
            double2 v = a[i + (long)j * n];
            a[i + (long)j * n] = make_double2(v.x * inv, v.y * inv);
        }
        __syncthreads();
        const int m = n - j - 1;
        for (long idx = threadIdx.x; idx < (long)m * m; idx += blockDim.x) {
            const int i = j + 1 + (int)(idx % m), k = j + 1 + (int)(idx / m);
            if (i >= k) {
                const double2 lij = a[i + (long)j * n], lkj = a[k + (long)j * n];
                double2 v = a[i + (long)k * n];
                const double2 p = zmul(lij, zconj(lkj));
                a[i + (long)k * n] = make_double2(v.x - p.x, v.y - p.y);
            }
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) *info = bad;
}

// In place on h: h <- L^-1 h L^-H, with L the lower factor in l.  w is n*n
// scratch.  One thread per column for each triangular solve.
__global__ __launch_bounds__(SS_THREADS) void k_to_standard(const double2 *l, double2 *h, double2 *w,
                                                            int n) {
    // w = L^-1 h  (forward substitution on each column of h)
    for (int c = threadIdx.x; c < n; c += blockDim.x) {
        for (int i = 0; i < n; i++) {
            double2 s = h[i + (long)c * n];
            for (int k = 0; k < i; k++) {
                const double2 p = zmul(l[i + (long)k * n], w[k + (long)c * n]);
                s.x -= p.x;
                s.y -= p.y;
            }
            const double d = 1.0 / l[i + (long)i * n].x;
            w[i + (long)c * n] = make_double2(s.x * d, s.y * d);
        }
    }
    __syncthreads();
    // h = L^-1 w^H, so that h^H = w L^-H = L^-1 h_in L^-H
    for (int c = threadIdx.x; c < n; c += blockDim.x) {
        for (int i = 0; i < n; i++) {
            double2 s = zconj(w[c + (long)i * n]);
            for (int k = 0; k < i; k++) {
                const double2 p = zmul(l[i + (long)k * n], h[k + (long)c * n]);
                s.x -= p.x;
                s.y -= p.y;
            }
            const double d = 1.0 / l[i + (long)i * n].x;
            h[i + (long)c * n] = make_double2(s.x * d, s.y * d);
        }
    }
    __syncthreads();
    // h <- h^H (the result is Hermitian: symmetrise exactly)
    for (long idx = threadIdx.x; idx < (long)n * n; idx += blockDim.x) {
        const int i = (int)(idx % n), j = (int)(idx / n);
        if (i < j) {
            const double2 a = h[i + (long)j * n], b = h[j + (long)i * n];
            // result_ij = conj(h_ji) = h_ij for an exactly Hermitian result: average
            const double2 m = make_double2(0.5 * (b.x + a.x), 0.5 * (-b.y + a.y));
            h[i + (long)j * n] = m;
            h[j + (long)i * n] = make_double2(m.x, -m.y);
        } else if (i == j) {
            h[i + (long)i * n].y = 0.0;
        }
    }
}

// index at slot i in round r of the round-robin schedule of np (even) positions
__device__ __forceinline__ int rr_slot(int i, int r, int np) {
    if (i == 0) return 0;
    int m = (i - 1 - r) % (np - 1);
    if (m < 0) m += np - 1;
    return 1 + m;
}

constexpr int JAC_MAXPAIR = 1024;  // n <= 2048

// In place on v: v <- L^-H v (backward substitution, one thread per column)
__global__ __launch_bounds__(SS_THREADS) void k_back_substitute(const double2 *l, double2 *v, int n) {
    for (int c = threadIdx.x; c < n; c += blockDim.x) {
        for (int i = n - 1; i >= 0; i--) {
            double2 s = v[i + (long)c * n];
            for (int k = i + 1; k < n; k++) {
                // (L^H)_{ik} = conj(L_{ki})
                const double2 p = zmulc(l[k + (long)i * n], v[k + (long)c * n]);
                s.x -= p.x;
                s.y -= p.y;
            }
            const double d = 1.0 / l[i + (long)i * n].x;
            v[i + (long)c * n] = make_double2(s.x * d, s.y * d);
        }
    }
}

// res[n] = sum_i |hpsi_n[i] - eig[n] psi_n[i]|^2  (one block per band, fixed-order tree)
__global__ __launch_bounds__(256) void k_residual(const double2 *__restrict__ psi, long ldp,
                                                  const double2 *__restrict__ hpsi, long ldh,
                                                  const double *__restrict__ eig,
                                                  double *__restrict__ res, int mtxd) {
    __shared__ double red[256];
    const int n = blockIdx.x;
    const double e = eig[n];
    double s = 0.0;
    // eight rows in flight per thread (clamped), added in order: a column is one
    // block's, and a memory round trip per row took twice the time
    constexpr int U = 8;
    for (int i0 = threadIdx.x; i0 < mtxd; i0 += U * 256) {
        double2 p[U], h[U];
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int i = min(i0 + u * 256, mtxd - 1);
            p[u] = psi[(long)n * ldp + i];
            h[u] = hpsi[(long)n * ldh + i];
        }
#pragma unroll
        for (int u = 0; u < U; u++) {
            const double rx = h[u].x - e * p[u].x, ry = h[u].y - e * p[u].y;
            if (i0 + u * 256 < mtxd) s += rx * rx + ry * ry;
        }
    }
    red[threadIdx.x] = s;
    __syncthreads();
    for (int k = blockDim.x / 2; k > 0; k >>= 1) {
        if (threadIdx.x < k) red[threadIdx.x] += red[threadIdx.x + k];
        __syncthreads();
    }
    if (threadIdx.x == 0) res[n] = red[0];
}

// copy nb columns of mtxd rows (ld src -> ld dst)
__global__ void k_copy_cols(const double2 *__restrict__ src, long lds, double2 *__restrict__ dst,
                            long ldd, int rows, int cols) {
    const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= (long)rows * cols) return;
    const int c = (int)(t / rows), r = (int)(t - (long)c * rows);
    dst[(long)c * ldd + r] = src[(long)c * lds + r];
}

}  // namespace cpwgpu
