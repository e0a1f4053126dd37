// The small dense steps of the FP64 Rayleigh-Ritz step: Cholesky factor of the
// overlap, the two triangular solves that bring the subspace matrix to standard
// form, the Hermitian eigenproblem by cyclic Jacobi, and the back-substitution.
// (subspace.hpp holds the one-workgroup solves that matrices beyond SE_MAX take.)
//
// What bounds them is latency, not arithmetic: n is at most a few hundred, a
// step depends on the one before, and every global round trip or division on
// that chain is paid n or more times.  So: the matrix in LDS where it fits
// (Cholesky, Jacobi), one wavefront per column with the column in registers
// (solves, no barrier), and for larger Jacobi matrices one launch per round with
// the matrix spread over the compute units (one memory round trip a round).
// us at n = 128, one workgroup in global memory before / now: Cholesky 382 / 184,
// solves 2263 / 82, Jacobi 28,275 / 3,900 (1,016 rounds of 3.7), back-substitution
// 871 / 300; n = 64, the whole step 4,492 / 1,709.
//
// Every value is computed by the same operations in the same order whatever the
// kernel, with the fused products written out: the phases of the Ritz vectors are
// those of rotations by small elements (an element of 1e-8 |a| turns a vector by a
// phase known to 1e-8), so another order or another choice of the rounded product
// would change them.
#pragma once

#include "subspace.hpp"

namespace cpwgpu {

constexpr int SE_MAX = 256;      // largest n of the solves by columns
constexpr int SE_TRI_MAX = 140;  // largest n whose lower triangle fits in LDS
constexpr int SE_FULL_MAX = 96;  // largest n whose matrix fits in LDS
constexpr int SE_DIAG_MAX = 128; // largest n of k_jacobi_tri (one lane per pair)
constexpr int SE_THREADS = 1024;

// a b and conj(a) b with the second product of each sum rounded first
__device__ __forceinline__ double2 fmul2(double2 a, double2 b) {
    return make_double2(fma(a.x, b.x, -(a.y * b.y)), fma(a.y, b.x, a.x * b.y));
}
__device__ __forceinline__ double2 fmulc2(double2 a, double2 b) {
    return make_double2(fma(a.x, b.x, a.y * b.y), fma(a.x, b.y, -(a.y * b.x)));
}

__host__ __device__ __forceinline__ int tri(int r) { return r * (r + 1) / 2; }  // row r of a packed lower triangle
constexpr size_t se_lds_bytes(int n) { return 16 * (size_t)(n * (n + 1) / 2); }

// Lower Cholesky factor of the Hermitian positive definite a (n x n,
// column-major, lower triangle read): l (lower, column-major; may be a) and
// dinv[j] = 1 / l_jj.  info = 0, or j + 1 if the j-th pivot is not positive.  The
// columns are scaled where they are used, so that a step takes one barrier.
__global__ __launch_bounds__(SE_THREADS) void k_cholesky_lds(const double2 *a, double2 *l,
                                                             double *__restrict__ dinv, int n, int *info) {
    extern __shared__ __align__(16) unsigned char smem_raw[];
    double2 *P = reinterpret_cast<double2 *>(smem_raw);
    const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
    for (int c = ty; c < n; c += 32)
        for (int r = c + tx; r < n; r += 32) P[tri(r) + c] = a[r + (long)c * n];
    __syncthreads();
    int bad = 0;
    for (int j = 0; j < n; j++) {
        const double d = P[tri(j) + j].x;
        if (!(d > 0.0) && !bad) bad = j + 1;
        const double piv = d > 0.0 ? sqrt(d) : 1.0;
        const double inv = 1.0 / piv;
        for (int i = j + 1 + tx; i < n; i += 32) {
            const double2 x = P[tri(i) + j];
            const double2 lij = make_double2(x.x * inv, x.y * inv);
            for (int k = j + 1 + ty; k <= i; k += 32) {
                const double2 y = P[tri(k) + j];
                const double2 lkj = make_double2(y.x * inv, y.y * inv);
                const double2 p = fmulc2(lkj, lij);
                double2 &v = P[tri(i) + k];
                v = make_double2(v.x - p.x, v.y - p.y);
            }
        }
        __syncthreads();
    }
    for (int c = ty; c < n; c += 32) {
        const double d = P[tri(c) + c].x;
        const double piv = d > 0.0 ? sqrt(d) : 1.0;
        const double inv = 1.0 / piv;
        for (int r = c + tx; r < n; r += 32) {
            const double2 x = P[tri(r) + c];
            l[r + (long)c * n] = r == c ? make_double2(piv, 0.0) : make_double2(x.x * inv, x.y * inv);
        }
        if (tx == 0) dinv[c] = inv;
    }
    if (threadIdx.x == 0) *info = bad;
}

// dinv of a factor made elsewhere
__global__ void k_factor_dinv(const double2 *__restrict__ l, double *__restrict__ dinv, int n) {
    const int c = blockIdx.x * blockDim.x + threadIdx.x;
    if (c < n) dinv[c] = 1.0 / l[c + (long)c * n].x;
}

__device__ __forceinline__ double lane_value(double x, int lane) {
    const unsigned long long b = __builtin_bit_cast(unsigned long long, x);
    const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)b, lane);
    const unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)(b >> 32), lane);
    return __builtin_bit_cast(double, ((unsigned long long)hi << 32) | lo);
}

// One forward substitution per wavefront: column c of out = L^-1 in, with L
// column-major in t and dinv its reciprocal diagonal.  in: column c of the matrix,
// or with HERM row c conjugated; INVH: the identity, and out is L^-H (the column
// stored as a conjugated row).  Lane j holds rows j, j + 64, ... (RPL of
// them); a solved value goes to all lanes by readlane, so the chain has no
// memory access: the columns of L are loaded SE_PRE ahead.  Each row subtracts its
// terms in the order of the columns.
constexpr int SE_PRE = 8;
template <int RPL, bool HERM, bool INVH = false>
__global__ __launch_bounds__(64) void k_solve_cols(const double2 *__restrict__ t, const double *__restrict__ dinv,
                                                   const double2 *__restrict__ in, double2 *__restrict__ out, int n) {
    const int c = blockIdx.x, lane = threadIdx.x;
    double2 s[RPL];
    double di[RPL];
#pragma unroll
    for (int q = 0; q < RPL; q++) {
        const int i = min(lane + 64 * q, n - 1);
        s[q] = INVH ? make_double2(i == c ? 1.0 : 0.0, 0.0) : HERM ? zconj(in[c + (long)i * n]) : in[i + (long)c * n];
        di[q] = dinv[i];
    }
    // column k of L at this lane's rows (clamped: rows not below k are not used)
    const auto col = [&](double2(&b)[RPL], int k) {
        const long kc = (long)min(k, n - 1) * n;
#pragma unroll
        for (int q = 0; q < RPL; q++) b[q] = t[min(lane + 64 * q, n - 1) + kc];
    };
    double2 buf[SE_PRE][RPL];
#pragma unroll
    for (int j = 0; j < SE_PRE; j++) col(buf[j], j);
#pragma unroll
    for (int q = 0; q < RPL; q++) {
        const int lo = 64 * q, m = min(n - lo, 64);
        for (int k0 = 0; k0 < m; k0 += SE_PRE) {
#pragma unroll
            for (int j = 0; j < SE_PRE; j++) {
                const int kk = k0 + j;
                if (kk < m) {
                    const double d = lane_value(di[q], kk);
                    const double2 x = make_double2(lane_value(s[q].x, kk) * d, lane_value(s[q].y, kk) * d);
#pragma unroll
                    for (int r = 0; r < RPL; r++) {
                        const double2 p = fmul2(buf[j][r], x);
                        if (lane + 64 * r > lo + kk) s[r] = make_double2(s[r].x - p.x, s[r].y - p.y);
                    }
                    if (lane == kk) s[q] = x;
                    col(buf[j], lo + kk + SE_PRE);
                }
            }
        }
    }
#pragma unroll
    for (int q = 0; q < RPL; q++)
        if (lane + 64 * q < n) {
            if (INVH) out[c + (long)(lane + 64 * q) * n] = zconj(s[q]);
            else out[lane + 64 * q + (long)c * n] = s[q];
        }
}

// In place on v: v <- L^-H v.  Row i subtracts conj(L_ki) v_k for k = i + 1, i + 2,
// ...: a serial chain of n^2 / 2 steps per column, bound by the issue of its FP64
// instructions and LDS reads.  So a lane pair takes a column, one lane the real
// and one the imaginary parts; the columns of a wavefront and the current row of
// L^H are in LDS, the next row on its way.
constexpr int SE_BW = 32;  // columns per block
template <int RPL>
__global__ __launch_bounds__(64) void k_back_cols(const double2 *__restrict__ l, const double *__restrict__ dinv,
                                                  double2 *__restrict__ v, int n) {
    extern __shared__ __align__(16) unsigned char smem_raw[];
    double2 *x = reinterpret_cast<double2 *>(smem_raw);  // [n][SE_BW]
    double2 *row = x + n * SE_BW;                         // [64 * RPL]
    const int lane = threadIdx.x;
    const int c0 = blockIdx.x * SE_BW, nc = min(SE_BW, n - c0);
    for (int e = lane; e < n * nc; e += 64) {
        const int c = e / n, i = e - c * n;
        x[i * SE_BW + c] = v[i + (long)(c0 + c) * n];
    }
    // re: p = fma(l.x, v.x, l.y v.y), im: p = fma(l.x, v.y, (-l.y) v.x)
    const int im = lane & 1;
    double *mine = reinterpret_cast<double *>(x + min(lane >> 1, nc - 1)) + im;
    const double *other = reinterpret_cast<double *>(x + min(lane >> 1, nc - 1)) + (1 - im);
    const double sign = im ? -1.0 : 1.0;
    const auto sync = [] {
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
    };
    double2 nx[RPL];
    const auto fetch = [&](int i) {
#pragma unroll
        for (int q = 0; q < RPL; q++) nx[q] = l[min(lane + 64 * q, n - 1) + (long)i * n];
    };
    fetch(n - 1);
    for (int i = n - 1; i >= 0; i--) {
        sync();
#pragma unroll
        for (int q = 0; q < RPL; q++) row[lane + 64 * q] = nx[q];
        if (i > 0) fetch(i - 1);
        const double d = dinv[i];
        sync();
        double s = mine[2 * i * SE_BW];
        int k = i + 1;
        constexpr int U = 8;
        for (; k + U <= n; k += U) {
            double2 lv[U];
            double a[U], b[U];
#pragma unroll
            for (int j = 0; j < U; j++) {
                lv[j] = row[k + j];
                a[j] = mine[2 * (k + j) * SE_BW];
                b[j] = other[2 * (k + j) * SE_BW];
            }
#pragma unroll
            for (int j = 0; j < U; j++) s -= fma(lv[j].x, a[j], (sign * lv[j].y) * b[j]);
        }
        for (; k < n; k++) s -= fma(row[k].x, mine[2 * k * SE_BW], (sign * row[k].y) * other[2 * k * SE_BW]);
        if ((lane >> 1) < nc) mine[2 * i * SE_BW] = s * d;
    }
    sync();
    for (int e = lane; e < n * nc; e += 64) {
        const int c = e / n, i = e - c * n;
        v[i + (long)(c0 + c) * n] = x[i * SE_BW + c];
    }
}

// ---- cyclic two-sided Jacobi ---------------------------------------------------
// For the Hermitian average of h and h^H: each round applies n/2 disjoint
// rotations at once (round-robin pairing); a sweep is np - 1 rounds (np = n, or
// n + 1 with a dummy index); it stops when off(a) <= tol*|a| or after max_sweeps
// sweeps; elements below tol*|a|/n are not rotated: together they stay below the
// stopping bound (n^2 thr^2 = tol^2 |a|^2), and rotating them only stirs rounding
// noise that keeps the sweeps from ever meeting it.  Round r pairs the positions
// (slot k, slot np-1-k) of the rotating schedule: slot 0 holds index 0 and slot i
// >= 1 holds index 1 + (i - 1 - r) mod (np - 1).  A round updates the matrix by
// 2 x 2 blocks J_k^H A_kl J_l, one per two pairs: rows first, then columns, in
// one read and one write of it.
__device__ __forceinline__ void rr_pair(int k, int r, int np, int &p, int &q) {
    p = rr_slot(k, r, np);
    q = rr_slot(np - 1 - k, r, np);
    if (p > q) {
        const int t = p;
        p = q;
        q = t;
    }
}

__device__ __forceinline__ double2 hermitian_average(const double2 *h, int i, int j, int n) {
    if (i == j) return make_double2(h[i + (long)i * n].x, 0.0);
    const double2 a = i < j ? h[i + (long)j * n] : h[j + (long)i * n];
    const double2 b = i < j ? h[j + (long)i * n] : h[i + (long)j * n];
    const double2 m = make_double2(0.5 * (b.x + a.x), 0.5 * (-b.y + a.y));
    return i < j ? m : zconj(m);
}

struct Rotation {
    double c, s;
    double2 u;
};

// rotation that annihilates apq of the pair with diagonal app, aqq; identity for
// |apq| <= thr.  No branch: a wavefront has lanes of both kinds, and the values of
// an identity's chain (infinite or NaN for apq = 0) are not taken.
__device__ __forceinline__ Rotation jacobi_rotation(double app, double aqq, double2 apq, double thr) {
    // |apq| without squaring: once the element has decayed below ~1e-154,
    // apq.x^2 + apq.y^2 is denormal and keeps only a few digits, |u| drifts from
    // 1 and the phase factor would rescale row and column q
    const double g = hypot(apq.x, apq.y);
    const double zeta = (aqq - app) / (2.0 * g);
    const double t = (zeta >= 0.0 ? 1.0 : -1.0) / (fabs(zeta) + sqrt(fma(zeta, zeta, 1.0)));
    const bool on = g > thr && t != 0.0;  // a zero angle is the identity: no phase either
    const double c = 1.0 / sqrt(fma(t, t, 1.0));
    const double ux = apq.x / g, uy = -apq.y / g;  // exp(-i phi)
    return Rotation{on ? c : 1.0, on ? t * c : 0.0, make_double2(on ? ux : 1.0, on ? uy : 0.0)};
}

// (p, q) -> (c p - s t, s p + c t)
__device__ __forceinline__ void rotate2(const Rotation &r, double2 t, double2 &p, double2 &q) {
    const double2 a = p;
    p = make_double2(fma(r.c, a.x, -(r.s * t.x)), fma(r.c, a.y, -(r.s * t.y)));
    q = make_double2(fma(r.s, a.x, r.c * t.x), fma(r.s, a.y, r.c * t.y));
}
// rows: p' = c p - conj(u) s q ; q' = s p + conj(u) c q
__device__ __forceinline__ void rotate_rows(const Rotation &r, double2 &ap, double2 &aq) {
    rotate2(r, fmulc2(r.u, aq), ap, aq);
}
// columns: p' = c p - u s q ; q' = s p + u c q
__device__ __forceinline__ void rotate_cols(const Rotation &r, double2 &ap, double2 &aq) {
    rotate2(r, fmul2(r.u, aq), ap, aq);
}

// off-diagonal and total squared norm of a (LDS or global), by SE_THREADS threads
__device__ __forceinline__ void jacobi_norms(const double2 *a, int n, double *red, double &off, double &tot) {
    off = tot = 0.0;
    for (long idx = threadIdx.x; idx < (long)n * n; idx += SE_THREADS) {
        const int i = (int)(idx % n), j = (int)(idx / n);
        const double2 x = a[idx];
        const double m = fma(x.x, x.x, x.y * x.y);
        tot += m;
        if (i != j) off += m;
    }
    for (int w = 0; w < 2; w++) {
        __syncthreads();
        red[threadIdx.x] = w == 0 ? off : tot;
        __syncthreads();
        for (int s = SE_THREADS / 2; s > 0; s >>= 1) {
            if ((int)threadIdx.x < s) red[threadIdx.x] += red[threadIdx.x + s];
            __syncthreads();
        }
        (w == 0 ? off : tot) = red[0];
    }
}
__device__ __forceinline__ bool jacobi_done(double off, double tot, double tol) {
    return off <= tol * tol * tot || off == 0.0;
}
__device__ __forceinline__ double jacobi_threshold(double tot, double tol, int n) {
    return fmax(1e-300, tol * sqrt(tot) / n);
}

// n <= SE_FULL_MAX: all sweeps in one workgroup with the matrix in LDS.  On exit
// the eigenvalues ascend in eig, pos[i] is the rank of index i, and rec holds the
// rotations of each round (sweeps_out[0] * (np - 1) rounds of np/2) for
// k_jacobi_vectors.  A wavefront takes one l and its lanes the k: rows of
// consecutive lanes are consecutive.
__global__ __launch_bounds__(SE_THREADS) void k_jacobi_lds(const double2 *__restrict__ h, double4 *__restrict__ rec,
                                                           double *__restrict__ eig, int n, int max_sweeps, double tol,
                                                           int *__restrict__ pos, int *__restrict__ sweeps_out) {
    extern __shared__ __align__(16) unsigned char smem_raw[];
    double2 *a = reinterpret_cast<double2 *>(smem_raw);
    constexpr int HMAX = (SE_FULL_MAX + 1) / 2;
    __shared__ double red[SE_THREADS];
    __shared__ Rotation rot[HMAX];
    __shared__ int rp[HMAX], rq[HMAX];
    static_assert(HMAX <= 64, "one lane per pair");
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int np = (n + 1) & ~1, half = np / 2;
    for (int idx = tid; idx < n * n; idx += SE_THREADS) a[idx] = hermitian_average(h, idx % n, idx / n, n);
    int sweep = 0;
    for (; sweep < max_sweeps; sweep++) {
        double off, tot;
        jacobi_norms(a, n, red, off, tot);
        if (jacobi_done(off, tot, tol)) break;
        const double thr = jacobi_threshold(tot, tol, n);
        for (int round = 0; round < np - 1; round++) {
            if (tid < half) {
                int p, q;
                rr_pair(tid, round, np, p, q);
                Rotation r{1.0, 0.0, make_double2(1.0, 0.0)};
                if (q < n) r = jacobi_rotation(a[p + p * n].x, a[q + q * n].x, a[p + q * n], thr);
                rot[tid] = r;
                rp[tid] = p;
                rq[tid] = q;
                rec[((long)sweep * (np - 1) + round) * half + tid] = make_double4(r.c, r.s, r.u.x, r.u.y);
            }
            __syncthreads();
            if (lane < half) {
                const Rotation rk = rot[lane];
                const int pk = rp[lane], qk = rq[lane];
                for (int l = wave; l < half; l += SE_THREADS / 64) {
                    const Rotation rl = rot[l];
                    if (rk.s == 0.0 && rl.s == 0.0) continue;  // two identities
                    const int pl = rp[l] * n, ql = rq[l] * n;
                    const bool kq = qk < n, lq = rq[l] < n;  // the dummy index has no row
                    const double2 z = make_double2(0.0, 0.0);
                    double2 a00 = a[pk + pl], a01 = lq ? a[pk + ql] : z, a10 = kq ? a[qk + pl] : z,
                            a11 = kq && lq ? a[qk + ql] : z;
                    if (rk.s != 0.0) {
                        rotate_rows(rk, a00, a10);
                        rotate_rows(rk, a01, a11);
                    }
                    if (rl.s != 0.0) {
                        rotate_cols(rl, a00, a01);
                        rotate_cols(rl, a10, a11);
                    }
                    a[pk + pl] = a00;
                    if (lq) a[pk + ql] = a01;
                    if (kq) a[qk + pl] = a10;
                    if (kq && lq) a[qk + ql] = a11;
                }
            }
            __syncthreads();
        }
    }
    __syncthreads();
    for (int i = tid; i < n; i += SE_THREADS) {
        const double e = a[i + i * n].x;
        int r = 0;
        for (int j = 0; j < n; j++) {
            const double f = a[j + j * n].x;
            r += (f < e) || (f == e && j < i);
        }
        pos[i] = r;
        eig[r] = e;
    }
    if (tid == 0) *sweeps_out = sweep;
}

// Jacobi of the iterative diagonalisation's subspace matrix, n <= SE_DIAG_MAX: all
// sweeps in one workgroup on the packed lower triangle in LDS (h: lower triangle,
// column-major).  Each step of that iteration starts from Ritz vectors, so the
// matrix comes nearly diagonal and few sweeps do.  A round is one chain of
// latencies, so it is kept short: the rotation from three reciprocal square
// roots (k_jacobi_lds, whose results the caller of a Rayleigh-Ritz step keeps to
// the bit, takes a hypot, four divisions and two square roots), and with half of
// the blocks gone by symmetry one to three blocks per thread.  Outputs as
// k_jacobi_lds; info: 1 if max_sweeps did not do.  us at n = 72, from Ritz vectors: 292 on
// average (from 172), with the vectors 359, with the refinement below 403, zheevd 1,600.
__device__ __forceinline__ double fast_rsqrt(double x) {
    double r = __builtin_amdgcn_rsq(x);  // refined by two Newton steps
#pragma unroll
    for (int i = 0; i < 2; i++) r = fma(0.5 * r, fma(-x * r, r, 1.0), r);
    return r;
}

__global__ __launch_bounds__(SE_THREADS) void k_jacobi_tri(const double2 *__restrict__ h, double4 *__restrict__ rec,
                                                           double *__restrict__ eig, int n, int max_sweeps, double tol,
                                                           int *__restrict__ pos, int *__restrict__ sweeps_out,
                                                           int *__restrict__ info) {
    extern __shared__ __align__(16) unsigned char smem_raw[];
    double2 *P = reinterpret_cast<double2 *>(smem_raw);
    constexpr int HMAX = SE_DIAG_MAX / 2;
    __shared__ double red[2][SE_THREADS / 64];
    __shared__ Rotation rot[HMAX];
    __shared__ int rp[HMAX], rq[HMAX];
    static_assert(HMAX <= 64, "one lane per pair");
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int np = (n + 1) & ~1, half = np / 2, nblk = half * (half + 1) / 2;
    const auto get = [&](int i, int j) {
        const double2 v = P[i >= j ? tri(i) + j : tri(j) + i];
        return i >= j ? v : zconj(v);
    };
    const auto put = [&](int i, int j, double2 v) { P[i >= j ? tri(i) + j : tri(j) + i] = i >= j ? v : zconj(v); };
    for (int c = wave; c < n; c += SE_THREADS / 64)
        for (int r = c + lane; r < n; r += 64) {
            const double2 v = h[r + (long)c * n];
            P[tri(r) + c] = r == c ? make_double2(v.x, 0.0) : v;
        }
    // blocks (k, l), k >= l, of this thread: fixed over the rounds
    constexpr int MAXB = (HMAX * (HMAX + 1) / 2 + SE_THREADS - 1) / SE_THREADS;
    int bk[MAXB], bl[MAXB];
#pragma unroll
    for (int u = 0; u < MAXB; u++) {
        const int t = tid + u * SE_THREADS;
        int k = (int)((sqrtf(8.f * t + 1.f) - 1.f) * 0.5f);
        if (tri(k) > t) k--;
        if (tri(k + 1) <= t) k++;
        bk[u] = k;
        bl[u] = t - tri(k);
    }
    int sweep = 0;
    for (; sweep < max_sweeps; sweep++) {
        __syncthreads();
        double off = 0.0, tot = 0.0;
        for (int r = wave; r < n; r += SE_THREADS / 64)
            for (int c = lane; c <= r; c += 64) {
                const double2 x = P[tri(r) + c];
                const double m = fma(x.x, x.x, x.y * x.y);
                if (c < r) off += 2.0 * m;
                tot += c < r ? 2.0 * m : m;
            }
        for (int s = 1; s < 64; s <<= 1) {
            off += __shfl_xor(off, s);
            tot += __shfl_xor(tot, s);
        }
        if (lane == 0) {
            red[0][wave] = off;
            red[1][wave] = tot;
        }
        __syncthreads();
        off = tot = 0.0;
        for (int w = 0; w < SE_THREADS / 64; w++) {
            off += red[0][w];
            tot += red[1][w];
        }
        if (jacobi_done(off, tot, tol)) break;
        const double thr = jacobi_threshold(tot, tol, n), thr2 = fmax(thr * thr, 1e-280);  // squares stay normal
        for (int round = 0; round < np - 1; round++) {
            if (tid < half) {
                int p, q;
                rr_pair(tid, round, np, p, q);
                Rotation r{1.0, 0.0, make_double2(1.0, 0.0)};
                if (q < n) {
                    const double app = P[tri(p) + p].x, aqq = P[tri(q) + q].x;
                    const double2 apq = zconj(P[tri(q) + p]);  // q > p
                    const double g2 = fma(apq.x, apq.x, apq.y * apq.y);
                    if (g2 > thr2) {
                        const double d = aqq - app;
                        const double rg = fast_rsqrt(g2), rh = fast_rsqrt(fma(d, d, 4.0 * g2));
                        const double c2 = fma(0.5 * fabs(d), rh, 0.5), rc = fast_rsqrt(c2);
                        r.u = make_double2(apq.x * rg, -apq.y * rg);
                        r.c = c2 * rc;
                        r.s = (d >= 0.0 ? g2 : -g2) * rg * rh * rc;
                    }
                }
                rot[tid] = r;
                rp[tid] = p;
                rq[tid] = q;
                rec[((long)sweep * (np - 1) + round) * half + tid] = make_double4(r.c, r.s, r.u.x, r.u.y);
            }
            __syncthreads();
#pragma unroll
            for (int u = 0; u < MAXB; u++) {
                if (tid + u * SE_THREADS >= nblk) break;
                const int k = bk[u], l = bl[u];
                const Rotation rk = rot[k], rl = rot[l];
                if (rk.s == 0.0 && rl.s == 0.0) continue;  // two identities
                const int pk = rp[k], qk = rq[k], pl = rp[l], ql = rq[l];
                const bool kq = qk < n, lq = ql < n;  // the dummy index has no row
                const double2 z = make_double2(0.0, 0.0);
                double2 a00 = get(pk, pl), a01 = lq ? get(pk, ql) : z, a10 = kq ? get(qk, pl) : z,
                        a11 = kq && lq ? get(qk, ql) : z;
                rotate_rows(rk, a00, a10);
                rotate_rows(rk, a01, a11);
                rotate_cols(rl, a00, a01);
                rotate_cols(rl, a10, a11);
                if (k == l) {  // the annihilated pair: real diagonal, one off-diagonal element
                    put(pk, pk, make_double2(a00.x, 0.0));
                    if (kq) {
                        put(qk, qk, make_double2(a11.x, 0.0));
                        put(qk, pk, z);
                    }
                } else {
                    put(pk, pl, a00);
                    if (lq) put(pk, ql, a01);
                    if (kq) put(qk, pl, a10);
                    if (kq && lq) put(qk, ql, a11);
                }
            }
            __syncthreads();
        }
    }
    for (int i = tid; i < n; i += SE_THREADS) {
        const double e = P[tri(i) + i].x;
        int r = 0;
        for (int j = 0; j < n; j++) {
            const double f = P[tri(j) + j].x;
            r += (f < e) || (f == e && j < i);
        }
        pos[i] = r;
        eig[r] = e;
    }
    if (tid == 0) {
        *sweeps_out = sweep;
        *info = sweep == max_sweeps;
    }
}

// Eigenvectors of k_jacobi_lds and k_jacobi_tri: v = J_1 J_2 ... with columns in the order of
// pos.  A row of v depends on no other: SE_VROWS rows per wavefront, in LDS, all
// rotations of a round at once, no block barrier; the next round's rotations are
// loaded while this one's are applied.
constexpr int SE_VROWS = 2;
__global__ __launch_bounds__(64) void k_jacobi_vectors(const double4 *__restrict__ rec, const int *__restrict__ sweeps,
                                                       const int *__restrict__ pos, double2 *__restrict__ v, int n) {
    __shared__ double2 row[SE_VROWS][SE_DIAG_MAX + 1];  // + the dummy index of an odd n
    const int lane = threadIdx.x, i0 = blockIdx.x * SE_VROWS;
    const int np = (n + 1) & ~1, half = np / 2;
    for (int j = lane; j < np; j += 64)
        for (int w = 0; w < SE_VROWS; w++) row[w][j] = make_double2(i0 + w == j ? 1.0 : 0.0, 0.0);
    const long rounds = (long)*sweeps * (np - 1);
    const int k = min(lane, half - 1);
    double4 nx = rounds > 0 ? rec[k] : make_double4(1.0, 0.0, 1.0, 0.0);
    int rr = 0;
    for (long r = 0; r < rounds; r++) {
        const double4 cur = nx;
        if (r + 1 < rounds) nx = rec[(r + 1) * half + k];
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
        if (lane < half && cur.y != 0.0) {
            int p, q;
            rr_pair(k, rr, np, p, q);
            const Rotation rt{cur.x, cur.y, make_double2(cur.z, cur.w)};
#pragma unroll
            for (int w = 0; w < SE_VROWS; w++) rotate_cols(rt, row[w][p], row[w][q]);
        }
        if (++rr == np - 1) rr = 0;
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    for (int j = lane; j < n; j += 64)
        for (int w = 0; w < SE_VROWS; w++)
            if (i0 + w < n) v[i0 + w + (long)pos[j] * n] = row[w][j];
}

// ---- refinement of the eigenpairs of k_jacobi_tri ----------------------------------
// A column of v has gone through a rotation per round, each unitary only to its
// rounding: at 72 columns v is orthonormal to 2e-14 and A v = v w holds to
// 3e-15 |A|, where zheevd leaves 2e-15 and 2e-16.  So the pairs are refined against
// the matrix itself (one step of the iteration of T. Ogita and K. Aishima,
// Jpn. J. Ind. Appl. Math. 35, 1007 (2018), in the form that keeps the rotation part
// exactly anti-Hermitian): with R = 1 - v^H v and S = v^H A v,
//   v <- v + v (R/2 + K),  K_ij = (S_ij + (w_i + w_j)/2 R_ij) / (w_j - w_i),
//   w_i <- S_ii (1 + R_ii).
// Pairs so close that |K_ij| would exceed SE_REF_MAX stay as the sweeps left them.
// Two steps (the second takes away the K^2 of the first) at 17 to 127 columns: v
// orthonormal to 1e-15, A v = v w to 4e-16 |A|, close pairs included.
// Three products of n <= 128 per step, one 16 x 16 tile per block: bound by
// their launches (7.8 + 7.3 + 6.9 us at 72).  Block iteration on the 64-atom cell, 42 vectors, 76 steps: vectors
// orthonormal to 2.6e-15 (without the refinement 4e-13, with zheevd 4e-14), 222 ms (217,
// 269).
constexpr int SE_RT = 16;
constexpr double SE_REF_MAX = 1e-5;

// s += conj(a) b or a b
__device__ __forceinline__ void zmac(double2 &s, double2 a, double2 b) {
    s.x = fma(a.x, b.x, fma(-a.y, b.y, s.x));
    s.y = fma(a.x, b.y, fma(a.y, b.x, s.y));
}
__device__ __forceinline__ void zmacc(double2 &s, double2 a, double2 b) {
    s.x = fma(a.x, b.x, fma(a.y, b.y, s.x));
    s.y = fma(a.x, b.y, fma(-a.y, b.x, s.y));
}

// out = a b (HERM: a Hermitian, its lower triangle given) or b0 + a b (b0 = a);
// grid ceil(n/16) x ceil(n/16).
template <bool HERM>
__global__ __launch_bounds__(SE_RT *SE_RT) void k_refine_product(const double2 *__restrict__ a,
                                                                 const double2 *__restrict__ b,
                                                                 double2 *__restrict__ out, int n) {
    __shared__ double2 sa[SE_RT][SE_RT + 1], sb[SE_RT][SE_RT + 1];
    const int tx = threadIdx.x % SE_RT, ty = threadIdx.x / SE_RT;
    const int i = blockIdx.x * SE_RT + tx, j = blockIdx.y * SE_RT + ty;
    const double2 zero = make_double2(0.0, 0.0);
    double2 s = !HERM && i < n && j < n ? a[i + (long)j * n] : zero;
    for (int k0 = 0; k0 < n; k0 += SE_RT) {
        const int ka = k0 + ty, kb = k0 + tx;  // a's column, b's row
        double2 x = zero;
        if (i < n && ka < n) {
            if (!HERM || i > ka) x = a[i + (long)ka * n];
            else if (i == ka) x = make_double2(a[i + (long)i * n].x, 0.0);
            else x = zconj(a[ka + (long)i * n]);
        }
        sa[ty][tx] = x;
        sb[ty][tx] = kb < n && j < n ? b[kb + (long)j * n] : zero;
        __syncthreads();
#pragma unroll
        for (int k = 0; k < SE_RT; k++) zmac(s, sa[k][tx], sb[ty][k]);
        __syncthreads();
    }
    if (i < n && j < n) out[i + (long)j * n] = s;
}

// e = R/2 + K and wout of the step above, from v and t = A v.  The tiles on and
// below the diagonal: an element and its mirror come from one thread, so that K is
// exactly anti-Hermitian.
__global__ __launch_bounds__(SE_RT *SE_RT) void k_refine_step(const double2 *__restrict__ v,
                                                              const double2 *__restrict__ t,
                                                              const double *__restrict__ w, double2 *__restrict__ e,
                                                              double *__restrict__ wout, int n) {
    __shared__ double2 si[SE_RT][SE_RT + 1], sj[SE_RT][SE_RT + 1], st[SE_RT][SE_RT + 1];
    if (blockIdx.x < blockIdx.y) return;  // the whole block
    const int tx = threadIdx.x % SE_RT, ty = threadIdx.x / SE_RT;
    const int i0 = blockIdx.x * SE_RT, j0 = blockIdx.y * SE_RT, i = i0 + tx, j = j0 + ty;
    const double2 zero = make_double2(0.0, 0.0);
    double2 s = zero, p = make_double2(i == j ? -1.0 : 0.0, 0.0);  // p = v^H v - 1
    for (int k0 = 0; k0 < n; k0 += SE_RT) {
        const int k = k0 + tx;
        si[ty][tx] = k < n && i0 + ty < n ? v[k + (long)(i0 + ty) * n] : zero;
        sj[ty][tx] = k < n && j < n ? v[k + (long)j * n] : zero;
        st[ty][tx] = k < n && j < n ? t[k + (long)j * n] : zero;
        __syncthreads();
#pragma unroll
        for (int q = 0; q < SE_RT; q++) {
            zmacc(s, si[tx][q], st[ty][q]);
            zmacc(p, si[tx][q], sj[ty][q]);
        }
        __syncthreads();
    }
    if (i >= n || j >= n || i < j) return;
    if (i == j) {
        e[i + (long)i * n] = make_double2(-0.5 * p.x, 0.0);
        wout[i] = s.x - s.x * p.x;
        return;
    }
    const double wi = w[i], wj = w[j], d = wj - wi, m = -0.5 * (wi + wj);
    const double2 num = make_double2(fma(m, p.x, s.x), fma(m, p.y, s.y));
    const bool far = fabs(num.x) + fabs(num.y) <= SE_REF_MAX * fabs(d) && d != 0.0;
    const double2 k = far ? make_double2(num.x / d, num.y / d) : zero;
    const double2 r = make_double2(-0.5 * p.x, -0.5 * p.y);
    e[i + (long)j * n] = make_double2(r.x + k.x, r.y + k.y);
    e[j + (long)i * n] = make_double2(r.x - k.x, k.y - r.y);
}

// ---- larger n: one launch per round ----------------------------------------------
struct JacobiCtl {
    double thr;
    int stop;    // converged: the rounds that follow do nothing
    int sweeps;  // sweeps begun
};

// a = average of h and h^H, v = 1
__global__ __launch_bounds__(256) void k_jacobi_init(const double2 *__restrict__ h, double2 *__restrict__ a,
                                                     double2 *__restrict__ v, int n, JacobiCtl *ctl) {
    const long idx = (long)blockIdx.x * 256 + threadIdx.x;
    if (idx == 0) *ctl = JacobiCtl{0.0, 0, 0};
    if (idx >= (long)n * n) return;
    const int i = (int)(idx % n), j = (int)(idx / n);
    a[idx] = hermitian_average(h, i, j, n);
    v[idx] = make_double2(i == j ? 1.0 : 0.0, 0.0);
}

// start of a sweep: threshold, or stop
__global__ __launch_bounds__(SE_THREADS) void k_jacobi_check(const double2 *__restrict__ a, int n, double tol,
                                                             JacobiCtl *ctl, int *host_stop) {
    __shared__ double red[SE_THREADS];
    double off, tot;
    jacobi_norms(a, n, red, off, tot);
    if (threadIdx.x == 0) {
        const bool done = jacobi_done(off, tot, tol);
        ctl->thr = jacobi_threshold(tot, tol, n);
        ctl->stop = done;
        ctl->sweeps += !done;
        *host_stop = done;
    }
}

// One round: blocks y < nl4 update the matrix (a to b: other blocks read a's
// elements for their rotations), a wavefront per l and its lanes the k; the
// others rotate the columns of v in place, a wavefront per pair and its lanes the
// rows.  Rotations are recomputed where they are used: a round is one trip to
// memory and one chain of square roots and divisions, with no barrier.  So all
// loads go out together, and a wavefront that holds pair l among its own k takes
// that rotation from its lane (n <= 128: always).  us per round at n = 128: 4.4 with
// the threshold awaited first and both rotations computed, 3.7 so.
__global__ __launch_bounds__(256) void k_jacobi_round(const double2 *__restrict__ a, double2 *__restrict__ b,
                                                      double2 *__restrict__ v, int n, int round,
                                                      const JacobiCtl *__restrict__ ctl) {
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int np = (n + 1) & ~1, half = np / 2, nl4 = (half + 3) / 4;
    const double thr = ctl->thr;
    const int stop = ctl->stop;
    // rotation of the pair (p, q); elements of a pair with the dummy index n are not used
    const auto pair_rotation = [&](int p, int q, double app, double aqq, double2 apq) {
        const Rotation r = jacobi_rotation(app, aqq, apq, thr);
        return q < n ? r : Rotation{1.0, 0.0, make_double2(1.0, 0.0)};
    };
    const auto at = [&](int i, int j) { return a[min(i, n - 1) + (long)min(j, n - 1) * n]; };
    if ((int)blockIdx.y < nl4) {
        const int k0 = blockIdx.x * 64, k = min(k0 + lane, half - 1), l = blockIdx.y * 4 + wave;
        if (l >= half) return;
        int pk, qk, pl, ql;
        rr_pair(k, round, np, pk, qk);
        rr_pair(l, round, np, pl, ql);
        const bool kq = qk < n, lq = ql < n;  // the dummy index has no row
        const double2 z = make_double2(0.0, 0.0);
        double2 a00 = at(pk, pl), a01 = at(pk, ql), a10 = at(qk, pl), a11 = at(qk, ql);
        const double kpp = at(pk, pk).x, kqq = at(qk, qk).x;
        const double2 kpq = at(pk, qk);
        Rotation rl;
        const bool held = l >= k0 && l < k0 + 64;  // the same for the wavefront
        if (!held) rl = pair_rotation(pl, ql, at(pl, pl).x, at(ql, ql).x, at(pl, ql));
        if (stop) return;
        const Rotation rk = pair_rotation(pk, qk, kpp, kqq, kpq);
        if (held)
            rl = Rotation{lane_value(rk.c, l - k0), lane_value(rk.s, l - k0),
                          make_double2(lane_value(rk.u.x, l - k0), lane_value(rk.u.y, l - k0))};
        if (!lq) a01 = z;
        if (!kq) a10 = z;
        if (!(kq && lq)) a11 = z;
        if (rk.s != 0.0) {
            rotate_rows(rk, a00, a10);
            rotate_rows(rk, a01, a11);
        }
        if (rl.s != 0.0) {
            rotate_cols(rl, a00, a01);
            rotate_cols(rl, a10, a11);
        }
        if (k0 + lane >= half) return;
        const long cp = (long)pl * n, cq = (long)ql * n;
        b[pk + cp] = a00;
        if (lq) b[pk + cq] = a01;
        if (kq) b[qk + cp] = a10;
        if (kq && lq) b[qk + cq] = a11;
    } else {
        const int k = (blockIdx.y - nl4) * 4 + wave;
        if (k >= half) return;
        int p, q;
        rr_pair(k, round, np, p, q);
        if (q >= n) return;
        const int i0 = blockIdx.x * 64 + lane, ic = min(i0, n - 1);
        double2 vp = v[ic + (long)p * n], vq = v[ic + (long)q * n];
        const Rotation r = pair_rotation(p, q, at(p, p).x, at(q, q).x, at(p, q));
        if (stop || r.s == 0.0) return;
        // the first rows were loaded with the rotation's elements
        rotate_cols(r, vp, vq);
        if (i0 < n) {
            v[i0 + (long)p * n] = vp;
            v[i0 + (long)q * n] = vq;
        }
        for (int i = i0 + gridDim.x * 64; i < n; i += gridDim.x * 64)
            rotate_cols(r, v[i + (long)p * n], v[i + (long)q * n]);
    }
}

// eigenvalues in ascending order (rank by value, ties by index)
__global__ __launch_bounds__(256) void k_jacobi_order(const double2 *__restrict__ a, double *__restrict__ eig, int n,
                                                      int *__restrict__ pos) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    const double e = a[i + (long)i * n].x;
    int r = 0;
    for (int j = 0; j < n; j++) {
        const double f = a[j + (long)j * n].x;
        r += (f < e) || (f == e && j < i);
    }
    pos[i] = r;
    eig[r] = e;
}
// out(:, pos[j]) = v(:, j)
__global__ __launch_bounds__(256) void k_jacobi_permute(const double2 *__restrict__ v, const int *__restrict__ pos,
                                                        double2 *__restrict__ out, int n) {
    const long idx = (long)blockIdx.x * 256 + threadIdx.x;
    if (idx >= (long)n * n) return;
    const int i = (int)(idx % n), j = (int)(idx / n);
    out[i + (long)pos[j] * n] = v[idx];
}

}  // namespace cpwgpu
