// Host state shared by the translation units of libcpwgpu: the error text, the
// library stream, device buffers, the measurement hook and the plan of one
// k-point.
#pragma once

#include <hip/hip_runtime.h>
#include <hip/hip_ext.h>

#include <algorithm>
#include <cstdarg>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <mutex>
#include <string>
#include <vector>

#include "../../include/cpwgpu.h"
#include "fft_local.hpp"

namespace cpwgpu {

inline thread_local std::string g_err;
inline std::mutex g_mu;
inline int g_device = 0;
inline int g_prec = CPWGPU_PREC_FP64;
inline int g_ditsp_method = CPWGPU_DITSP_CHEB;
inline int g_overlap = 1;
inline hipStream_t g_stream = nullptr;

inline int fail(int code, const char *fmt, ...) __attribute__((format(printf, 2, 3)));
inline int fail(int code, const char *fmt, ...) {
    char buf[512];
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(buf, sizeof buf, fmt, ap);
    va_end(ap);
    g_err = buf;
    return code;
}

#define HIPCHK(x)                                                                          \
    do {                                                                                   \
        hipError_t e_ = (x);                                                               \
        if (e_ != hipSuccess)                                                              \
            return fail(e_ == hipErrorOutOfMemory ? CPWGPU_ERR_NOMEM : CPWGPU_ERR_HIP,     \
                        "%s: %s (%s:%d)", #x, hipGetErrorString(e_), __FILE__, __LINE__);  \
    } while (0)

inline int ensure_stream() {
    if (!g_stream) {
        HIPCHK(hipSetDevice(g_device));
        HIPCHK(hipStreamCreateWithFlags(&g_stream, hipStreamNonBlocking));
    }
    return CPWGPU_OK;
}

// grow-only device buffer
struct DevBuf {
    void *p = nullptr;
    size_t n = 0;
    int reserve(size_t bytes) {
        if (bytes <= n) return CPWGPU_OK;
        if (p) hipFree(p);
        p = nullptr;
        n = 0;
        HIPCHK(hipMalloc(&p, std::max<size_t>(bytes, 256)));
        n = bytes;
        return CPWGPU_OK;
    }
    void release() {
        if (p) hipFree(p);
        p = nullptr;
        n = 0;
    }
};

// ---- per-kernel event timing (measurement hook) ----------------------------
struct Prof {
    bool on = false;
    unsigned mask = 0;
    struct Rec { int k; hipEvent_t a, b; };
    std::vector<Rec> recs;
    std::vector<hipEvent_t> pool;
    hipEvent_t get() {
        if (!pool.empty()) { hipEvent_t e = pool.back(); pool.pop_back(); return e; }
        // timing only (read after the whole stream has finished): no
        // system-scope fence, so recording them does not write back and
        // invalidate the caches in the middle of the work they time
        hipEvent_t e = nullptr;
        if (hipEventCreateWithFlags(&e, hipEventDisableSystemFence) != hipSuccess) return nullptr;
        return e;
    }
};
inline Prof g_prof;

// Launches kernel f on stream s.  With the measurement hook on for kernel id
// k, the start and stop events travel with the dispatch itself (the kernel's
// own timestamps, hipExtLaunchKernelGGL) instead of as marker packets
// recorded around it, which would idle the stream between the kernels.
template <typename... Args, typename F = void (*)(Args...)>
void launch_timed(int k, F f, dim3 grid, dim3 block, size_t shmem, hipStream_t s, Args... args) {
    if (g_rec) {  // a kernel that cannot be batched
        g_rec->ok = false;
        return;
    }
    if (g_prof.on && (g_prof.mask >> k & 1u)) {
        hipEvent_t a = g_prof.get(), b = a ? g_prof.get() : nullptr;
        if (a && b) {
            hipExtLaunchKernelGGL(f, grid, block, (std::uint32_t)shmem, s, a, b, 0u, args...);
            g_prof.recs.push_back({k, a, b});
            return;
        }
        if (a) g_prof.pool.push_back(a);
    }
    hipLaunchKernelGGL(f, grid, block, shmem, s, args...);
}

// The same for kernel f whose body is K::run: recorded for a batch when a
// recorder is set.
template <class K, typename... Args, typename F = void (*)(Args...)>
void launch_batchable(int k, F f, dim3 grid, dim3 block, size_t shmem, hipStream_t s, Args... args) {
    if (g_rec) {
        const auto p = make_pack(args...);
        static_assert(std::is_trivially_copyable<decltype(p)>::value, "arguments are copied to the device");
        const char *b = reinterpret_cast<const char *>(&p);
        g_rec->steps.push_back({(const void *)k_batch<K, Args...>, grid, block.x, shmem, {b, b + sizeof p}});
        return;
    }
    launch_timed(k, f, grid, block, shmem, s, args...);
}

}  // namespace cpwgpu

using namespace cpwgpu;

struct cpwgpu_plan_s {
    FftGeom g{};
    int mtxd = 0, ng = 0, nanl = 0;
    int kdmax[3] = {0, 0, 0};
    double inv_n = 1.0;
    size_t ntot = 0;          // id*n2*n3
    int mwrk = 0;
    // host copies used to recognise an unchanged k-point in the drop-in
    std::vector<long> key_pts;
    std::vector<double> h_ekpg;
    // device arrays
    DevBuf col_ptr, col_uy, ent_i, ent_cz, ekpg, tw[3];
    DevBuf zmap;              // [col][z] -> psi row or -1 (register column kernels)
    DevBuf v64, v32;          // V(r) in FP64 and FP32
    double v0 = 0.0;          // mean of V(r) over the mesh = V(G=0), the local part of diag(H)
    DevBuf anl64, anl32, xnl; // projectors
    long lda = 0;             // leading dimension of anl64
    long lda32 = 0;           // of anl32: lda rounded up to even (16-byte aligned rows)
    bool anl32_valid = false;
    // plane-stage kernel per precision (index 0 FP64, 1 FP32): -1 = default for
    // the mesh, else a variant number (set by the tuner or by the caller)
    int plane_var[2] = {-1, -1};
    // column kernels: 0 LDS lines, 1 register lines; -1 default
    int col_var[2] = {-1, -1};
    // stream schedule: 0 (default) one stream; 1 the projection beside the
    // local term; 2 the inverse columns and planes beside the non-local term
    int sched_var[2] = {-1, -1};
    // split-K target blocks of the projection GEMM per precision (-1 and
    // SPLITK_DEFAULT: whole rounds of the compute units)
    int splitk[2] = {-1, -1};
    // projection and back-projection GEMM kernel per precision (-1 and
    // PROJ_DEFAULT, BACK_DEFAULT: by size)
    int proj_var[2] = {-1, -1};
    int back_var[2] = {-1, -1};
    // where the kinetic term ekpg*psi is added when the non-local term is on:
    // 0 the back-projection epilogue, 1 the gather of the forward column kernel
    // (-1 = default, 0)
    int kin_var[2] = {-1, -1};
    // plane kernel of the coupled two-component case (nsp = 4): 0 LDS
    // two-pass, 1 register lines (-1 = default)
    int spin_var[2] = {-1, -1};
    // workspaces
    DevBuf colbuf, part, dhd;
    DevBuf gw;                // g_j of each plane wave as doubles [3][mtxd] (force projections)
    // spinor path (hk_psi_spin_c16): potential components in the layout of
    // k_spin_potential, projectors on the 2*mtxd interleaved rows, split bands
    int nsp = 0;
    DevBuf vsp64, vsp32;
    DevBuf sanl64, sanl32, sxnl;
    long slda = 0, slda32 = 0;
    int snanl = 0;
    bool sanl32_valid = false;
    DevBuf spsi, shpsi;
    ~cpwgpu_plan_s() {
        col_ptr.release(); col_uy.release(); ent_i.release(); ent_cz.release(); ekpg.release(); zmap.release();
        for (auto &t : tw) t.release();
        v64.release(); v32.release(); anl64.release(); anl32.release(); xnl.release();
        colbuf.release(); part.release(); dhd.release(); gw.release();
        vsp64.release(); vsp32.release(); sanl64.release(); sanl32.release(); sxnl.release();
        spsi.release(); shpsi.release();
    }
};
