// Copies of large host matrices to and from the device.  The host arrays of the
// drop-in calls are ordinary (pageable) memory: the runtime moves those through
// its own staging at 30 GB/s in and 18 GB/s out on one thread, where pinned memory
// runs at 57.  Here a few threads each copy pieces of the matrix through pinned
// pieces of their own, in chunks that alternate between two of them, so the DMA of
// one chunk runs beside the host copy of the next.
// 128 bands and 256 projectors of the 64-atom cell (147 MB in, 49 MB out), the whole
// call: 10,600 us through the runtime, 5,950 so (4,300 of it the DMA and the kernels).
// With other threads on every CPU (a BLAS's workers spin for 0.1 s after a call) the
// copies wait for them: 10-12 ms.
#pragma once

#include "host.hpp"

#include <atomic>
#include <exception>
#include <thread>

namespace cpwgpu {

constexpr int HC_LANES = 8;                    // threads, the caller's own among them
constexpr size_t HC_CHUNK = 2ull << 20;        // bytes per pinned piece; two per lane
constexpr size_t HC_MIN = 4ull << 20;          // smaller copies go to the runtime

// The library's device is the current one while this lives; the caller's is again
// afterwards.
struct OnDevice {
    int before = 0;
    hipError_t err;
    OnDevice() {
        err = hipGetDevice(&before);
        if (err == hipSuccess && before != g_device) err = hipSetDevice(g_device);
    }
    ~OnDevice() {
        if (before != g_device) (void)hipSetDevice(before);
    }
};

// Pinned pieces, kept from the first large copy to cpwgpu_finalize or a copy for
// another device (32 MB).  Used under the library's lock, by one copy at a time.
struct HostCopy {
    struct Lane {
        char *pin[2] = {nullptr, nullptr};
        hipEvent_t ev[2] = {nullptr, nullptr};  // end of the last DMA from or to the piece
        bool used[2] = {false, false};
    } lane[HC_LANES];
    int lanes = 0;      // those that have their pieces
    int device = 0;     // of the events

    // the lanes that are missing: also those that could not be had at an earlier copy
    void init() {
        if (device != g_device) release();
        device = g_device;
        const int want = std::max(1, std::min<int>(HC_LANES, (int)std::thread::hardware_concurrency()));
        for (; lanes < want; lanes++)
            for (int i = 0; i < 2; i++) {
                Lane &l = lane[lanes];
                if (!l.pin[i] && hipHostMalloc((void **)&l.pin[i], HC_CHUNK, hipHostMallocDefault) != hipSuccess)
                    l.pin[i] = nullptr;
                if (!l.ev[i] && hipEventCreateWithFlags(&l.ev[i], hipEventDisableTiming) != hipSuccess) l.ev[i] = nullptr;
                if (!l.pin[i] || !l.ev[i]) {
                    (void)hipGetLastError();
                    return;
                }
            }
    }
    void release() {
        for (Lane &l : lane)
            for (int i = 0; i < 2; i++) {
                if (l.used[i]) (void)hipEventSynchronize(l.ev[i]);
                if (l.ev[i]) (void)hipEventDestroy(l.ev[i]);
                if (l.pin[i]) (void)hipHostFree(l.pin[i]);
                l = i ? Lane{} : l;
            }
        lanes = 0;
    }
};
inline HostCopy g_hc;

// Bytes [off, off + len) of the packed matrix (columns of width bytes) between
// buf and the columns of the strided one at a (ld bytes apart).
template <bool GATHER> inline void copy_piece(char *buf, char *a, size_t ld, size_t width, size_t off, size_t len) {
    for (size_t done = 0; done < len;) {
        const size_t c = (off + done) / width, r = off + done - c * width, n = std::min(width - r, len - done);
        if (GATHER) memcpy(buf + done, a + c * ld + r, n);
        else memcpy(a + c * ld + r, buf + done, n);
        done += n;
    }
}

// cols columns of width bytes between host (ldh bytes apart) and dev (ldd bytes
// apart) in the order of stream s.  IN: returns once host has been read; out:
// once it has been written.
template <bool IN>
int host_copy_2d(void *dev, size_t ldd, void *host, size_t ldh, size_t width, size_t cols, hipStream_t s) {
    const size_t total = width * cols;
    OnDevice on;
    if (on.err != hipSuccess) return fail(CPWGPU_ERR_HIP, "device %d: %s", g_device, hipGetErrorString(on.err));
    if (total >= HC_MIN) g_hc.init();
    if (total < HC_MIN || g_hc.lanes == 0) {
        if (IN) HIPCHK(hipMemcpy2DAsync(dev, ldd, host, ldh, width, cols, hipMemcpyHostToDevice, s));
        else {
            HIPCHK(hipMemcpy2DAsync(host, ldh, dev, ldd, width, cols, hipMemcpyDeviceToHost, s));
            HIPCHK(hipStreamSynchronize(s));
        }
        return CPWGPU_OK;
    }
    const size_t nchunk = (total + HC_CHUNK - 1) / HC_CHUNK;
    std::atomic<size_t> next{0};
    std::atomic<int> err{(int)hipSuccess};
    const auto dma = [&](char *pin, size_t off, size_t len) -> hipError_t {
        // device columns that follow each other are one piece
        for (size_t done = 0; done < len;) {
            const size_t c = (off + done) / width, r = off + done - c * width;
            const size_t n = ldd == width ? len : std::min(width - r, len - done);
            char *d = (char *)dev + c * ldd + r;
            const hipError_t e = IN ? hipMemcpyAsync(d, pin + done, n, hipMemcpyHostToDevice, s)
                                    : hipMemcpyAsync(pin + done, d, n, hipMemcpyDeviceToHost, s);
            if (e != hipSuccess) return e;
            done += n;
        }
        return hipSuccess;
    };
    const auto work = [&](int id) {
        HostCopy::Lane &l = g_hc.lane[id];
        hipError_t e = hipSetDevice(g_device);
        size_t last = nchunk, last_len = 0;  // out: the chunk whose DMA is on its way
        int slot = 0;
        const auto drain = [&](int i) {  // out: the chunk in piece i to the host array
            if (last == nchunk) return;
            if (e == hipSuccess) e = hipEventSynchronize(l.ev[i]);
            if (e == hipSuccess) copy_piece<false>(l.pin[i], (char *)host, ldh, width, last * HC_CHUNK, last_len);
            last = nchunk;
        };
        while (e == hipSuccess && err.load() == (int)hipSuccess) {
            const size_t c = next.fetch_add(1);
            if (c >= nchunk) break;
            const size_t off = c * HC_CHUNK, len = std::min(HC_CHUNK, total - off);
            if (l.used[slot]) e = hipEventSynchronize(l.ev[slot]);
            if (IN && e == hipSuccess) copy_piece<true>(l.pin[slot], (char *)host, ldh, width, off, len);
            if (e == hipSuccess) e = dma(l.pin[slot], off, len);
            if (e == hipSuccess) e = hipEventRecord(l.ev[slot], s);
            l.used[slot] = e == hipSuccess;
            if (!IN) {
                drain(1 - slot);
                last = c;
                last_len = len;
            }
            slot = 1 - slot;
        }
        if (!IN) drain(1 - slot);
        if (e != hipSuccess) err.store((int)e);
    };
    std::thread helper[HC_LANES];
    int started = 0;
    const int want = (int)std::min<size_t>(g_hc.lanes, nchunk);
    try {
        for (; started < want - 1; started++) helper[started] = std::thread(work, started + 1);
    } catch (const std::exception &) {
        // no more threads: those that run do the work
    }
    work(0);
    for (int i = 0; i < started; i++) helper[i].join();
    const hipError_t e = (hipError_t)err.load();
    if (e != hipSuccess) {
        (void)hipStreamSynchronize(s);  // no DMA is left in a piece
        return fail(e == hipErrorOutOfMemory ? CPWGPU_ERR_NOMEM : CPWGPU_ERR_HIP, "host copy: %s", hipGetErrorString(e));
    }
    return CPWGPU_OK;
}

inline int copy_in(void *dev, size_t ldd, const void *host, size_t ldh, size_t width, size_t cols, hipStream_t s) {
    return host_copy_2d<true>(dev, ldd, const_cast<void *>(host), ldh, width, cols, s);
}
inline int copy_out(void *host, size_t ldh, const void *dev, size_t ldd, size_t width, size_t cols, hipStream_t s) {
    return host_copy_2d<false>(const_cast<void *>(dev), ldd, host, ldh, width, cols, s);
}

}  // namespace cpwgpu
