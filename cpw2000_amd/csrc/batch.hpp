// Several launches of one kernel as one: the k-points of a small cell take the
// same kernels on their own arrays, and each launch is a few microseconds however
// little it does, with most of the GPU idle.  A kernel that can be launched so has
// its body in a struct K (K::run(Blk, args...), threads K::T, waves per SIMD K::W);
// its own __global__ function calls the body for its one grid, k_batch<K> for
// the grid of each member, their blocks one after the other.
#pragma once

#include <hip/hip_runtime.h>

#include <type_traits>
#include <vector>

namespace cpwgpu {

// the block that a body runs as: its index in the grid of its launch
struct Blk {
    int x, y, z, gx, gy, gz;
    static __device__ __forceinline__ Blk here() {
        return {(int)blockIdx.x, (int)blockIdx.y, (int)blockIdx.z, (int)gridDim.x, (int)gridDim.y, (int)gridDim.z};
    }
};

// the arguments of one member's launch, as they lie in device memory
template <typename... A> struct Pack {};
template <typename H, typename... T> struct Pack<H, T...> {
    H h;
    Pack<T...> t;
};
inline Pack<> make_pack() { return {}; }
template <typename H, typename... T> Pack<H, T...> make_pack(H h, T... t) { return {h, make_pack(t...)}; }

template <class K, typename... D> __device__ __forceinline__ void run_pack(Blk b, const Pack<> &, D... d) {
    K::run(b, d...);
}
template <class K, typename H, typename... T, typename... D>
__device__ __forceinline__ void run_pack(Blk b, const Pack<H, T...> &p, D... d) {
    run_pack<K>(b, p.t, d..., p.h);
}

// Members: at most one per lane.  first: the first block of the member, a
// multiple of 8 so that a block's XCD (blocks go round robin to the 8) is that of
// its index in its own grid.
constexpr int BATCH_MAX = 64;
struct BatchDim {
    int first, gx, gy, gz;
};
template <class K, typename... A>
__global__ __launch_bounds__(K::T, K::W) void k_batch(const BatchDim *__restrict__ dims,
                                                      const Pack<A...> *__restrict__ packs, int n) {
    const int id = blockIdx.x, lane = threadIdx.x & 63;
    const bool before = lane < n && dims[lane < n ? lane : 0].first <= id;
    const int k = __builtin_amdgcn_readfirstlane(__popcll(__ballot(before)) - 1);
    const BatchDim d = dims[k];
    const int b = id - d.first;
    if (b >= d.gx * d.gy * d.gz) return;  // padding to a multiple of 8
    const int r = b / d.gx;
    run_pack<K>(Blk{b - r * d.gx, r % d.gy, r / d.gy, d.gx, d.gy, d.gz}, packs[k]);
}

// Launches recorded instead of made (host, per thread): those of one k-point, in
// order.  ok: all of them can be batched.
struct BatchStep {
    const void *fn;  // k_batch<K, A...>
    dim3 grid;
    unsigned threads;
    size_t shmem;
    std::vector<char> args;  // Pack<A...>
};
struct Recorder {
    std::vector<BatchStep> steps;
    bool ok = true;
};
inline thread_local Recorder *g_rec = nullptr;

}  // namespace cpwgpu
