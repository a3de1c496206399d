// What the whole-solve kernels need of HIP to be compiled for the host, one lane per wavefront: a workgroup of one (64 threads)
// or two wavefronts (128) runs as one or two host threads, each standing for lane 0 of its wavefront.  A vote of the
// wavefront is the lane's own condition, a shuffle its own value, a barrier one between the threads; the dynamic LDS of a
// launch is a heap block of exactly the bytes asked for.  Loops in which the lanes share out work (evaluation times into
// LDS) reach their first element only: a batch of one sample with one evaluation point.
#pragma once
#include <math.h>
#include <stddef.h>
#include <stdint.h>
#include <string.h>

#include <condition_variable>
#include <functional>
#include <mutex>
#include <thread>
#include <vector>

#define __device__
#define __host__
#define __global__
#define __shared__
#define __forceinline__ inline
#define __launch_bounds__(...)

struct dim3 {
    unsigned x, y, z;
    dim3(unsigned x_ = 1, unsigned y_ = 1, unsigned z_ = 1) : x(x_), y(y_), z(z_) {}
};
typedef void *hipStream_t;
typedef int hipError_t;
inline hipError_t hipGetLastError() { return 0; }

namespace host {
struct Barrier {
    std::mutex m;
    std::condition_variable cv;
    int waiting = 0, turn = 0, threads = 1;
    void wait() {
        std::unique_lock<std::mutex> lock(m);
        const int mine = turn;
        if (++waiting == threads) {
            waiting = 0, ++turn;
            cv.notify_all();
        } else {
            cv.wait(lock, [&] { return turn != mine; });
        }
    }
};
extern thread_local dim3 thread_idx, block_idx, grid_dim;
extern unsigned char *lds;
extern Barrier barrier;

inline void launch(const std::function<void()> &kernel, dim3 grid, dim3 block, size_t lds_bytes) {
    for (unsigned b = 0; b < grid.x; ++b) {
        lds = new unsigned char[lds_bytes];
        const int waves = (int)(block.x + 63) / 64;
        barrier.threads = waves;
        std::vector<std::thread> threads;
        for (int w = 0; w < waves; ++w)
            threads.emplace_back([&, w] {
                thread_idx = dim3(64 * w, 0, 0), block_idx = dim3(b, 0, 0), grid_dim = grid;
                kernel();
            });
        for (auto &t : threads) t.join();
        delete[] lds;
    }
}
template <typename To, typename From> inline To bits(From v) {
    static_assert(sizeof(To) == sizeof(From), "sizes");
    To r;
    memcpy(&r, &v, sizeof r);
    return r;
}
}  // namespace host

#define threadIdx host::thread_idx
#define blockIdx host::block_idx
#define gridDim host::grid_dim
#define hipLaunchKernelGGL(kernel, grid, block, lds, stream, ...) host::launch([&] { kernel(__VA_ARGS__); }, grid, block, lds)

template <typename A> inline A min(A a, A b) { return b < a ? b : a; }
template <typename A> inline A max(A a, A b) { return a < b ? b : a; }
inline void __syncthreads() { host::barrier.wait(); }
template <typename T> inline T __shfl_xor(T v, int) { return v; }
inline void atomicMax(int32_t *p, int v) {
    static std::mutex m;
    std::lock_guard<std::mutex> lock(m);
    if (*p < v) *p = v;
}
inline int __float_as_int(float v) { return host::bits<int>(v); }
inline unsigned __float_as_uint(float v) { return host::bits<unsigned>(v); }
inline float __int_as_float(int v) { return host::bits<float>(v); }
inline float __uint_as_float(unsigned v) { return host::bits<float>(v); }
inline double __longlong_as_double(long long v) { return host::bits<double>(v); }
inline int __double2hiint(double v) { return (int)(host::bits<unsigned long long>(v) >> 32); }
inline int __double2loint(double v) { return (int)host::bits<unsigned long long>(v); }
inline double __hiloint2double(int hi, int lo) { return host::bits<double>(((unsigned long long)(unsigned)hi << 32) | (unsigned)lo); }

#define __HIP_MEMORY_SCOPE_AGENT 0
#define __HIP_MEMORY_SCOPE_SYSTEM 0
#define __hip_atomic_fetch_add(p, v, order, scope) __atomic_fetch_add(p, v, __ATOMIC_SEQ_CST)
#define __hip_atomic_exchange(p, v, order, scope) __atomic_exchange_n(p, v, __ATOMIC_SEQ_CST)
#define __hip_atomic_store(p, v, order, scope) __atomic_store_n(p, v, __ATOMIC_SEQ_CST)
#define __builtin_amdgcn_fence(...)
#define __builtin_amdgcn_s_barrier() __syncthreads()
#define __builtin_amdgcn_mov_dpp(v, ...) (v)
#define __builtin_amdgcn_readlane(v, lane) (v)
#define __builtin_amdgcn_ballot_w64(c) ((c) ? 1ull : 0ull)
#define __builtin_amdgcn_inverse_ballot_w64(l) (((l) & 1ull) != 0)
#define __builtin_amdgcn_rcpf(x) (1.0f / (x))
#define __builtin_amdgcn_rcp(x) (1.0 / (x))
#define __builtin_amdgcn_rsqf(x) (1.0f / sqrtf(x))
#define __builtin_amdgcn_rsq(x) (1.0 / sqrt(x))
#define __builtin_amdgcn_ldexpf(x, e) ldexpf(x, e)
#define __builtin_amdgcn_ldexp(x, e) ldexp(x, e)
