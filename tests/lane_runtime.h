// A wavefront on the host: 64 lanes as cooperative contexts that meet at every wavefront operation
// (ballot, shuffle, barrier), so that device code written for one wavefront per block compiles with
// the host compiler and its sanitizers. Every lane has to make the same wavefront operations, as on
// the device. Stands in for <hip/hip_runtime.h>.
#pragma once

#include <stdint.h>
#include <ucontext.h>

#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <functional>
#include <vector>

#define __device__
#define __host__
#define __global__
#define __forceinline__ inline

namespace lanes {

constexpr int kLanes = 64, kStack = 256 * 1024;
struct Lane {
    ucontext_t ctx;
    std::vector<char> stack = std::vector<char>(kStack);
    unsigned long long word[2];   // what the lane brings to this operation and the one before
    unsigned ops = 0;
    bool done = false;
};
inline Lane lane[kLanes];
inline ucontext_t home;
inline std::function<void()> body;
inline int here = 0;

inline void enter()
{
    body();
    lane[here].done = true;
    swapcontext(&lane[here].ctx, &home);
}

// Runs `f` on the 64 lanes.
inline void run(std::function<void()> f)
{
    body = std::move(f);
    for (auto& l : lane) {
        l.done = false;
        l.ops = 0;
        getcontext(&l.ctx);
        l.ctx.uc_stack.ss_sp = l.stack.data();
        l.ctx.uc_stack.ss_size = l.stack.size();
        l.ctx.uc_link = nullptr;
        makecontext(&l.ctx, enter, 0);
    }
    for (bool more = true; more;) {
        more = false;
        for (here = 0; here < kLanes; ++here) {
            swapcontext(&home, &lane[here].ctx);
            more = more || !lane[here].done;
            if (lane[here].done != lane[0].done || lane[here].ops != lane[0].ops) {
                std::fprintf(stderr, "lane %d is not at the wavefront operation of lane 0\n", here);
                std::abort();
            }
        }
    }
}

// Brings `v` and waits for the other lanes; returns which of the two words holds theirs.
inline int meet(unsigned long long v)
{
    Lane& l = lane[here];
    const int w = static_cast<int>(l.ops++ & 1u);
    l.word[w] = v;
    swapcontext(&l.ctx, &home);
    return w;
}

}  // namespace lanes

struct LaneIndex {
    struct X { operator unsigned() const { return static_cast<unsigned>(lanes::here); } } x;
};
static const LaneIndex threadIdx;
static const int warpSize = 64;

inline unsigned long long __ballot(bool p)
{
    const int w = lanes::meet(p ? 1u : 0u);
    unsigned long long m = 0;
    for (int i = 0; i < 64; ++i) m |= lanes::lane[i].word[w] << i;
    return m;
}
inline bool __any(bool p) { return __ballot(p) != 0; }
template <typename T> T __shfl(T v, int from)
{
    static_assert(sizeof(T) <= 8, "one word");
    unsigned long long b = 0;
    std::memcpy(&b, &v, sizeof(T));
    const int w = lanes::meet(b);
    std::memcpy(&v, &lanes::lane[from & 63].word[w], sizeof(T));
    return v;
}
template <typename T> T __shfl_xor(T v, int k) { return __shfl(v, lanes::here ^ k); }
inline void __syncthreads() { lanes::meet(0); }
inline int __builtin_amdgcn_readfirstlane(int v) { return __shfl(v, 0); }
inline int __popcll(unsigned long long v) { return __builtin_popcountll(v); }
inline int __popc(unsigned v) { return __builtin_popcount(v); }
inline int __ffsll(long long v) { return __builtin_ffsll(v); }
inline long long __double_as_longlong(double v) { long long b; std::memcpy(&b, &v, 8); return b; }
inline double __longlong_as_double(long long b) { double v; std::memcpy(&v, &b, 8); return v; }
template <typename T> T atomicAdd(T* p, T v) { const T old = *p; *p += v; return old; }
template <typename T> T atomicMax(T* p, T v) { const T old = *p; *p = old < v ? v : old; return old; }
template <typename T> T atomicMin(T* p, T v) { const T old = *p; *p = v < old ? v : old; return old; }
template <typename T> T atomicOr(T* p, T v) { const T old = *p; *p |= v; return old; }
inline int min(int a, int b) { return b < a ? b : a; }
inline int max(int a, int b) { return a < b ? b : a; }
using std::fmax; using std::fmin;

// Buffer loads: 0 at or beyond the buffer's size.
struct __amdgpu_buffer_rsrc_t {
    const char* base;
    uint32_t bytes;
};
inline __amdgpu_buffer_rsrc_t __builtin_amdgcn_make_buffer_rsrc(void* p, int, int bytes, int)
{
    return {static_cast<const char*>(p), static_cast<uint32_t>(bytes)};
}
template <typename T> T lane_buffer_load(__amdgpu_buffer_rsrc_t r, uint32_t off)
{
    T v = 0;
    if (off + sizeof(T) <= r.bytes && off < r.bytes) std::memcpy(&v, r.base + off, sizeof(T));
    return v;
}
inline uint8_t __builtin_amdgcn_raw_buffer_load_b8(__amdgpu_buffer_rsrc_t r, uint32_t o, int, int) { return lane_buffer_load<uint8_t>(r, o); }
inline uint16_t __builtin_amdgcn_raw_buffer_load_b16(__amdgpu_buffer_rsrc_t r, uint32_t o, int, int) { return lane_buffer_load<uint16_t>(r, o); }
inline uint32_t __builtin_amdgcn_raw_buffer_load_b32(__amdgpu_buffer_rsrc_t r, uint32_t o, int, int) { return lane_buffer_load<uint32_t>(r, o); }
inline uint64_t __builtin_amdgcn_raw_buffer_load_b64(__amdgpu_buffer_rsrc_t r, uint32_t o, int, int) { return lane_buffer_load<uint64_t>(r, o); }
