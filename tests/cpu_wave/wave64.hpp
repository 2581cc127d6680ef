// wave64.hpp -- runs this library's device code on the CPU, a workgroup at a
// time, for tests of what its kernels read and launch: every lane is a fiber,
// and the operations across lanes (ballots, shuffles, barriers) wait for the
// workgroup's or wavefront's lanes that have not returned.  The lanes of a
// wavefront have to reach the same ones of these in the same order, so a
// kernel can be run here only where none of them is in divergent code.
//
// Include it before any header or source of the library, compiled as plain C++.
#pragma once
#include <hip/hip_runtime.h>
#include <signal.h>
#include <sys/mman.h>
#include <ucontext.h>
#include <unistd.h>

#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <functional>
#include <memory>
#include <vector>

#undef __shared__
#define __shared__ static
#undef __launch_bounds__
#define __launch_bounds__(...)
#define amdgpu_waves_per_eu(...) unused
#undef threadIdx
#undef blockIdx
#undef blockDim
#undef gridDim

namespace wave64 {

struct Lane {
    ucontext_t ctx;
    std::unique_ptr<char[]> stack;
    bool done = false;
    uint64_t waits = 0, value = 0;  // barriers passed; the value published at the last
};
inline std::vector<Lane> lanes;
inline ucontext_t home;
inline size_t cur = 0;
inline dim3 tid, bid, bdim, gdim;
inline std::function<void()> body;
inline uint64_t launches = 0;
inline dim3 last_grid, last_block;
inline bool execute = true;  // false: launches are only recorded

inline void fiber() {
    body();
    lanes[cur].done = true;
    swapcontext(&lanes[cur].ctx, &home);
}

// Waits until every lane of [first, first + count) that has not returned has
// come here as often as this one.
inline void wait(size_t first, size_t count) {
    const uint64_t mine = ++lanes[cur].waits;
    for (;;) {
        bool all = true;
        for (size_t l = first; l < first + count && l < lanes.size(); l++) all &= lanes[l].done || lanes[l].waits >= mine;
        if (all) return;
        swapcontext(&lanes[cur].ctx, &home);
    }
}
inline void wave_wait() { wait(cur & ~size_t(63), 64); }

// f over the wavefront's live lanes' values, which stay published until each
// lane has read them.
template <class F>
auto gather(uint64_t v, F&& f) {
    lanes[cur].value = v;
    wave_wait();
    const auto r = f(cur & ~size_t(63));
    wave_wait();
    return r;
}
inline bool live(size_t l) { return l < lanes.size() && !lanes[l].done; }

inline uint64_t ballot(bool b) {
    return gather(b, [](size_t w) {
        uint64_t m = 0;
        for (size_t l = 0; l < 64; l++)
            if (live(w + l) && lanes[w + l].value) m |= 1ull << l;
        return m;
    });
}
inline uint32_t read_lane(uint32_t v, size_t l) {
    return gather(v, [=](size_t w) { return live(w + l) ? (uint32_t)lanes[w + l].value : 0u; });
}
inline uint32_t read_first(uint32_t v) {
    return gather(v, [](size_t w) {
        size_t l = w;
        while (!live(l)) l++;
        return (uint32_t)lanes[l].value;
    });
}

template <class K, class... A>
void launch(K kernel, dim3 grid, dim3 block, A... args) {
    launches++;
    last_grid = grid;
    last_block = block;
    if (!execute) return;
    gdim = grid;
    bdim = block;
    body = [=] { kernel(args...); };
    for (uint64_t b = 0; b < (uint64_t)grid.x * grid.y; b++) {
        bid = dim3((uint32_t)(b % grid.x), (uint32_t)(b / grid.x), 0);
        lanes.clear();
        lanes.resize(block.x);
        for (Lane& l : lanes) {
            l.stack.reset(new char[1 << 17]);
            getcontext(&l.ctx);
            l.ctx.uc_stack.ss_sp = l.stack.get();
            l.ctx.uc_stack.ss_size = 1 << 17;
            l.ctx.uc_link = &home;
            makecontext(&l.ctx, fiber, 0);
        }
        for (bool more = true; more;) {
            more = false;
            for (cur = 0; cur < lanes.size(); cur++) {
                if (lanes[cur].done) continue;
                tid = dim3((uint32_t)cur, 0, 0);
                swapcontext(&home, &lanes[cur].ctx);
                more |= !lanes[cur].done;
            }
        }
    }
}

// n words in the middle of an otherwise unreadable range: a read at an index
// that is off by any number of 32 bits ends the program with status 1.
constexpr size_t kGuard = size_t(1) << 35;
inline std::vector<char*> guards;
inline void outside(int sig, siginfo_t* info, void*) {
    const char* at = static_cast<const char*>(info->si_addr);
    for (const char* g : guards)
        if (at >= g && at < g + kGuard) {
            const char text[] = "a read outside of a guarded array\n";
            if (write(1, text, sizeof(text) - 1) > 0) _exit(1);
        }
    signal(sig, SIG_DFL);
}
inline uint32_t* guarded(size_t n) {
    const size_t span = kGuard, bytes = (4 * n + 4095) & ~size_t(4095);
    char* p = static_cast<char*>(mmap(nullptr, span + bytes + 4096, PROT_NONE, MAP_PRIVATE | MAP_ANONYMOUS | MAP_NORESERVE, -1, 0));
    if (p == MAP_FAILED || mprotect(p + span / 2, bytes, PROT_READ | PROT_WRITE) != 0) {
        std::perror("guarded");
        std::exit(2);
    }
    static const bool installed = [] {
        struct sigaction a = {};
        a.sa_sigaction = outside;
        a.sa_flags = SA_SIGINFO;
        return sigaction(SIGSEGV, &a, nullptr) == 0;
    }();
    if (installed) guards.push_back(p);
    return reinterpret_cast<uint32_t*>(p + span / 2 + bytes - 4 * n);  // the last word ends at the unreadable part
}

}  // namespace wave64

#define threadIdx (wave64::tid)
#define blockIdx (wave64::bid)
#define blockDim (wave64::bdim)
#define gridDim (wave64::gdim)
#undef hipLaunchKernelGGL
#define hipLaunchKernelGGL(kernel, grid, block, lds, stream, ...) wave64::launch(kernel, grid, block, __VA_ARGS__)

inline uint32_t __lane_id() { return (uint32_t)(wave64::cur & 63); }
inline uint64_t __ballot(int b) { return wave64::ballot(b != 0); }
inline int __any(int b) { return wave64::ballot(b != 0) != 0; }
inline int __shfl_up(int v, unsigned d) {
    const uint32_t l = __lane_id();
    return (int)wave64::read_lane((uint32_t)v, l >= d ? l - d : l);
}
inline int __shfl(int v, int l) { return (int)wave64::read_lane((uint32_t)v, (size_t)l); }
inline float __shfl(float v, int l) {
    uint32_t u;
    std::memcpy(&u, &v, 4);
    u = wave64::read_lane(u, (size_t)l);
    std::memcpy(&v, &u, 4);
    return v;
}
inline void __syncthreads() { wave64::wait(0, wave64::lanes.size()); }
inline uint32_t __builtin_amdgcn_readfirstlane(uint32_t v) { return wave64::read_first(v); }
inline uint32_t __builtin_amdgcn_readlane(uint32_t v, int l) { return wave64::read_lane(v, (size_t)l); }
inline uint32_t __builtin_amdgcn_mbcnt_lo(uint32_t m, uint32_t v) {
    const uint32_t l = __lane_id();
    return v + (uint32_t)__builtin_popcount(l < 32 ? m & ((1u << l) - 1u) : m);
}
inline uint32_t __builtin_amdgcn_mbcnt_hi(uint32_t m, uint32_t v) {
    const uint32_t l = __lane_id();
    return v + (uint32_t)__builtin_popcount(l < 32 ? 0u : m & ((1u << (l - 32)) - 1u));
}
inline uint32_t __builtin_amdgcn_alignbit(uint32_t hi, uint32_t lo, uint32_t s) {
    return (uint32_t)((((uint64_t)hi << 32) | lo) >> (s & 31));
}
inline float __builtin_amdgcn_fmed3f(float a, float b, float c) { return std::fmax(std::fmin(a, b), std::fmin(std::fmax(a, b), c)); }
inline float __builtin_amdgcn_rsqf(float v) { return 1.0f / std::sqrt(v); }
inline float __builtin_amdgcn_rcpf(float v) { return 1.0f / v; }
inline float __builtin_amdgcn_sqrtf(float v) { return std::sqrt(v); }
inline uint32_t __builtin_bitreverse32(uint32_t v) {
    uint32_t r = 0;
    for (int k = 0; k < 32; k++) r |= ((v >> k) & 1u) << (31 - k);
    return r;
}
#define __builtin_amdgcn_wave_barrier() wave64::wave_wait()
#define __builtin_amdgcn_fence(order, scope) ((void)0)
inline int __ffs(int v) { return __builtin_ffs(v); }
inline int __ffsll(long long v) { return __builtin_ffsll(v); }
inline int __popc(uint32_t v) { return __builtin_popcount(v); }
inline int __popcll(uint64_t v) { return __builtin_popcountll(v); }
inline uint32_t __float_as_uint(float v) {
    uint32_t u;
    std::memcpy(&u, &v, 4);
    return u;
}
inline float __fmaf_rn(float a, float b, float c) { return std::fma(a, b, c); }
// (one fiber runs at a time)
inline uint32_t atomicAdd(uint32_t* p, uint32_t v) { const uint32_t o = *p; *p += v; return o; }
inline uint32_t atomicMin(uint32_t* p, uint32_t v) { const uint32_t o = *p; if (v < o) *p = v; return o; }
inline uint32_t atomicMax(uint32_t* p, uint32_t v) { const uint32_t o = *p; if (v > o) *p = v; return o; }
inline uint32_t atomicOr(uint32_t* p, uint32_t v) { const uint32_t o = *p; *p |= v; return o; }
#define __hip_atomic_fetch_add(p, v, order, scope) atomicAdd(p, v)
template <class A, class B>
inline auto min(A a, B b) { using T = std::common_type_t<A, B>; return (T)a < (T)b ? (T)a : (T)b; }
template <class A, class B>
inline auto max(A a, B b) { using T = std::common_type_t<A, B>; return (T)a > (T)b ? (T)a : (T)b; }
