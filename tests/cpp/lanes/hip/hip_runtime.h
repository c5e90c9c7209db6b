// Stand-in for <hip/hip_runtime.h> that compiles the device headers as host
// code and runs a launch on the CPU: every lane of a workgroup is a fiber, a
// barrier or a cross-lane read lets the others run until all have arrived.
// Test infrastructure: with it the kernels themselves, indexes, LDS and
// barriers included, run under the compiler's address and undefined-behaviour
// checks.  Cross-lane reads need all live lanes of a wave, as the kernels
// promise; lanes that disagree are reported.
#pragma once

#include <ucontext.h>

#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <functional>
#include <memory>
#include <vector>

#if defined(__SANITIZE_ADDRESS__)
#include <sanitizer/asan_interface.h>
#include <sanitizer/common_interface_defs.h>
#endif

#define __host__
#define __device__
#define __global__
#define __shared__ static
#define __launch_bounds__(...)
#define amdgpu_waves_per_eu(...)
#define __align__(n) __attribute__((aligned(n)))
#define HIP_DYNAMIC_SHARED(type, var) type* var = reinterpret_cast<type*>(lanes::lds());
#define __HIP_MEMORY_SCOPE_AGENT 0
#define __hip_atomic_store(p, v, order, scope) (*(p) = (v))
#define __builtin_nontemporal_store(v, p) (*(p) = (v))
#define __builtin_amdgcn_sched_barrier(mask)
#define __builtin_amdgcn_wave_barrier()
#define __builtin_amdgcn_fence(...)

struct dim3_value
{
    unsigned x, y, z;
};
struct int4
{
    int x, y, z, w;
};

inline dim3_value threadIdx, blockIdx, blockDim, gridDim;

namespace lanes
{

struct lane
{
    ucontext_t context;
    char*      stack    = nullptr;
    void*      shadow   = nullptr; // the sanitizer's record of the fiber's stack
    bool       done     = false;
    uint64_t   barriers = 0, reads = 0; // passed or waited for
};

constexpr size_t kStack = 128 * 1024;

// A stack for lane t, used again by the next workgroup.
inline char* stack_of(unsigned t)
{
    static std::vector<std::unique_ptr<char[]>> stacks;
    if (stacks.size() <= t) stacks.resize(t + 1);
    if (!stacks[t]) stacks[t].reset(new char[kStack]);
#if defined(__SANITIZE_ADDRESS__)
    ASAN_UNPOISON_MEMORY_REGION(stacks[t].get(), kStack); // the last lane's frames
#endif
    return stacks[t].get();
}

struct workgroup
{
    std::vector<lane>     lane_of;
    ucontext_t            scheduler;
    void*                 scheduler_shadow = nullptr;
    const void*           scheduler_stack  = nullptr;
    size_t                scheduler_size   = 0;
    unsigned              current          = 0;
    uint64_t              progress         = 0;
    std::vector<uint64_t> value[2]; // what each lane offers to a cross-lane read, alternately
    std::vector<char>     lds;
    std::function<void()> body;
};

inline workgroup* g_group = nullptr;

inline void* lds() { return g_group->lds.data(); }

inline void switch_to_scheduler(bool finished)
{
    workgroup& g = *g_group;
    lane&      l = g.lane_of[g.current];
#if defined(__SANITIZE_ADDRESS__)
    __sanitizer_start_switch_fiber(finished ? nullptr : &l.shadow, g.scheduler_stack, g.scheduler_size);
#endif
    (void)finished;
    swapcontext(&l.context, &g.scheduler);
#if defined(__SANITIZE_ADDRESS__)
    __sanitizer_finish_switch_fiber(l.shadow, &g.scheduler_stack, &g.scheduler_size);
#endif
}

inline void enter()
{
#if defined(__SANITIZE_ADDRESS__)
    __sanitizer_finish_switch_fiber(nullptr, &g_group->scheduler_stack, &g_group->scheduler_size);
#endif
    g_group->body();
    g_group->lane_of[g_group->current].done = true;
    ++g_group->progress;
    switch_to_scheduler(true);
}

// Lets the other lanes run until arrived() holds.
template <class Fn>
void wait(Fn&& arrived)
{
    ++g_group->progress;
    while (!arrived()) switch_to_scheduler(false);
}

inline void barrier()
{
    workgroup&     g = *g_group;
    const uint64_t k = ++g.lane_of[g.current].barriers;
    wait([&] {
        for (auto const& l : g.lane_of)
            if (!l.done && l.barriers < k) return false;
        return true;
    });
}

// Offers v to the wave's other lanes and returns what all 64 offered (0 where
// a lane has ended).
inline const uint64_t* offer(uint64_t v)
{
    workgroup&     g    = *g_group;
    const unsigned me   = g.current, first = me / 64 * 64;
    const uint64_t k    = ++g.lane_of[me].reads;
    g.value[k & 1][me]  = v;
    wait([&] {
        for (unsigned l = first; l < first + 64; ++l)
            if (g.lane_of[l].done)
                g.value[k & 1][l] = 0;
            else if (g.lane_of[l].reads < k)
                return false;
        return true;
    });
    return &g.value[k & 1][first];
}

// What lane from(lane) of the wave offered (0 from none).
template <class Fn>
uint64_t read_lane(uint64_t v, Fn&& from)
{
    const uint64_t* all = offer(v);
    const int       f   = from(static_cast<int>(threadIdx.x % 64));
    return f < 0 || f > 63 ? 0 : all[f];
}

inline void run_workgroup(unsigned nt, size_t lds_bytes, std::function<void()> body)
{
    workgroup g;
    g_group   = &g;
    g.lane_of = std::vector<lane>(nt);
    g.body    = std::move(body);
    g.lds.assign(lds_bytes, '\xff'); // NaNs: what is read before it is written shows
    for (auto& v : g.value) v.assign(nt, 0);
    for (unsigned t = 0; t < nt; ++t)
    {
        lane& l = g.lane_of[t];
        l.stack = stack_of(t);
        getcontext(&l.context);
        l.context.uc_stack.ss_sp   = l.stack;
        l.context.uc_stack.ss_size = kStack;
        l.context.uc_link          = nullptr;
        makecontext(&l.context, enter, 0);
    }
    for (bool live = true; live;)
    {
        const uint64_t before = g.progress;
        live                  = false;
        for (unsigned t = 0; t < nt; ++t)
        {
            if (g.lane_of[t].done) continue;
            live        = true;
            g.current   = t;
            threadIdx.x = t;
#if defined(__SANITIZE_ADDRESS__)
            __sanitizer_start_switch_fiber(&g.scheduler_shadow, g.lane_of[t].stack, kStack);
#endif
            swapcontext(&g.scheduler, &g.lane_of[t].context);
#if defined(__SANITIZE_ADDRESS__)
            __sanitizer_finish_switch_fiber(g.scheduler_shadow, nullptr, nullptr);
#endif
        }
        if (live && g.progress == before)
        {
            std::fprintf(stderr, "lanes wait for each other: a barrier or cross-lane read not all of them reach\n");
            std::abort();
        }
    }
    g_group = nullptr;
}

// kernel(arguments...) on `blocks` workgroups of nt lanes, one after another.
template <class Kernel, class... Args>
void launch(Kernel kernel, unsigned blocks, unsigned nt, size_t lds_bytes, Args... args)
{
    gridDim  = { blocks, 1, 1 };
    blockDim = { nt, 1, 1 };
    for (unsigned b = 0; b < blocks; ++b)
    {
        blockIdx = { b, 0, 0 };
        run_workgroup(nt, lds_bytes, [&] { kernel(args...); });
    }
}

template <class T>
uint64_t bits_of(T v)
{
    uint64_t b = 0;
    static_assert(sizeof(T) <= 8);
    std::memcpy(&b, &v, sizeof(T));
    return b;
}
template <class T>
T value_of(uint64_t b)
{
    T v;
    std::memcpy(&v, &b, sizeof(T));
    return v;
}

// The wave's value of `old` for a lane that a DPP move leaves out.
inline int dpp(int old, int v, int ctrl, bool zero)
{
    bool       none = false;
    const auto got  = read_lane(bits_of(v), [&](int l) {
        const int row = l & ~15, x = l & 15;
        int       from = -1;
        if (ctrl > 0x100 && ctrl < 0x110) from = x + (ctrl - 0x100) < 16 ? l + (ctrl - 0x100) : -1;       // row_shl
        else if (ctrl > 0x110 && ctrl < 0x120) from = x - (ctrl - 0x110) >= 0 ? l - (ctrl - 0x110) : -1;  // row_shr
        else if (ctrl > 0x120 && ctrl < 0x130) from = row + ((x - (ctrl - 0x120)) & 15);                  // row_ror
        else if (ctrl == 0x130) from = l < 63 ? l + 1 : -1;                                               // wave_shl
        else if (ctrl == 0x138) from = l - 1;                                                             // wave_shr
        else
            std::abort();
        none = from < 0;
        return from;
    });
    return none ? (zero ? 0 : old) : value_of<int>(got);
}

struct pair
{
    unsigned v[2];
    unsigned operator[](int k) const { return v[k]; }
};

// v_permlane{16,32}_swap: the odd rows (halves) of a against the even ones of b.
inline pair permlane_swap(unsigned a, unsigned b, int width)
{
    const unsigned other_a = value_of<unsigned>(read_lane(bits_of(a), [&](int l) { return l ^ width; }));
    const unsigned other_b = value_of<unsigned>(read_lane(bits_of(b), [&](int l) { return l ^ width; }));
    const bool     odd     = (threadIdx.x & static_cast<unsigned>(width)) != 0;
    return { { odd ? other_b : a, odd ? b : other_a } };
}

} // namespace lanes

#define __builtin_amdgcn_update_dpp(old, v, ctrl, rows, banks, bound) lanes::dpp(old, v, ctrl, bound)
#define __builtin_amdgcn_readlane(v, l) lanes::value_of<unsigned>(lanes::read_lane(lanes::bits_of(v), [&](int) { return l; }))
#define __builtin_amdgcn_readfirstlane(v) \
    lanes::value_of<std::remove_const_t<decltype(v)>>(lanes::read_lane(lanes::bits_of(v), [&](int) { return 0; }))
#define __builtin_amdgcn_permlane32_swap(a, b, fi, bound) lanes::permlane_swap(a, b, 32)
#define __builtin_amdgcn_permlane16_swap(a, b, fi, bound) lanes::permlane_swap(a, b, 16)

inline void __syncthreads() { lanes::barrier(); }
inline void __threadfence_system() {}
inline int  __any(int v)
{
    const uint64_t* all = lanes::offer(v != 0);
    int             any = 0;
    for (int l = 0; l < 64; ++l) any |= static_cast<int>(all[l]);
    return any;
}
template <class T>
T __shfl(T v, int l, int = 64)
{
    return lanes::value_of<T>(lanes::read_lane(lanes::bits_of(v), [&](int) { return l & 63; }));
}
// past the wave's end a lane keeps its own value
template <class T>
T __shfl_down(T v, unsigned by, int = 64)
{
    return lanes::value_of<T>(
        lanes::read_lane(lanes::bits_of(v), [&](int l) { return l + static_cast<int>(by) < 64 ? l + static_cast<int>(by) : l; }));
}
template <class T>
T __shfl_up(T v, unsigned by, int = 64)
{
    return lanes::value_of<T>(
        lanes::read_lane(lanes::bits_of(v), [&](int l) { return l >= static_cast<int>(by) ? l - static_cast<int>(by) : l; }));
}
template <class T>
T __shfl_xor(T v, int mask, int = 64)
{
    return lanes::value_of<T>(lanes::read_lane(lanes::bits_of(v), [&](int l) { return l ^ mask; }));
}
inline double    __longlong_as_double(long long v) { return lanes::value_of<double>(lanes::bits_of(v)); }
inline long long __double_as_longlong(double v) { return lanes::value_of<long long>(lanes::bits_of(v)); }

// one lane runs at a time
template <class T, class V>
T atomicMin(T* p, V v)
{
    const T old = *p;
    if (v < old) *p = static_cast<T>(v);
    return old;
}
template <class T, class V>
T atomicMax(T* p, V v)
{
    const T old = *p;
    if (v > old) *p = static_cast<T>(v);
    return old;
}
template <class T, class V>
T atomicOr(T* p, V v)
{
    const T old = *p;
    *p          = static_cast<T>(old | v);
    return old;
}
template <class T, class V>
T atomicAdd(T* p, V v)
{
    const T old = *p;
    *p          = static_cast<T>(old + v);
    return old;
}
