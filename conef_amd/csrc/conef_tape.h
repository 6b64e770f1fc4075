// Kernel launches that can be kept and made again.
//
// A training step's round of a bucket is the same launches with the same arguments as the step before: forming the
// tables they take (places, tiles, workspace regions of up to 24 matrices), and passing what they are formed from
// through the C interface, is half of what a round costs the host.  While a tape records on a thread, conef_launch also keeps
// the launch with a copy of its arguments.  Rounds of several buckets on two streams wait for the host: a BERT
// step at rank 8 takes 498 us with kept launches and 530 to 545 without, a WRN-28-10 step at rank 4 375 to 410 and
// 430 to 470.
#pragma once
#include <hip/hip_runtime.h>
#include <atomic>
#include <memory>
#include <tuple>
#include <utility>
#include <vector>

struct ConefTape {
    struct Launch {
        virtual ~Launch() {}
        virtual void go(hipStream_t s) = 0;
    };
    std::vector<std::unique_ptr<Launch>> launches;
    bool whole = true;                 // false: something was launched that cannot be made again from here
    std::vector<char> items;           // the caller's table as it was when these launches were formed
};

inline thread_local ConefTape* conef_recording = nullptr;

// A launch tag (workgroups that meet through records in memory know their launch by it): never 0, another one
// every time.
inline unsigned conef_next_tag(std::atomic<unsigned>& counter)
{
    const unsigned tag = (counter.fetch_add(1u) + 1u) * 0x9E3779B9u;
    return tag == 0u ? 1u : tag;
}

template <typename... P>
struct ConefKeptLaunch : ConefTape::Launch {
    void (*kernel)(P...);
    dim3 grid, block;
    unsigned lds;
    std::tuple<P...> args;
    unsigned* tag = nullptr;                       // the argument that is a launch tag, if one is
    std::atomic<unsigned>* counter = nullptr;

    template <typename... A>
    ConefKeptLaunch(void (*k)(P...), dim3 g, dim3 b, size_t l, const A&... a)
        : kernel(k), grid(g), block(b), lds((unsigned)l), args(a...) {}

    template <size_t... I>
    void make(hipStream_t s, std::index_sequence<I...>)
    {
        void* at[] = {(void*)&std::get<I>(args)...};
        (void)hipLaunchKernel((const void*)kernel, grid, block, at, lds, s);      // an error stays for hipGetLastError
    }
    void go(hipStream_t s) override
    {
        if (tag) *tag = conef_next_tag(*counter);
        make(s, std::index_sequence_for<P...>());
    }
};

// hipLaunchKernelGGL, kept where a tape records.  The arguments are copied then only: with a copy for every launch an
// LSTM step of unbiased random blocks, five hooks bound by the host, took 72.2 us against 70.7 without tapes (73.3 and
// 74.4 as it is, on a slower host).
template <typename... P, typename... A>
void conef_launch(void (*kernel)(P...), dim3 grid, dim3 block, size_t lds, hipStream_t s, const A&... args)
{
    hipLaunchKernelGGL(kernel, grid, block, (unsigned)lds, s, P(args)...);
    if (conef_recording) conef_recording->launches.emplace_back(new ConefKeptLaunch<P...>(kernel, grid, block, lds, args...));
}

// The same with argument I a launch tag drawn from `counter`.
template <size_t I, typename... P, typename... A>
void conef_launch_tagged(std::atomic<unsigned>& counter, void (*kernel)(P...), dim3 grid, dim3 block, size_t lds, hipStream_t s,
                         const A&... args)
{
    ConefKeptLaunch<P...> now(kernel, grid, block, lds, args...);
    std::get<I>(now.args) = conef_next_tag(counter);
    now.make(s, std::index_sequence_for<P...>());
    if (!conef_recording) return;
    auto* kept = new ConefKeptLaunch<P...>(std::move(now));
    conef_recording->launches.emplace_back(kept);
    kept->tag = &std::get<I>(kept->args);
    kept->counter = &counter;
}

// Something else is launched that a tape does not keep.
inline void conef_launch_unkept()
{
    if (conef_recording) conef_recording->whole = false;
}
