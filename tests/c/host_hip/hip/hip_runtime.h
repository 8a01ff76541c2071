// A workgroup on host threads, for device code that uses only what is here:
// a barrier is met when every thread of the workgroup (or of the wave, for a
// shuffle) has come to it, and a workgroup in which some thread never comes
// ends the program with status 3.
#pragma once
#include <math.h>
#include <stdint.h>
#include <stdio.h>
#include <stdlib.h>

#include <chrono>
#include <condition_variable>
#include <memory>
#include <mutex>
#include <thread>
#include <vector>

#define __device__
#define __host__
#define __forceinline__ inline
#define __align__(n) __attribute__((aligned(n)))
#define __HIP_MEMORY_SCOPE_AGENT 0
#define __hip_atomic_load(p, order, scope) (*(p))

struct HostIndex { unsigned x; };
inline thread_local HostIndex threadIdx;

class HostBarrier {
public:
    explicit HostBarrier(int n) : n_(n) {}
    void meet()
    {
        std::unique_lock<std::mutex> l(m_);
        const int turn = turn_;
        if (++here_ == n_) {
            here_ = 0;
            ++turn_;
            cv_.notify_all();
            return;
        }
        if (cv_.wait_for(l, std::chrono::seconds(20), [&] { return turn_ != turn; })) return;
        fprintf(stderr, "%d of %d threads at a barrier\n", here_, n_);
        fflush(stderr);
        _Exit(3);
    }

private:
    int n_, here_ = 0, turn_ = 0;
    std::mutex m_;
    std::condition_variable cv_;
};

struct HostBlock {
    explicit HostBlock(int n) : all(n), lane(n)
    {
        for (int w = 0; w < n; w += 64) wave.push_back(std::make_unique<HostBarrier>(64));
    }
    HostBarrier all;
    std::vector<std::unique_ptr<HostBarrier>> wave;
    std::vector<double> lane;
};
inline HostBlock *host_block;

inline void __syncthreads() { host_block->all.meet(); }
inline double __shfl_down(double v, int o, int)
{
    const unsigned t = threadIdx.x, w = t / 64;
    host_block->lane[t] = v;
    host_block->wave[w]->meet();
    const double r = t % 64 + o < 64 ? host_block->lane[t + o] : v;
    host_block->wave[w]->meet();
    return r;
}

// f() by n threads (a multiple of 64)
template <class F> void run_block(int n, F f)
{
    HostBlock b(n);
    host_block = &b;
    std::vector<std::thread> ts;
    for (int t = 0; t < n; ++t)
        ts.emplace_back([t, &f] {
            threadIdx.x = (unsigned)t;
            f();
        });
    for (auto &t : ts) t.join();
}
