// One workgroup of a HIP kernel run on the host, for tests: every thread is a
// context of its own that runs until it reaches a barrier or a wave
// intrinsic, in an order the test chooses.  A value that one thread reads
// from another without such a point between is seen as it was before.
#pragma once
#include <ucontext.h>

#include <algorithm>
#include <cstdint>
#include <cstdlib>
#include <functional>
#include <memory>
#include <vector>

#define __global__
#define __device__
#define __host__
#define __forceinline__ inline
#define __launch_bounds__(x)
#define __shared__ static

struct Dim {
  int x;
};
static Dim threadIdx, blockIdx;

namespace emu {

constexpr int kWave = 64;
constexpr size_t kStack = 32 << 10;

enum Wait { kRun, kBlock, kWaveSync, kDone };

struct Thread {
  ucontext_t ctx;
  std::unique_ptr<char[]> stack;
  Wait wait = kRun;
};

static std::vector<Thread> threads;
static std::vector<int> lane_value;
static std::function<void()> body;
static ucontext_t scheduler;

inline void yield(Wait w) {
  Thread& t = threads[threadIdx.x];
  t.wait = w;
  swapcontext(&t.ctx, &scheduler);
}

inline void entry() {
  body();
  yield(kDone);
}

// Runs `fn` as a workgroup of order.size() threads; `order` is the sequence
// in which runnable threads take their turns.
inline void run(const std::vector<int>& order, std::function<void()> fn) {
  body = std::move(fn);
  threads = std::vector<Thread>(order.size());
  lane_value.assign(order.size(), 0);
  for (Thread& t : threads) {
    t.stack.reset(new char[kStack]);
    getcontext(&t.ctx);
    t.ctx.uc_stack.ss_sp = t.stack.get();
    t.ctx.uc_stack.ss_size = kStack;
    t.ctx.uc_link = nullptr;
    makecontext(&t.ctx, entry, 0);
  }
  auto release = [](size_t lo, size_t hi, Wait w) {  // when all that have not ended wait there
    bool any = false;
    for (size_t i = lo; i < hi; ++i) {
      if (threads[i].wait != w && threads[i].wait != kDone) return false;
      any = any || threads[i].wait == w;
    }
    for (size_t i = lo; any && i < hi; ++i)
      if (threads[i].wait == w) threads[i].wait = kRun;
    return any;
  };
  for (;;) {
    bool ran = false;
    for (int t : order) {
      if (threads[t].wait != kRun) continue;
      threadIdx.x = t;
      swapcontext(&scheduler, &threads[t].ctx);
      ran = true;
    }
    for (size_t w = 0; w < threads.size(); w += kWave) ran = release(w, w + kWave, kWaveSync) || ran;
    ran = release(0, threads.size(), kBlock) || ran;
    if (!ran) break;
  }
  for (const Thread& t : threads)
    if (t.wait != kDone) std::abort();  // a barrier that not every thread reaches
}

inline int from_lane(int v, int lane) {
  const int me = threadIdx.x, base = me / kWave * kWave;
  lane_value[me] = v;
  yield(kWaveSync);
  const int got = lane_value[base + lane];
  yield(kWaveSync);
  return got;
}

}  // namespace emu

inline void __syncthreads() { emu::yield(emu::kBlock); }
inline int __shfl_xor(int v, int mask) { return emu::from_lane(v, (threadIdx.x % 64) ^ mask); }
inline int __shfl_up(int v, int d) {
  const int lane = threadIdx.x % 64;
  return emu::from_lane(v, lane >= d ? lane - d : lane);
}
inline int atomicAdd(int* p, int v) {
  const int old = *p;
  *p += v;
  return old;
}
using std::max;
using std::min;
