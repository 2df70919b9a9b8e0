// A model of a kernel's lanes on the CPU, in place of the HIP runtime, for kernels whose lanes
// meet at __syncthreads(), at wave_sync() and in the quad exchanges (b3_quad_compress).
//
// A block's lanes are coroutines that run one after another, each as far as its next meeting
// point, so what a lane reads that another lane wrote is there only if a meeting point stands
// between the two: an order that a kernel merely happens to get from the compiler is not given
// here. Lanes of a quad meet in wave_sync() and in the exchanges (the waves of the kernels
// modelled share nothing else between barriers); all lanes of a block meet in __syncthreads().
#pragma once

#include <stddef.h>
#include <stdint.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>
#include <ucontext.h>

#include <algorithm>
#include <functional>
#include <vector>

#define __global__ static
#define __device__
#define __host__
#define __shared__ static
#define __forceinline__ inline
#define __launch_bounds__(...)
#define __align__(n) __attribute__((aligned(n)))

struct dim3 {
  uint32_t x, y, z;
  dim3(uint32_t x_ = 1, uint32_t y_ = 1, uint32_t z_ = 1) : x(x_), y(y_), z(z_) {}
};
struct uint4 {
  uint32_t x, y, z, w;
} __attribute__((aligned(16)));
inline uint4 make_uint4(uint32_t x, uint32_t y, uint32_t z, uint32_t w) { return {x, y, z, w}; }

using std::max;
using std::min;
inline int __clzll(unsigned long long v) { return v ? __builtin_clzll(v) : 64; }
inline int __popcll(unsigned long long v) { return __builtin_popcountll(v); }

namespace lanes {

constexpr size_t kStack = 64 << 10;

struct Lane {
  ucontext_t at;
  std::vector<char> stack;
  enum { kReady, kQuad, kBlock, kDone } state = kReady;
  uint32_t shown = 0;  // what the lane brings to an exchange
};

inline std::vector<Lane> g_lanes;
inline ucontext_t g_main;
inline uint32_t g_cur = 0;
inline std::function<void()> g_body;
inline bool g_last_first = false;  // lanes run from the last to the first

inline void entry() {
  g_body();
  g_lanes[g_cur].state = Lane::kDone;
}

inline void wait_in(decltype(Lane::state) s) {
  Lane& l = g_lanes[g_cur];
  l.state = s;
  swapcontext(&l.at, &g_main);
}

// Lets the lanes that wait in `s` among [a, b) go once every one of them that still runs does.
inline void release(uint32_t a, uint32_t b, decltype(Lane::state) s) {
  bool any = false;
  for (uint32_t i = a; i < b; i++) {
    if (g_lanes[i].state == s) any = true;
    else if (g_lanes[i].state != Lane::kDone) return;
  }
  for (uint32_t i = a; any && i < b; i++)
    if (g_lanes[i].state == s) g_lanes[i].state = Lane::kReady;
}

}  // namespace lanes

inline dim3 blockIdx, gridDim, blockDim;
// (a lane's own index, also after another lane has run)
struct LaneIndex {
  struct X {
    operator uint32_t() const { return lanes::g_cur; }
  } x;
};
inline LaneIndex threadIdx;

inline void __syncthreads() { lanes::wait_in(lanes::Lane::kBlock); }

inline uint32_t lanes_quad_exchange(uint32_t v, int perm) {
  using namespace lanes;
  g_lanes[g_cur].shown = v;
  wait_in(Lane::kQuad);
  const uint32_t from = (g_cur & ~3u) + ((uint32_t)perm >> (2 * (g_cur & 3)) & 3u);
  const uint32_t got = g_lanes[from].shown;
  wait_in(Lane::kQuad);  // every lane has read before one shows its next value
  return got;
}

#define __builtin_amdgcn_update_dpp(old, v, perm, row, bank, bound) \
  ((int)lanes_quad_exchange((uint32_t)(v), (perm)))
#define __builtin_amdgcn_fence(order, scope) ((void)0)
#define __builtin_amdgcn_wave_barrier() lanes::wait_in(lanes::Lane::kQuad)

namespace lanes {

inline void run_block(uint32_t n) {
  g_lanes.clear();
  g_lanes.resize(n);
  for (Lane& l : g_lanes) {
    l.stack.resize(kStack);
    getcontext(&l.at);
    l.at.uc_stack.ss_sp = l.stack.data();
    l.at.uc_stack.ss_size = kStack;
    l.at.uc_link = &g_main;
    makecontext(&l.at, entry, 0);
  }
  for (;;) {
    bool ran = false;
    for (uint32_t t = 0; t < n; t++) {
      g_cur = g_last_first ? n - 1 - t : t;
      if (g_lanes[g_cur].state != Lane::kReady) continue;
      ran = true;
      swapcontext(&g_main, &g_lanes[g_cur].at);
    }
    for (uint32_t q = 0; q < n; q += 4) release(q, q + 4, Lane::kQuad);
    release(0, n, Lane::kBlock);
    if (!ran) break;
  }
  for (uint32_t t = 0; t < n; t++)
    if (g_lanes[t].state != Lane::kDone) {
      fprintf(stderr, "lane %u waits for lanes that never come\n", t);
      exit(2);
    }
}

}  // namespace lanes

typedef int hipError_t;
typedef void* hipStream_t;
enum { hipSuccess = 0, hipErrorOutOfMemory = 2 };
enum hipMemcpyKind { hipMemcpyHostToDevice, hipMemcpyDeviceToHost };
inline hipError_t hipGetLastError() { return hipSuccess; }
inline hipError_t hipDeviceSynchronize() { return hipSuccess; }
inline hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) {
  memcpy(d, s, n);
  return hipSuccess;
}

template <class Kernel, class... Args>
void hipLaunchKernelGGL(Kernel kernel, dim3 grid, dim3 block, size_t, hipStream_t, Args... args) {
  gridDim = grid;
  blockDim = block;
  lanes::g_body = [=] { kernel(args...); };
  for (uint32_t b = 0; b < grid.x; b++) {
    blockIdx = dim3(b);
    lanes::run_block(block.x);
  }
}
