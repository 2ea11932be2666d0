// Just enough of HIP on the CPU for the tests to run this library's host code
// and single device functions under g++: a block's threads are threads, with a
// barrier that a thread's end leaves and cross-lane steps over 64 of them; a
// stream is a thread that runs its work in order, later than it was asked for.
#pragma once

#include <algorithm>
#include <atomic>
#include <barrier>
#include <chrono>
#include <cmath>
#include <condition_variable>
#include <cstdint>
#include <cstdlib>
#include <cstring>
#include <deque>
#include <functional>
#include <memory>
#include <mutex>
#include <thread>
#include <vector>

#define __global__
#define __device__
#define __host__
#define __forceinline__ inline
#define __launch_bounds__(...)
#define __shared__ static
#define __align__(n) alignas(n)
using std::max;
using std::min;

struct dim3 {
  unsigned x, y, z;
  dim3(unsigned a = 1, unsigned b = 1, unsigned c = 1) : x(a), y(b), z(c) {}
};
struct uint4 {
  unsigned x, y, z, w;
};
inline thread_local dim3 threadIdx(0, 0, 0), blockIdx(0, 0, 0);
inline dim3 blockDim, gridDim;

// ---- a block of threads (x only)
namespace model {
struct Block {
  std::barrier<> all;
  std::vector<std::unique_ptr<std::barrier<>>> wave;
  std::vector<unsigned> lane;  // a word per thread, exchanged within its wave
  explicit Block(int n) : all(n), lane(n) {
    for (int w = 0; w < n / 64; ++w) wave.emplace_back(new std::barrier<>(64));
  }
};
inline Block* block = nullptr;
// body by n threads of block b; before(w) runs in each thread of wave w ahead of it
template <class F, class H>
void run_block(int b, int n, F body, H before) {
  Block B(n);
  block = &B;
  std::vector<std::thread> t;
  for (int i = 0; i < n; ++i)
    t.emplace_back([&, i] {
      threadIdx = dim3(i, 0, 0);
      blockIdx = dim3(b, 0, 0);
      before(i / 64);
      body();
      B.all.arrive_and_drop();
    });
  for (auto& x : t) x.join();
}
inline unsigned from_lane(unsigned v, int src) {  // src: lane of the same wave
  const int w = threadIdx.x / 64;
  block->lane[threadIdx.x] = v;
  block->wave[w]->arrive_and_wait();
  const unsigned r = block->lane[64 * w + src];
  block->wave[w]->arrive_and_wait();
  return r;
}
struct Pair {
  unsigned v[2];
  unsigned operator[](int i) const { return v[i]; }
};
inline Pair swap_with(unsigned v, int bit) {  // the lane's value and its partner's, lower lane's first
  const int lane = threadIdx.x % 64;
  const unsigned o = from_lane(v, lane ^ bit);
  return (lane & bit) ? Pair{{o, v}} : Pair{{v, o}};
}
inline int rotated(int v, int n) {
  const int lane = threadIdx.x % 64;
  return (int)from_lane((unsigned)v, (lane & ~15) | ((lane - n) & 15));
}
}  // namespace model
inline void __syncthreads() { model::block->all.arrive_and_wait(); }
#define __builtin_amdgcn_permlane32_swap(a, b, c, d) model::swap_with(a, 32)
#define __builtin_amdgcn_permlane16_swap(a, b, c, d) model::swap_with(a, 16)
#define __builtin_amdgcn_update_dpp(o, v, ctrl, rm, bm, bc) model::rotated(v, (ctrl) - 0x120)
inline int __double2loint(double v) { uint64_t u; std::memcpy(&u, &v, 8); return (int)(uint32_t)u; }
inline int __double2hiint(double v) { uint64_t u; std::memcpy(&u, &v, 8); return (int)(uint32_t)(u >> 32); }
inline double __hiloint2double(int hi, int lo) {
  const uint64_t u = ((uint64_t)(uint32_t)hi << 32) | (uint32_t)lo;
  double v;
  std::memcpy(&v, &u, 8);
  return v;
}

// ---- types that the headers name
enum hipError_t { hipSuccess = 0, hipErrorOutOfMemory = 2, hipErrorUnknown = 999 };
inline const char* hipGetErrorString(hipError_t) { return "model"; }
struct ModelStream;
using hipStream_t = ModelStream*;
