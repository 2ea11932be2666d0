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

// ---- the runtime: streams, events, pinned memory
namespace model {
inline thread_local int newsLeft = -1;  // C++ allocations of this thread until one fails (-1: none does)
struct Spare {                          // the model's own allocations do not fail
  int keep = newsLeft;
  Spare() { newsLeft = -1; }
  ~Spare() { newsLeft = keep; }
};
inline std::atomic<int> pinnedNow{0}, pinnedCalls{0}, eventsNow{0};
inline std::atomic<size_t> pinnedLimit{~size_t(0)};  // bytes of the largest pinned allocation that succeeds
inline std::atomic<int> launchesUntilError{-1}, eventsRecorded{0};
inline std::mutex streamsMutex;
inline std::vector<ModelStream*> streams;
}  // namespace model

struct ModelStream {
  std::mutex m;
  std::condition_variable cv;
  std::deque<std::function<void()>> todo;
  unsigned long long asked = 0, ran = 0;
  bool end = false;
  std::thread t{[this] {
    unsigned seed = 1;
    for (;;) {
      std::function<void()> f;
      {
        std::unique_lock<std::mutex> l(m);
        cv.wait(l, [&] { return end || !todo.empty(); });
        if (todo.empty()) return;
        f = std::move(todo.front());
        todo.pop_front();
      }
      if ((seed = seed * 1664525u + 1013904223u) >> 30 == 0) std::this_thread::sleep_for(std::chrono::microseconds(200));
      f();
      {
        std::lock_guard<std::mutex> l(m);
        ++ran;
      }
      cv.notify_all();
    }
  }};
  ModelStream() {
    std::lock_guard<std::mutex> l(model::streamsMutex);
    model::streams.push_back(this);
  }
  ~ModelStream() {
    {
      std::lock_guard<std::mutex> l(model::streamsMutex);
      model::streams.erase(std::find(model::streams.begin(), model::streams.end(), this));
    }
    {
      std::lock_guard<std::mutex> l(m);
      end = true;
    }
    cv.notify_all();
    t.join();
  }
  unsigned long long push(std::function<void()> f) {
    std::lock_guard<std::mutex> l(m);
    todo.push_back(std::move(f));
    cv.notify_all();
    return ++asked;
  }
  void wait(unsigned long long upTo) {
    std::unique_lock<std::mutex> l(m);
    cv.wait(l, [&] { return ran >= upTo; });
  }
};
struct ModelEvent {
  ModelStream* s = nullptr;
  unsigned long long at = 0;
};
using hipEvent_t = ModelEvent*;
enum { hipEventDisableTiming = 2, hipHostMallocCoherent = 0x40000000 };
enum hipMemcpyKind { hipMemcpyHostToDevice = 1, hipMemcpyDeviceToHost = 2 };
enum hipMemoryType { hipMemoryTypeUnregistered = 0, hipMemoryTypeHost = 1 };
struct hipPointerAttribute_t {
  hipMemoryType type;
};
inline hipError_t hipPointerGetAttributes(hipPointerAttribute_t* a, const void*) {
  a->type = hipMemoryTypeUnregistered;
  return hipSuccess;
}
inline hipError_t hipGetLastError() { return hipSuccess; }
inline thread_local int modelDevice = 0;
inline hipError_t hipGetDevice(int* d) {
  *d = modelDevice;
  return hipSuccess;
}
inline hipError_t hipSetDevice(int d) {
  modelDevice = d;
  return hipSuccess;
}
inline hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
  ++model::pinnedCalls;
  if (n > model::pinnedLimit) return hipErrorOutOfMemory;
  *p = std::aligned_alloc(4096, (n + 4095) / 4096 * 4096);
  ++model::pinnedNow;
  return hipSuccess;
}
inline hipError_t hipHostFree(void* p) {
  std::memset(p, 0xCD, 4096);  // whoever still reads or fills it shows
  std::free(p);
  --model::pinnedNow;
  return hipSuccess;
}
inline hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) {
  model::Spare s;
  *e = new ModelEvent;
  ++model::eventsNow;
  return hipSuccess;
}
inline hipError_t hipEventDestroy(hipEvent_t e) {
  delete e;
  --model::eventsNow;
  return hipSuccess;
}
inline hipError_t hipEventRecord(hipEvent_t e, hipStream_t st) {
  model::Spare s;
  ++model::eventsRecorded;
  e->s = st;
  e->at = st->push([] {});
  return hipSuccess;
}
inline hipError_t hipEventSynchronize(hipEvent_t e) {
  if (e->s) e->s->wait(e->at);
  return hipSuccess;
}
inline hipError_t hipStreamSynchronize(hipStream_t st) {
  model::Spare s;
  st->wait(st->push([] {}));
  return hipSuccess;
}
inline hipError_t hipDeviceSynchronize() {
  model::Spare s;
  std::lock_guard<std::mutex> l(model::streamsMutex);
  for (ModelStream* st : model::streams) st->wait(st->push([] {}));
  return hipSuccess;
}
inline hipError_t hipMemcpyAsync(void* d, const void* h, size_t n, hipMemcpyKind, hipStream_t st) {
  model::Spare s;
  st->push([=] { std::memcpy(d, h, n); });
  return hipSuccess;
}
// kernels of the form (const char*, char*, unsigned)
inline hipError_t hipLaunchKernel(const void* f, dim3 grid, dim3 threads, void** args, size_t, hipStream_t st) {
  if (model::launchesUntilError >= 0 && model::launchesUntilError-- == 0) return hipErrorUnknown;
  model::Spare s;
  auto* k = (void (*)(const char*, char*, unsigned))f;
  const char* a = *(const char**)args[0];
  char* b = *(char**)args[1];
  const unsigned n = *(unsigned*)args[2];
  st->push([=] {
    for (unsigned g = 0; g < grid.x; ++g)
      for (unsigned t = 0; t < threads.x; ++t) {
        blockIdx = dim3(g, 0, 0);
        threadIdx = dim3(t, 0, 0);
        k(a, b, n);
      }
  });
  return hipSuccess;
}
