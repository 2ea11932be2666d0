// Pinned-ring host transfers (t3x_stage.h).
#include "t3x_stage.h"

#include <algorithm>
#include <atomic>
#include <cstdint>
#include <cstring>
#include <exception>
#include <mutex>
#include <thread>

namespace t3x {

struct StageJob {
  char *dev, *host;
  size_t bytes, chunk, chunks;
  int slots;
  bool up;
  hipStream_t s;
  std::atomic<size_t> next{0};
  std::atomic<int> err{0};
  std::atomic<size_t> issued[32] = {};  // per slot: chunks sent down the stream so far

  void fail(hipError_t e) {
    int none = 0;
    err.compare_exchange_strong(none, (int)e);
  }
};

// 16 bytes per thread, both sides 16-byte aligned; the last n % 16 bytes by the
// last thread
__global__ __launch_bounds__(256) void k_stage_copy(const char* __restrict__ src, char* __restrict__ dst, unsigned n) {
  const unsigned i = (blockIdx.x * 256 + threadIdx.x) * 16;
  if (i + 16 <= n) *(uint4*)(dst + i) = *(const uint4*)(src + i);
  else
    for (unsigned j = i; j < n; ++j) dst[j] = src[j];
}

// Rings that no object holds, for the next one that asks.  A ring costs more than
// a handle's first copies gain by it (0.1 ms to make, 0.28 a megabyte for the first
// touch of its pages, 0.3 to free): made per handle, they brought creating a
// 36x60x36 model from 3.98 to 5.09 ms and closing it from 4.35 to 4.97; lent, 3.84
// and 4.35.
// The rings kept are the largest given back, at most kRings of them and kBytes in
// all, until the process ends.
class RingPool {
 public:
  // the smallest kept ring of at least `bytes`, or null
  char* take(size_t* bytes, int device) {
    std::lock_guard<std::mutex> lk(m_);
    Ring* best = nullptr;
    for (Ring& r : kept_)
      if (r.p && r.device == device && r.bytes >= *bytes && (!best || r.bytes < best->bytes)) best = &r;
    if (!best) return nullptr;
    char* p = best->p;
    *bytes = best->bytes;
    sum_ -= best->bytes;
    best->p = nullptr;
    return p;
  }
  // an idle ring
  void give(char* p, size_t bytes, int device) {
    char* out[kRings + 1] = {};
    int n = 0;
    {
      std::lock_guard<std::mutex> lk(m_);
      for (;;) {
        Ring *place = nullptr, *least = nullptr;
        for (Ring& r : kept_) {
          if (!r.p) place = &r;
          else if (!least || r.bytes < least->bytes) least = &r;
        }
        if (place && sum_ + bytes <= kBytes) {
          *place = Ring{p, bytes, device};
          sum_ += bytes;
          break;
        }
        if (!least || least->bytes >= bytes) {
          out[n++] = p;
          break;
        }
        out[n++] = least->p;
        sum_ -= least->bytes;
        least->p = nullptr;
      }
    }
    while (n > 0) (void)hipHostFree(out[--n]);
  }

 private:
  static constexpr int kRings = 4;
  static constexpr size_t kBytes = 32 << 20;
  struct Ring {
    char* p = nullptr;
    size_t bytes = 0;
    int device = 0;
  };
  Ring kept_[kRings];
  size_t sum_ = 0;
  std::mutex m_;
};
static RingPool gRings;

HostStage::~HostStage() {
  const bool idle = (!used_ || hipDeviceSynchronize() == hipSuccess) &&  // (drained() is the owner's way)
                    (!busy_ || hipEventSynchronize(ev_[last_]) == hipSuccess);
  for (hipEvent_t e : ev_)
    if (e) (void)hipEventDestroy(e);
  if (!ring_) return;
  if (idle) gRings.give(ring_, ringBytes_, device_);
  else (void)hipHostFree(ring_);
}

// a ring for a copy of this size
bool HostStage::reserve(size_t bytes, hipStream_t s) {
  size_t want = kMinRing;
  while (want < kMaxRing && want < bytes) want *= 2;
  if (ringBytes_ >= want) return true;
  if (failed_) return ringBytes_ > 0;
  if (drain(s) != hipSuccess) return false;
  int device = 0;
  if (hipGetDevice(&device) != hipSuccess) return false;
  char* ring = gRings.take(&want, device);
  if (!ring && hipHostMalloc((void**)&ring, want, hipHostMallocCoherent) != hipSuccess) {
    (void)hipGetLastError();  // the ring that is there, if any, serves on
    failed_ = true;
    return ringBytes_ > 0;
  }
  if (ring_) gRings.give(ring_, ringBytes_, device_);
  ring_ = ring;
  ringBytes_ = want;
  device_ = device;
  return true;
}

hipError_t HostStage::record(int slot, hipStream_t s) {
  if (!ev_[slot]) {
    const hipError_t e = hipEventCreateWithFlags(&ev_[slot], hipEventDisableTiming);
    if (e != hipSuccess) return e;
  }
  return hipEventRecord(ev_[slot], s);
}

// no upload reads the ring any more
hipError_t HostStage::drain(hipStream_t s) {
  const hipError_t e = used_ ? hipStreamSynchronize(s) : busy_ ? hipEventSynchronize(ev_[last_]) : hipSuccess;
  if (e == hipSuccess) drained();
  return e;
}

// n bytes between pinned and device memory
static hipError_t copy_pinned(char* dev, char* pin, size_t n, bool up, hipStream_t s) {
  if ((uintptr_t)dev % 16 != 0)
    return hipMemcpyAsync(up ? dev : pin, up ? pin : dev, n, up ? hipMemcpyHostToDevice : hipMemcpyDeviceToHost, s);
  const char* src = up ? pin : dev;
  char* dst = up ? dev : pin;
  unsigned len = (unsigned)n;
  void* args[] = {&src, &dst, &len};  // (its own status: the thread's last error may be another call's)
  return hipLaunchKernel((const void*)k_stage_copy, dim3((len + 4095) / 4096), dim3(256), args, 0, s);
}

// Copies of up to kMinRing bytes: one chunk, and no event, which would cost the
// stream 5 us and, waited for instead of the stream, the next call 10.  An upload
// goes behind those before it in the ring.
hipError_t HostStage::put(char* dev, const char* host, size_t bytes, hipStream_t s) {
  if (busy_ || used_ + bytes > ringBytes_) {
    const hipError_t e = drain(s);
    if (e != hipSuccess) return e;
  }
  char* pin = ring_ + used_;
  std::memcpy(pin, host, bytes);
  used_ += (bytes + 15) & ~(size_t)15;
  return copy_pinned(dev, pin, bytes, true, s);
}
hipError_t HostStage::get(char* dev, char* host, size_t bytes, hipStream_t s) {
  hipError_t e = copy_pinned(dev, ring_, bytes, false, s);  // (on the stream behind the uploads)
  if (e == hipSuccess) e = hipStreamSynchronize(s);
  if (e != hipSuccess) return e;
  drained();
  std::memcpy(host, ring_, bytes);
  return e;
}

// Chunk c between its slot and the device, and the slot's event behind it
// where somebody waits for it.
hipError_t HostStage::issue(StageJob& job, size_t c) {
  const int slot = (int)(c % job.slots);
  const size_t n = std::min(job.chunk, job.bytes - c * job.chunk);
  hipError_t e = copy_pinned(job.dev + c * job.chunk, ring_ + slot * job.chunk, n, job.up, job.s);
  if (e == hipSuccess && (!job.up || c + job.slots < job.chunks)) e = record(slot, job.s);
  job.issued[slot].store(c / job.slots + 1, std::memory_order_release);
  return e;
}

// One thread's share: the next chunk that no thread has taken, one after the
// other.  An upload fills the chunk's slot once the chunk before it in that
// slot has left it; a download waits for the chunk, empties the slot and sends
// the next chunk of that slot.
hipError_t HostStage::part(StageJob& job) {
  for (;;) {
    const size_t c = job.next.fetch_add(1, std::memory_order_relaxed);
    if (c >= job.chunks || job.err.load(std::memory_order_relaxed)) return hipSuccess;
    const int slot = (int)(c % job.slots);
    const size_t round = c / job.slots + (job.up ? 0 : 1);
    while (job.issued[slot].load(std::memory_order_acquire) < round) {  // by the thread that had the slot before
      if (job.err.load(std::memory_order_relaxed)) return hipSuccess;
      std::this_thread::yield();
    }
    char *host = job.host + c * job.chunk, *pin = ring_ + slot * job.chunk;
    const size_t n = std::min(job.chunk, job.bytes - c * job.chunk);
    hipError_t e = round ? hipEventSynchronize(ev_[slot]) : hipSuccess;
    if (e != hipSuccess) return e;
    if (job.up) {
      std::memcpy(pin, host, n);
      e = issue(job, c);
    } else {
      std::memcpy(host, pin, n);
      if (c + job.slots < job.chunks) e = issue(job, c + job.slots);
    }
    if (e != hipSuccess) return e;
  }
}

hipError_t HostStage::move(char* dev, char* host, size_t bytes, bool up, hipStream_t s) {
  const size_t chunk = std::min(chunk_of(bytes), ringBytes_);  // (a ring that could not grow)
  const int slots = (int)std::min<size_t>(ringBytes_ / chunk, kMaxSlots);
  StageJob job{dev, host, bytes, chunk, (bytes + chunk - 1) / chunk, slots, up, s};
  static_assert(sizeof(job.issued) / sizeof(job.issued[0]) == kMaxSlots, "a count per slot");
  hipError_t e = hipSuccess;
  if (up) e = drain(s);  // (a download follows the uploads on the stream)
  if (e != hipSuccess) return e;
  if (!up)
    for (size_t c = 0; e == hipSuccess && c < std::min<size_t>(job.chunks, job.slots); ++c) e = issue(job, c);
  int device = 0;
  const int nt = hipGetDevice(&device) == hipSuccess ? threads_of(bytes) : 1;
  std::thread th[kMaxThreads];
  auto run = [&](int t) {
    hipError_t r = t ? hipSetDevice(device) : e;
    if (r == hipSuccess) r = part(job);
    if (r != hipSuccess) job.fail(r);
  };
  if (e == hipSuccess) {
    try {
      for (int t = 1; t < nt; ++t) th[t] = std::thread(run, t);
    } catch (const std::exception&) {  // no thread or no memory for one: those that run take all chunks
    }
  }
  run(0);
  for (std::thread& t : th)
    if (t.joinable()) t.join();
  e = (hipError_t)job.err.load();
  if (e != hipSuccess) {
    used_ = ringBytes_;  // no slot is left to a chunk in flight
    if (hipStreamSynchronize(s) == hipSuccess) drained();
    return e;
  }
  if (up) {
    last_ = (int)((job.chunks - 1) % job.slots);
    e = record(last_, s);
    busy_ = e == hipSuccess;
    if (!busy_) used_ = ringBytes_;
  } else {
    drained();
  }
  return e;
}

// Memory that the runtime knows (pinned, registered, managed, device) is at
// the link's rate without the ring.
static bool plain_memory(const void* p) {
  hipPointerAttribute_t a;
  if (hipPointerGetAttributes(&a, p) != hipSuccess) {
    (void)hipGetLastError();
    return true;
  }
  return a.type == hipMemoryTypeUnregistered;
}

hipError_t HostStage::to_device(void* dst, const void* src, size_t bytes, hipStream_t s) {
  if (bytes == 0) return hipSuccess;
  if (plain_memory(src) && reserve(bytes, s))
    return bytes <= kMinRing ? put((char*)dst, (const char*)src, bytes, s)
                             : move((char*)dst, (char*)src, bytes, true, s);
  const hipError_t e = hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, s);
  return e == hipSuccess ? hipStreamSynchronize(s) : e;
}

hipError_t HostStage::to_host(void* dst, const void* src, size_t bytes, hipStream_t s) {
  if (bytes == 0) return hipSuccess;
  if (plain_memory(dst) && reserve(bytes, s))
    return bytes <= kMinRing ? get((char*)src, (char*)dst, bytes, s)
                             : move((char*)src, (char*)dst, bytes, false, s);
  const hipError_t e = hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, s);
  return e == hipSuccess ? hipStreamSynchronize(s) : e;
}

}  // namespace t3x
