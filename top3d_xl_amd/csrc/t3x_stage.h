// Copies between a caller's pageable memory and the device through a ring of
// pinned chunks.
//
// Bound: the link (56 GB/s either way into pinned memory).  Handed pageable
// memory the runtime reaches 30-36 GB/s up and 17 GB/s down for 5 to 50 MB and
// 2.6 GB/s at 1 MB (390 us against 28 pinned), so a copy of any size goes
// through the ring, a chunk's memcpy beside the chunks on the link.  A chunk is
// moved by a kernel that reads or writes the pinned memory itself: the copy
// engine with an event per chunk leaves the link idle between chunks (15 MB
// down 716 us against 517, up 724 against 444, one thread).  Large copies are
// shared by threads: the memcpy out of memory that the device has written runs
// at 26 GB/s per thread, and result arrays are often fresh pages, whose faults
// (0.28 ms per MB in 4 KB pages, 0.1 in huge ones) are the memcpy's.  What the
// ring gains least in is 6 to 20 MB up with nothing else between (11.7 MB 413 us,
// 372 by the runtime; 422 and 518 with an operator application between).
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>

namespace t3x {

class HostStage {
 public:
  // Both are ordered on `s`, which is the same in every call of one object.
  // to_device returns when `src` may be changed or freed (its last chunks may
  // still be on the link), to_host when `dst` is written.
  hipError_t to_device(void* dst, const void* src, size_t bytes, hipStream_t s);
  hipError_t to_host(void* dst, const void* src, size_t bytes, hipStream_t s);
  // The caller has waited for the stream (as the last thing before it goes).
  void drained() {
    busy_ = false;
    used_ = 0;
  }
  ~HostStage();
  HostStage() = default;
  HostStage(const HostStage&) = delete;
  HostStage& operator=(const HostStage&) = delete;

 private:
  static constexpr size_t kMinRing = 256 << 10, kMaxRing = 16 << 20;  // pinned bytes: by the largest copy so far
  static constexpr int kMaxSlots = 32, kMaxThreads = 8;
  // A chunk costs the link 6 us beside its bytes (a kernel's start and end) and
  // the copy one chunk's memcpy; a thread 20 us to start.  15 MB down with 4
  // threads: 570, 450, 400 us in chunks of 256, 512, 1024 KB; 5 MB with one
  // thread 207, 167, 207.
  static size_t chunk_of(size_t bytes) {
    return bytes <= kMinRing ? kMinRing : bytes < (8u << 20) ? 512 << 10 : bytes < (32u << 20) ? 1 << 20 : 2 << 20;
  }
  // (7.0 and 8.2 MB up 307 and 389 us with one thread, 264 and 305 with two; 4.9 MB
  // 185 and 198)
  static int threads_of(size_t bytes) {
    return bytes < (5u << 20) ? 1 : bytes < (8u << 20) ? 2 : bytes < (64u << 20) ? 4 : kMaxThreads;
  }
  bool reserve(size_t bytes, hipStream_t s);
  hipError_t record(int slot, hipStream_t s);  // the slot's event, made when first used
  hipError_t drain(hipStream_t s);
  hipError_t put(char* dev, const char* host, size_t bytes, hipStream_t s);
  hipError_t get(char* dev, char* host, size_t bytes, hipStream_t s);
  hipError_t move(char* dev, char* host, size_t bytes, bool up, hipStream_t s);
  hipError_t issue(struct StageJob& job, size_t c);
  hipError_t part(struct StageJob& job);
  char* ring_ = nullptr;  // lent by the process's pool of rings
  size_t ringBytes_ = 0;
  int device_ = 0;  // where it was made
  hipEvent_t ev_[kMaxSlots] = {};
  // What may still be reading the ring: an upload of several chunks, ended by
  // ev_[last_], or small ones in its first used_ bytes.
  bool busy_ = false;
  int last_ = 0;
  size_t used_ = 0;
  bool failed_ = false;  // no pinned memory: the runtime's own path
};

}  // namespace t3x
