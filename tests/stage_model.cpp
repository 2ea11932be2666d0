// HostStage (t3x_stage.hip) on the CPU: exit status 0 if every check holds.
#include <hip/hip_runtime.h>

#include <cstdio>
#include <new>

#include "../top3d_xl_amd/csrc/t3x_stage.hip"

void* operator new(size_t n) {
  if (model::newsLeft >= 0 && model::newsLeft-- == 0) throw std::bad_alloc();
  if (void* p = std::malloc(n)) return p;
  throw std::bad_alloc();
}
void operator delete(void* p) noexcept { std::free(p); }
void operator delete(void* p, size_t) noexcept { std::free(p); }

using namespace t3x;

static int bad = 0;
static void check(bool ok, const char* what, size_t n) {
  if (!ok) std::printf("wrong: %s, %zu\n", what, n), ++bad;
}
static std::vector<char> pattern(size_t n, unsigned seed) {
  std::vector<char> v(n);
  for (size_t i = 0; i < n; ++i) v[i] = (char)((i * 2654435761u + seed) >> 13);
  return v;
}
// n bytes up and back, the source overwritten as soon as the call returns
static bool round_trip(HostStage& S, hipStream_t s, size_t n, unsigned seed) {
  std::vector<char> src = pattern(n, seed), dev(n + 16), out(n, 1);
  char* d = dev.data() + (16 - (uintptr_t)dev.data() % 16) % 16;
  if (S.to_device(d, src.data(), n, s) != hipSuccess) return false;
  std::fill(src.begin(), src.end(), 7);
  if (S.to_host(out.data(), d, n, s) != hipSuccess) return false;
  return out == pattern(n, seed);
}

// memory for a thread's start runs out: the threads that run take all chunks
static void no_more_threads() {
  ModelStream s;
  for (int left : {0, 1, 2, 5}) {
    HostStage S;
    for (size_t n : {(size_t)9 << 20, ((size_t)65 << 20) + 40}) {
      std::vector<char> src = pattern(n, 3), dev(n), out(n);
      char* d = dev.data();  // (malloc'ed: 16-byte aligned)
      model::newsLeft = left;
      const hipError_t a = S.to_device(d, src.data(), n, &s);
      model::newsLeft = left;
      const hipError_t b = S.to_host(out.data(), d, n, &s);
      model::newsLeft = -1;
      check(a == hipSuccess && b == hipSuccess && out == src, "a copy without its threads", n);
    }
  }
}

// rings outlive their objects, few of them, and serve the next one's stream
static void rings_serve_on() {
  const size_t n = (5 << 20) + 24;
  int made = 0;
  for (int i = 0; i < 6; ++i) {  // handles of one model, one after the other
    ModelStream s;
    HostStage S;
    check(round_trip(S, &s, 1000, i) && round_trip(S, &s, n, i), "a handle's copies", n);
    if (i == 0) made = model::pinnedCalls;
  }
  check(model::pinnedCalls == made, "rings made for handles after the first", model::pinnedCalls - made);
  {  // another device's handle
    ModelStream s;
    HostStage S;
    hipSetDevice(1);
    check(round_trip(S, &s, n, 9), "another device", n);
    hipSetDevice(0);
    check(model::pinnedCalls > made, "another device's ring", n);
  }
  std::vector<std::thread> t;  // many handles at once, each an upload in flight when it is closed
  std::atomic<int> wrong{0};
  for (int k = 0; k < 12; ++k)
    t.emplace_back([&, k] {
      for (int i = 0; i < 8; ++i) {
        ModelStream s;
        std::vector<char> last = pattern(70000 + 4000 * k, i), dev(last.size());
        {
          HostStage S;
          for (size_t m : {(size_t)4096, (size_t)300000 * (k + 1), (size_t)70000 * (i + 1) + 8})
            wrong += !round_trip(S, &s, m, 31 * k + i);
          wrong += S.to_device(dev.data(), last.data(), last.size(), &s) != hipSuccess;
        }
        (void)hipStreamSynchronize(&s);
        wrong += dev != last;
      }
    });
  for (auto& x : t) x.join();
  check(wrong == 0, "copies of handles at once", wrong);
  check(model::pinnedNow <= 4, "rings kept", model::pinnedNow);
}

// every number of threads, below, at and above each line, and the ring's slots
// used again: with all of it, and with a ring that could not grow
static void every_form() {
  for (size_t limit : {(size_t)256 << 10, (size_t)1 << 20, ~(size_t)0}) {
    model::pinnedLimit = limit;
    const int made = model::pinnedNow;
    ModelStream s;
    HostStage S;
    const size_t first = min(limit, (size_t)16 << 20);  // the ring is as large as it will be from the start
    check(round_trip(S, &s, first, 1) && model::pinnedNow == made + 1, "a ring of this size", first);
    check(round_trip(S, &s, 1, 1), "one byte", 1);
    for (size_t mb : {5, 8, 32, 64})
      for (size_t n : {(mb << 20) - 8, mb << 20, (mb << 20) + 4099}) check(round_trip(S, &s, n, (unsigned)n), "a copy", n);
    for (size_t n : {(size_t)262144, (size_t)262152, (size_t)3000001}) check(round_trip(S, &s, n, (unsigned)n), "a copy", n);
  }
  model::pinnedLimit = ~(size_t)0;
}
// a launch that fails ends the copy with its error, and the next one is whole
static void errors() {
  ModelStream s;
  HostStage S;
  for (size_t n : {(size_t)1000, (size_t)3 << 20, (size_t)20 << 20})
    for (int k : {0, 1, 5}) {
      std::vector<char> src = pattern(n, 2), dev(n);
      model::launchesUntilError = k;
      const hipError_t a = S.to_device(dev.data(), src.data(), n, &s);
      const hipError_t b = a == hipSuccess ? S.to_host(src.data(), dev.data(), n, &s) : hipSuccess;
      const bool hit = model::launchesUntilError < 0;
      model::launchesUntilError = -1;
      check(!hit || a != hipSuccess || b != hipSuccess, "an error reported", n);
      check(round_trip(S, &s, n, 4), "a copy after an error", n);
    }
}

// small copies follow each other through the ring, each source overwritten at
// once, with no event of their own; larger ones between them
static void small_copies() {
  ModelStream s;
  HostStage S;
  const size_t n = 4100, many = 200;
  std::vector<std::vector<char>> dev(many, std::vector<char>(n));
  const int before = model::eventsRecorded;
  int events = 0;
  for (size_t i = 0; i < many; ++i) {
    std::vector<char> src = pattern(n, (unsigned)i), back(n);
    check(S.to_device(dev[i].data(), src.data(), n, &s) == hipSuccess, "a small upload", i);
    std::fill(src.begin(), src.end(), 5);
    if (i % 70 == 30)
      check(S.to_host(back.data(), dev[i - 9].data(), n, &s) == hipSuccess && back == pattern(n, i - 9), "a small result", i);
    if (i == 90) events = model::eventsRecorded;
    if (i == 149) check(round_trip(S, &s, 3 << 20, 1), "a large copy among small ones", i);
  }
  check(events == before, "events behind small copies", events - before);
  (void)hipStreamSynchronize(&s);
  for (size_t i = 0; i < many; ++i) check(dev[i] == pattern(n, (unsigned)i), "a small upload's bytes", i);
}

int main() {
  every_form();  // first: no larger ring is there to be lent
  rings_serve_on();
  errors();
  small_copies();
  no_more_threads();
  check(model::pinnedNow <= 4 && model::eventsNow == 0, "all given back", model::pinnedNow);
  return bad != 0;
}
