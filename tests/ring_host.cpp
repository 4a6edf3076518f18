/*
 * The host side of reads (rhip_ring.h) on a stream made of one thread, without a GPU: pieces are written into their
 * slots when the stream gets to them (or as soon as they are queued: a GPU that is far ahead of the copies), events
 * complete in order, and allocations can be told to fail.
 * Usage: ring_host <check>; prints "ok" and returns 0, or says what differed.
 */
#include <dlfcn.h>
#include <errno.h>
#include <pthread.h>

#include <chrono>
#include <cstdarg>
#include <cstdio>
#include <cstdlib>
#include <ctime>
#include <deque>
#include <functional>
#include <new>
#include <string>

#include "rhip_ring.h"

/* ------------------------------------------------------------------ the stream */

namespace {

struct FakeStream {
  std::mutex m;
  std::condition_variable cv;
  std::deque<std::function<void()>> tasks;
  long long queued = 0, done = 0;
  bool at_once = false;
  FakeStream() { std::thread([this] { run(); }).detach(); }
  void run() {
    std::unique_lock<std::mutex> l(m);
    for (;;) {
      cv.wait(l, [&] { return !tasks.empty(); });
      auto t = tasks.front();
      tasks.pop_front();
      l.unlock();
      t();
      l.lock();
      done++;
      cv.notify_all();
    }
  }
  void push(std::function<void()> t) {
    if (at_once) return t();
    std::lock_guard<std::mutex> l(m);
    tasks.push_back(std::move(t));
    queued++;
    cv.notify_all();
  }
  void wait(long long n) {
    std::unique_lock<std::mutex> l(m);
    cv.wait(l, [&] { return done >= n; });
  }
};
FakeStream &stream() {
  static FakeStream *s = new FakeStream();
  return *s;
}
struct FakeEvent {
  long long at = 0;
};

size_t pinned_limit = (size_t)-1; /* larger allocations are refused */
hipError_t last_error = hipSuccess;
int events_left = 1 << 30; /* event creations that still succeed */
int pinned_blocks = 0;
size_t pinned_bytes = 0;

}  // namespace

extern "C" {
hipError_t hipHostMalloc(void **p, size_t n, unsigned int) {
  if (n > pinned_limit) return last_error = hipErrorOutOfMemory;
  pinned_blocks++;
  pinned_bytes += n;
  return (*p = malloc(n)) ? hipSuccess : hipErrorOutOfMemory;
}
hipError_t hipHostFree(void *p) {
  pinned_blocks--;
  free(p);
  return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) {
  if (events_left-- <= 0) return last_error = hipErrorOutOfMemory;
  *e = (hipEvent_t) new FakeEvent();
  return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t e) {
  delete (FakeEvent *)e;
  return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t e, hipStream_t) {
  if (!e) return hipErrorInvalidHandle;
  FakeStream &s = stream();
  std::lock_guard<std::mutex> l(s.m);
  ((FakeEvent *)e)->at = s.queued;
  return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t e) {
  stream().wait(((FakeEvent *)e)->at);
  return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) {
  long long n;
  {
    std::lock_guard<std::mutex> l(stream().m);
    n = stream().queued;
  }
  stream().wait(n);
  return hipSuccess;
}
hipError_t hipGetLastError() {
  const hipError_t e = last_error;
  last_error = hipSuccess;
  return e;
}
hipError_t hipMemcpyAsync(void *to, const void *from, size_t n, hipMemcpyKind, hipStream_t) {
  stream().push([=] { memcpy(to, from, n); });
  return hipSuccess;
}
const char *hipGetErrorString(hipError_t) { return "error"; }
}

/* ------------------------------------------------------------------ refused memory and threads */

namespace {
thread_local int news_left = 1 << 30; /* allocations of this thread that still succeed */
int threads_left = 1 << 30;           /* threads that can still be started */
}  // namespace
void *operator new(size_t n) {
  if (news_left-- <= 0) throw std::bad_alloc();
  if (void *p = malloc(n)) return p;
  throw std::bad_alloc();
}
void operator delete(void *p) noexcept { free(p); }
void operator delete(void *p, size_t) noexcept { free(p); }
extern "C" int pthread_create(pthread_t *t, const pthread_attr_t *a, void *(*f)(void *), void *arg) {
  if (threads_left-- <= 0) return EAGAIN;
  static auto real = (decltype(&pthread_create))dlsym(RTLD_NEXT, "pthread_create");
  return real(t, a, f, arg);
}

namespace rhip {
std::string message;
int fail(int code, const char *fmt, ...) {
  char b[256];
  va_list a;
  va_start(a, fmt);
  vsnprintf(b, sizeof b, fmt, a);
  va_end(a);
  message = b;
  return code;
}
}  // namespace rhip

using namespace rhip;

/* ------------------------------------------------------------------ checks */

namespace {

std::vector<char> device_memory(size_t n, uint32_t seed) {
  std::vector<char> v(n);
  uint32_t x = seed * 2654435761u + 1u;
  for (char &c : v) c = (char)((x = x * 1664525u + 1013904223u) >> 24);
  return v;
}

/* Reads n bytes; 0 when they and the error words arrive. */
int read(size_t n, uint32_t seed) {
  const std::vector<char> src = device_memory(n, seed);
  std::vector<char> out(n + 64, (char)0x5a);
  uint32_t err[kRingErrors] = {9, 9, 9, 9};
  int rc = readPieces(0, nullptr, n, out.data(), err, [&](size_t at, size_t bytes, char *slot, uint32_t *errors) {
    stream().push([=, &src] {
      memcpy(slot, src.data() + at, bytes);
      if (errors)
        for (int i = 0; i < kRingErrors; i++) errors[i] = seed + i;
    });
    return hipSuccess;
  });
  if (rc == kNoPinned) {
    const uint32_t dev_errors[kRingErrors] = {seed, seed + 1, seed + 2, seed + 3};
    rc = readPageable(nullptr, src.data(), n / 4, out.data(), dev_errors, err);
  }
  if (rc) {
    printf("%zu bytes: code %d, %s\n", n, rc, message.c_str());
    return 1;
  }
  if (memcmp(out.data(), src.data(), n)) {
    size_t at = 0;
    while (out[at] == src[at]) at++;
    printf("%zu bytes: differ from byte %zu on\n", n, at);
    return 1;
  }
  for (size_t i = n; i < out.size(); i++)
    if (out[i] != 0x5a) {
      printf("%zu bytes: written past the end\n", n);
      return 1;
    }
  for (int i = 0; i < kRingErrors; i++)
    if (err[i] != seed + i) {
      printf("%zu bytes: error word %d is %u\n", n, i, err[i]);
      return 1;
    }
  return 0;
}

/* Sizes about the pieces, the line to the helpers and the ring's end, and rings walked several times, with the helper
 * threads and without them, the stream slower and faster than the copies. */
int checkBytes() {
  const size_t K = kSlotBytes;
  const size_t sizes[] = {4,     64,    kSmallBytes, kSmallBytes + 4, K - 4,           K,          K + 4, kParallelBytes, kParallelBytes + 4, 15 * K + 8, kSlots * K,
                          kSlots * K + 4, 17 * K, 2 * kSlots * K + 12, 53 * K + 4};
  int bad = 0;
  for (int own = 0; own < 2; own++) {
    std::unique_lock<std::mutex> held;
    std::thread other;
    std::mutex hold;
    std::atomic<bool> taken{false};
    hold.lock();
    Copiers *c = copiers();
    if (own && c) { /* another read has the helpers */
      other = std::thread([&] {
        std::lock_guard<std::mutex> l(c->owner);
        taken = true;
        std::lock_guard<std::mutex> until(hold);
      });
      while (!taken) std::this_thread::yield();
    }
    uint32_t seed = 1;
    for (int fast = 0; fast < 2; fast++) {
      stream().at_once = fast;
      for (size_t n : sizes) bad += read(n, seed++);
      stream().at_once = false;
    }
    hold.unlock();
    if (other.joinable()) other.join();
  }
  return bad;
}

/* A read that could not make its ring leaves nothing behind for the next one. */
int checkEvents() {
  for (int k = 0; k < kSlots; k += 5) {
    events_left = k;
    std::vector<char> out(2 * kSlotBytes);
    (void)readPieces(0, nullptr, out.size(), out.data(), nullptr, [&](size_t, size_t, char *, uint32_t *) { return hipSuccess; });
    events_left = 1 << 30;
    if (pinned_blocks) {
      printf("%d pinned blocks kept of a ring without its events\n", pinned_blocks);
      return 1;
    }
    if (read(5 * kSlotBytes, 3)) return 1;
    readDeviceGone(); /* the good ring too */
    readDeviceAdded();
  }
  return 0;
}

/* While the stream still works on what was queued before the read, nothing of the read takes processor time. */
int checkIdle() {
  bool helpers = copiers() != nullptr;
  for (int k = 0; k < 2; k++) {
    stream().push([] { std::this_thread::sleep_for(std::chrono::milliseconds(400)); });
    const size_t n = 8 * kSlotBytes;
    const std::vector<char> src = device_memory(n, 1);
    std::vector<char> out(n);
    const clock_t c0 = clock(); /* of all threads */
    const int rc = readPieces(0, nullptr, n, out.data(), nullptr, [&](size_t at, size_t bytes, char *slot, uint32_t *) {
      stream().push([=, &src] { memcpy(slot, src.data() + at, bytes); });
      return hipSuccess;
    });
    const double ms = (clock() - c0) * 1e3 / CLOCKS_PER_SEC;
    if (rc || out != src) return 1;
    if (ms > 200) { /* 16 MiB copied: a few; one thread that spins: 400 */
      printf("%.0f ms of processor time in a read that waited 400 ms (helpers: %d)\n", ms, (int)helpers);
      return 1;
    }
  }
  return 0;
}

/* Where pinned memory is refused, reads copy through pageable memory, every layout, and leave no error behind; a small
 * read asks for little of it. */
int checkRefused() {
  if (read(64, 1)) return 1;
  if (pinned_bytes > 512 << 10) {
    printf("%zu bytes pinned for a read of 64\n", pinned_bytes);
    return 1;
  }
  readDeviceGone();
  readDeviceAdded();
  for (size_t limit : {(size_t)0, (size_t)1 << 20}) {
    pinned_limit = limit;
    for (size_t n : {(size_t)4, (size_t)64, kSlotBytes + 4, 5 * kSlotBytes})
      if (read(n, (uint32_t)n)) return 1;
    if (last_error != hipSuccess) {
      printf("the refused allocation's error is left for the next call\n");
      return 1;
    }
  }
  /* a 6 x 5 image stored column by column, with a column of padding */
  const uint32_t stored[35] = {0,  1,  2,  3,  4,  5,  6,  7,  8,  9,  10, 11, 12, 13, 14, 15, 16, 17,
                               18, 19, 20, 21, 22, 23, 24, 25, 26, 27, 28, 29, 30, 31, 32, 33, 34};
  const uint32_t dev_errors[kRingErrors] = {4, 3, 2, 1};
  uint32_t out[31], errors[kRingErrors];
  out[30] = 77;
  if (readPageable(nullptr, stored, 35, 6, 5, out, dev_errors, errors, [](int x, int y) { return (size_t)x * 5 + y; }))
    return 1;
  for (int i = 0; i < 30; i++)
    if (out[i] != (uint32_t)(i % 6 * 5 + i / 6)) return printf("pageable: texel %d is %u\n", i, out[i]), 1;
  return out[30] != 77 || memcmp(errors, dev_errors, sizeof errors);
}

/* Helpers that cannot be started, or not all, change no read and throw nothing. */
int checkHelpers() {
  if (read(64, 1)) return 1; /* the stream's own thread runs */
  for (int k = 0; k < 6; k++) {
    news_left = k;
    Copiers *c = copiers();
    news_left = 1 << 30;
    if (k == 0 && c) return printf("helpers without memory\n"), 1;
    if (read(20 * kSlotBytes, 10 + k)) return 1;
    readDeviceGone();
    readDeviceAdded();
  }
  for (int k = 0; k < kHelpers; k++) {
    threads_left = k;
    const int bad = read(20 * kSlotBytes + 4, 20 + k);
    threads_left = 1 << 30;
    if (bad) return 1;
    readDeviceGone();
    readDeviceAdded();
  }
  return 0;
}

}  // namespace

int main(int argc, char **argv) {
  const std::string what = argc > 1 ? argv[1] : "";
  readDeviceAdded();
  int bad = 1;
  if (what == "bytes") bad = checkBytes();
  if (what == "events") bad = checkEvents();
  if (what == "idle") bad = checkIdle();
  if (what == "refused") bad = checkRefused();
  if (what == "helpers") bad = checkHelpers();
  readDeviceGone();
  if (!bad && pinned_blocks) {
    printf("%d pinned blocks left\n", pinned_blocks);
    bad = 1;
  }
  if (!bad) printf("ok\n");
  return bad ? 1 : 0;
}
