/*
 * rhip_ring.h -- the host side of reads (rhip_read.hip): pieces of device memory
 * arrive in a ring of pinned slots and are copied out while the next ones arrive,
 * by the calling thread for a small read, by helper threads for a large one.
 * What puts a piece into a slot is the caller's; only HIP's host functions are
 * called here.
 */
#pragma once
#include <hip/hip_runtime_api.h>
#include <stdint.h>

#include <algorithm>
#include <atomic>
#include <condition_variable>
#include <cstring>
#include <exception>
#include <memory>
#include <mutex>
#include <thread>
#include <vector>

#include "rhip.h"

namespace rhip {

int fail(int code, const char *fmt, ...) __attribute__((format(printf, 2, 3)));

/* Measured with reads of 64 KiB to 31.6 MiB, us:
 *   pieces   256 KiB: 1 MiB 52, 8 MiB 307, 31.6 MiB 1,240; 512 KiB: 54, 242, 890; 1 MiB: 68, 234, 767; 2 MiB: 67, 252, 733
 *   slots    8, 16 and 32 alike at every size; 16 are as many as a full HD image has pieces, twice
 *   helpers  1: 8 MiB 271, 31.6 MiB 1,030; 2: 226, 764 to 814; 3: 234, 767; 5: 235, 769
 *   line     with the helpers (from the first byte) 1 MiB 81, 2 MiB 100, 3 MiB 124, 4 MiB 145; without 67, 104, 143, 183 */
constexpr size_t kSlotBytes = (size_t)1 << 20;
constexpr int kSlots = 16;
constexpr int kHelpers = 3;
constexpr size_t kParallelBytes = (size_t)2 << 20; /* larger reads are copied out by the helpers */
/* Reads up to here take a ring of one slot of this size: a program that reads a few numbers or thumbnails pins 260 KiB and
 * not 16 MiB (its first read takes about the same, 45 us; one that also reads larger images pays 35 us for the second ring). */
constexpr size_t kSmallBytes = (size_t)256 << 10;
constexpr int kRingErrors = 4;                     /* the device's error words come along with the first piece */
constexpr int kNoPinned = 1;                       /* readPieces: pinned memory was refused, nothing was queued */

/* ------------------------------------------------------------------ pinned rings
 * One per read in progress, shared by the process's devices: a read takes a
 * free one or makes one; they are freed with the last device. */
struct Ring {
  int hip_device = 0; /* its events belong to this GPU */
  int count = 0;      /* slots */
  size_t slot_bytes = 0;
  char *slots = nullptr; /* the slots, then the error words */
  hipEvent_t ev[kSlots] = {};
  uint32_t *errors() const { return (uint32_t *)(slots + count * slot_bytes); }
  /* false where pinned memory or an event is refused (its error is not left for a later call to report) */
  bool make() {
    bool ok = hipHostMalloc((void **)&slots, count * slot_bytes + 4096, hipHostMallocDefault) == hipSuccess;
    if (!ok) slots = nullptr;
    for (int i = 0; i < count && ok; i++) ok = hipEventCreateWithFlags(&ev[i], hipEventDisableTiming) == hipSuccess;
    if (!ok) (void)hipGetLastError();
    return ok;
  }
  ~Ring() {
    for (hipEvent_t e : ev)
      if (e) (void)hipEventDestroy(e);
    if (slots) (void)hipHostFree(slots);
  }
};

/* ------------------------------------------------------------------ helper threads
 * They copy pieces to the caller's buffer as these arrive, beside the calling
 * thread. One read at a time has them; another that runs meanwhile copies on
 * its own thread. */
struct Copiers {
  std::mutex owner; /* held by the read that uses the helpers */
  std::mutex m;     /* job, open, quit, active */
  std::condition_variable wake, rest;
  std::vector<std::thread> threads;
  long long job = 0;
  int active = 0;
  bool open = false, quit = false;
  /* the job: changed only while it is not open and no helper is active */
  const char *slots = nullptr;
  char *out = nullptr;
  size_t bytes = 0;
  int pieces = 0;
  std::atomic<int> next{0}, ready{0};
  std::atomic<int> copied[kSlots]; /* per slot: the last piece copied out of it */
  std::atomic<bool> stop{false};

  /* copies pieces until none is left */
  void work() {
    for (;;) {
      const int c = next.fetch_add(1);
      if (c >= pieces) return;
      while (ready.load(std::memory_order_acquire) <= c) {
        if (stop.load(std::memory_order_relaxed)) return;
        std::this_thread::yield();
      }
      const size_t at = (size_t)c * kSlotBytes;
      memcpy(out + at, slots + (size_t)(c % kSlots) * kSlotBytes, std::min(kSlotBytes, bytes - at));
      copied[c % kSlots].store(c, std::memory_order_release);
    }
  }
  void run() {
    long long seen = 0;
    std::unique_lock<std::mutex> l(m);
    for (;;) {
      wake.wait(l, [&] { return quit || (open && job != seen); });
      if (quit) return;
      seen = job;
      active++;
      l.unlock();
      work();
      l.lock();
      if (--active == 0) rest.notify_all();
    }
  }
  void start(const char *slots_, void *out_, size_t bytes_, int pieces_) {
    {
      std::lock_guard<std::mutex> l(m);
      slots = slots_;
      out = (char *)out_;
      bytes = bytes_;
      pieces = pieces_;
      next = ready = 0;
      stop = false;
      for (auto &c : copied) c = -1;
      job++;
      open = true;
    }
    wake.notify_all();
  }
  /* no helper joins any more; returns when the last one is out */
  void finish() {
    std::unique_lock<std::mutex> l(m);
    open = false;
    rest.wait(l, [&] { return active == 0; });
  }
};

constexpr int kKeptRings = 4; /* of either size: 65 MiB of pinned memory at most */
struct Shared {
  std::mutex m;
  std::vector<std::unique_ptr<Ring>> free_rings;
  std::unique_ptr<Copiers> copiers;
  int devices = 0;
  Shared() { free_rings.reserve(2 * kKeptRings); } /* giving a ring back allocates nothing */
};
/* never destroyed: a process may end with devices alive and helpers asleep */
inline Shared &shared() {
  static Shared *s = new Shared();
  return *s;
}

struct RingLease {
  std::unique_ptr<Ring> r;
  bool take(int hip_device, bool small) {
    const int count = small ? 1 : kSlots;
    Shared &s = shared();
    {
      std::lock_guard<std::mutex> l(s.m);
      for (auto &f : s.free_rings)
        if (f->hip_device == hip_device && f->count == count) {
          r = std::move(f);
          f = std::move(s.free_rings.back());
          s.free_rings.pop_back();
          return true;
        }
    }
    r.reset(new Ring());
    r->hip_device = hip_device;
    r->count = count;
    r->slot_bytes = small ? kSmallBytes : kSlotBytes;
    if (!r->make()) r.reset(); /* half made: not for another read */
    return r != nullptr;
  }
  ~RingLease() {
    if (!r) return;
    Shared &s = shared();
    std::lock_guard<std::mutex> l(s.m);
    const auto same = [&](const std::unique_ptr<Ring> &f) { return f->count == r->count; };
    if (s.devices > 0 && std::count_if(s.free_rings.begin(), s.free_rings.end(), same) < kKeptRings)
      s.free_rings.push_back(std::move(r));
  }
};

/* The helpers, started on first use. Null where the host has no cores to spare, starts no thread or has no memory for
 * them: a read that has queued its pieces goes on without them, so nothing may be thrown here. */
inline Copiers *copiers() noexcept {
  Shared &s = shared();
  std::lock_guard<std::mutex> l(s.m);
  if (!s.copiers) {
    const int n = std::min(kHelpers, (int)std::thread::hardware_concurrency() / 2);
    std::unique_ptr<Copiers> c;
    try {
      c.reset(new Copiers());
      c->threads.reserve(n); /* before any thread is: one that runs must not be dropped */
      for (int i = 0; i < n; i++) c->threads.emplace_back([q = c.get()] { q->run(); });
    } catch (const std::exception &) {
    }
    if (!c || c->threads.empty()) return nullptr;
    s.copiers = std::move(c);
  }
  return s.copiers.get();
}

/* `bytes` bytes of device memory to out, piece by piece: issue(at, n, slot, errors) queues on `stream` what puts bytes
 * [at, at + n) into a slot, and the device's error words to `errors` where that is not null. `errors` (kRingErrors
 * words, may be null) gets those. kNoPinned where no ring is to be had. */
template <typename Issue>
int readPieces(int hip_device, hipStream_t stream, size_t bytes, void *out, uint32_t *errors, Issue issue_piece) {
  RingLease lease;
  if (!lease.take(hip_device, bytes <= kSmallBytes)) return kNoPinned;
  Ring &R = *lease.r;
  const int pieces = (int)((bytes + kSlotBytes - 1) / kSlotBytes); /* of a small read: one */
  if (errors) memset(errors, 0, kRingErrors * 4);
  if (!pieces) return RHIP_OK;
  hipError_t he = hipSuccess;
  int issued = 0;
  auto issue = [&]() {
    const size_t at = (size_t)issued * kSlotBytes;
    const int slot = issued % kSlots;
    he = issue_piece(at, std::min(kSlotBytes, bytes - at), R.slots + slot * kSlotBytes,
                     errors && issued == 0 ? R.errors() : nullptr);
    if (he == hipSuccess) he = hipEventRecord(R.ev[slot], stream);
    if (he == hipSuccess) issued++;
  };
  /* the ring may be reused or freed only once nothing on the stream writes it */
  auto give_up = [&]() {
    (void)hipStreamSynchronize(stream);
    return fail(RHIP_E_HIP, "read: %s", hipGetErrorString(he));
  };
  while (issued < std::min(pieces, kSlots) && he == hipSuccess) issue();
  if (he != hipSuccess) return give_up();

  /* the work queued before the read is waited for here, with the first piece, and only then are helpers woken: they never
   * spin through it */
  if ((he = hipEventSynchronize(R.ev[0])) != hipSuccess) return give_up();
  Copiers *C = bytes > kParallelBytes ? copiers() : nullptr;
  std::unique_lock<std::mutex> own;
  if (C) own = std::unique_lock<std::mutex>(C->owner, std::try_to_lock);
  if (!C || !own.owns_lock()) {
    for (int c = 0; c < pieces; c++) {
      if (c && (he = hipEventSynchronize(R.ev[c % kSlots])) != hipSuccess) return give_up();
      const size_t at = (size_t)c * kSlotBytes;
      memcpy((char *)out + at, R.slots + (size_t)(c % kSlots) * kSlotBytes, std::min(kSlotBytes, bytes - at));
      if (issued < pieces) {
        issue();
        if (he != hipSuccess) return give_up();
      }
    }
  } else {
    C->start(R.slots, out, bytes, pieces);
    for (int c = 0; c < pieces && he == hipSuccess; c++) {
      if (c) he = hipEventSynchronize(R.ev[c % kSlots]);
      if (he != hipSuccess) break;
      C->ready.store(c + 1, std::memory_order_release);
      /* half a ring ahead of the copies: piece p + kSlots goes into p's slot once p is out of it */
      while (issued < pieces && issued - kSlots <= c - kSlots / 2 && he == hipSuccess) {
        const int p = issued - kSlots;
        while (C->copied[p % kSlots].load(std::memory_order_acquire) != p) std::this_thread::yield();
        issue();
      }
    }
    if (he == hipSuccess)
      C->work();
    else
      C->stop = true;
    C->finish();
    if (he != hipSuccess) return give_up();
  }
  if (errors) memcpy(errors, R.errors(), kRingErrors * 4);
  return RHIP_OK;
}

/* A read without pinned memory: `words` words of device memory to out, and the device's error words. */
inline int readPageable(hipStream_t stream, const void *src, size_t words, void *out, const uint32_t *dev_errors,
                        uint32_t *errors) {
  hipError_t he = hipMemcpyAsync(out, src, words * 4, hipMemcpyDeviceToHost, stream);
  if (he == hipSuccess && errors)
    he = hipMemcpyAsync(errors, dev_errors, kRingErrors * 4, hipMemcpyDeviceToHost, stream);
  const hipError_t se = hipStreamSynchronize(stream);
  if (he == hipSuccess) he = se;
  return he == hipSuccess ? RHIP_OK : fail(RHIP_E_HIP, "read: %s", hipGetErrorString(he));
}

/* The same for an image of w x h texels stored in `stored` words, texel (x, y) at index(x, y). */
template <typename Index>
int readPageable(hipStream_t stream, const void *src, size_t stored, int w, int h, void *out, const uint32_t *dev_errors,
                 uint32_t *errors, Index index) {
  std::vector<uint32_t> tmp(stored);
  const int rc = readPageable(stream, src, stored, tmp.data(), dev_errors, errors);
  if (rc) return rc;
  uint32_t *o = (uint32_t *)out;
  for (int y = 0; y < h; y++)
    for (int x = 0; x < w; x++) *o++ = tmp[index(x, y)];
  return RHIP_OK;
}

/* What the reads share (pinned memory, helper threads) lives while the process has devices. */
inline void readDeviceAdded() {
  Shared &s = shared();
  std::lock_guard<std::mutex> l(s.m);
  s.devices++;
}

inline void readDeviceGone() {
  Shared &s = shared();
  std::vector<std::unique_ptr<Ring>> rings;
  std::unique_ptr<Copiers> c;
  {
    std::lock_guard<std::mutex> l(s.m);
    if (--s.devices > 0) return;
    rings.swap(s.free_rings);
    c = std::move(s.copiers);
  }
  if (c) {
    {
      std::lock_guard<std::mutex> l(c->m);
      c->quit = true;
    }
    c->wake.notify_all();
    for (std::thread &t : c->threads) t.join();
  }
}

}  // namespace rhip
