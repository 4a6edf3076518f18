/*
 * rhip_read.hip -- results back to host memory.
 *
 * A read is bound by PCIe (56 GB/s into pinned memory here) only if nothing
 * else is in its way: hipMemcpy into pageable memory stages the copy and moves
 * it to the caller's buffer on one thread, one piece after the other (17 GB/s),
 * and images in a tiled layout, or simply not multisampled, were copied again
 * texel by texel. Here a kernel puts 1 MiB pieces of the image, in row order,
 * into a ring of pinned slots, and the pieces are copied out while the next
 * ones arrive: by the calling thread for a small read, by helper threads for a
 * large one. The device's error words come along with the first piece.
 * An 8.3 MB image took 500 us (now 233), a 33 MB one 1,860 us (780), 48 images of
 * 64 KiB to 1 MiB 5.9 ms (1.8).
 */
#include <hip/hip_runtime.h>

#include <atomic>
#include <condition_variable>
#include <cstring>
#include <mutex>
#include <system_error>
#include <thread>

#include "rhip_host.h"
#include "rhip_kernels.h"

namespace rhip {

namespace {

constexpr size_t kSlotBytes = (size_t)1 << 20;
constexpr int kSlots = 16;
constexpr size_t kParallelBytes = (size_t)2 << 20; /* larger reads are copied out by the helpers */

/* ------------------------------------------------------------------ pinned rings
 * One per read in progress, shared by the process's devices: a read takes a
 * free one or makes one; they are freed with the last device. */
struct Ring {
  int hip_device = 0;    /* its events belong to this GPU */
  char *slots = nullptr; /* kSlots x kSlotBytes, then the error words */
  hipEvent_t ev[kSlots] = {};
  uint32_t *errors() const { return (uint32_t *)(slots + kSlots * kSlotBytes); }
  int make() {
    if (hipHostMalloc((void **)&slots, kSlots * kSlotBytes + 4096, hipHostMallocDefault) != hipSuccess) {
      slots = nullptr;
      return fail(RHIP_E_OOM, "pinned memory for reads");
    }
    for (hipEvent_t &e : ev)
      if (hipEventCreateWithFlags(&e, hipEventDisableTiming) != hipSuccess) return fail(RHIP_E_HIP, "read events");
    return RHIP_OK;
  }
  ~Ring() {
    for (hipEvent_t e : ev)
      if (e) hipEventDestroy(e);
    if (slots) hipHostFree(slots);
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

struct Shared {
  std::mutex m;
  std::vector<std::unique_ptr<Ring>> free_rings;
  std::unique_ptr<Copiers> copiers;
  int devices = 0;
};
/* never destroyed: a process may end with devices alive and helpers asleep */
Shared &shared() {
  static Shared *s = new Shared();
  return *s;
}

struct RingLease {
  std::unique_ptr<Ring> r;
  int take(int hip_device) {
    Shared &s = shared();
    {
      std::lock_guard<std::mutex> l(s.m);
      for (auto &f : s.free_rings)
        if (f->hip_device == hip_device) {
          r = std::move(f);
          f = std::move(s.free_rings.back());
          s.free_rings.pop_back();
          return RHIP_OK;
        }
    }
    r.reset(new Ring());
    r->hip_device = hip_device;
    return r->make();
  }
  ~RingLease() {
    if (!r || !r->slots) return;
    Shared &s = shared();
    std::lock_guard<std::mutex> l(s.m);
    if (s.devices > 0 && s.free_rings.size() < 4) s.free_rings.push_back(std::move(r));
  }
};

/* The helpers, started on first use (null where the host has no cores to spare or starts no thread). */
Copiers *copiers() {
  Shared &s = shared();
  std::lock_guard<std::mutex> l(s.m);
  if (!s.copiers) {
    const int n = std::min(3, (int)std::thread::hardware_concurrency() / 2);
    std::unique_ptr<Copiers> c(new Copiers());
    try {
      for (int i = 0; i < n; i++) c->threads.emplace_back([q = c.get()] { q->run(); });
    } catch (const std::system_error &) {
    }
    if (c->threads.empty()) return nullptr;
    s.copiers = std::move(c);
  }
  return s.copiers.get();
}

/* ------------------------------------------------------------------ device side */

/* Words [w0, w0 + n) of a level's row-major image (w wide, stored in `layout`)
 * to dst; with `errors`, the device's error words too. */
__global__ __launch_bounds__(256) void k_read_words(const uint32_t *src, TexLevel lv, int layout, size_t w0, size_t n,
                                                    uint32_t *dst, const uint32_t *errors, uint32_t *errors_out) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x, stride = (size_t)gridDim.x * blockDim.x;
  if (errors && i < kErrSlots) errors_out[i] = errors[i];
  if (layout == LAYOUT_LINEAR) {
    /* both sides 16-byte aligned: levels start at multiples of 256 bytes, pieces at multiples of 1 MiB */
    const uint4 *s4 = (const uint4 *)(src + w0);
    for (size_t j = i; j < n / 4; j += stride) ((uint4 *)dst)[j] = s4[j];
    for (size_t j = (n & ~(size_t)3) + i; j < n; j += stride) dst[j] = src[w0 + j];
  } else {
    for (size_t j = i; j < n; j += stride) {
      const uint32_t k = (uint32_t)(w0 + j), y = k / (uint32_t)lv.w, x = k - y * (uint32_t)lv.w;
      dst[j] = src[colPart(lv, layout, x) + rowPart(lv, layout, y)];
    }
  }
}

/* `words` words from src (a level when lv is given) to out. */
int readWords(rhip_device d, const void *src, const TexLevel *lv, int layout, size_t words, void *out,
              uint32_t *errors) {
  RingLease lease;
  int rc = lease.take(d->hip_device);
  if (rc) return rc;
  Ring &R = *lease.r;
  const size_t bytes = words * 4, slot_words = kSlotBytes / 4;
  const int pieces = (int)((words + slot_words - 1) / slot_words);
  if (errors) memset(errors, 0, kErrSlots * 4);
  if (!pieces) return RHIP_OK;
  const TexLevel none{};
  hipError_t he = hipSuccess;
  int issued = 0;
  auto issue = [&]() {
    const size_t w0 = (size_t)issued * slot_words, n = std::min(slot_words, words - w0);
    const int slot = issued % kSlots;
    const unsigned grid = std::max(1u, std::min(blocks(n, 1024), 256u));
    k_read_words<<<grid, 256, 0, d->stream>>>((const uint32_t *)src, lv ? *lv : none, layout, w0, n,
                                              (uint32_t *)(R.slots + slot * kSlotBytes),
                                              errors && issued == 0 ? d->errors : nullptr, R.errors());
    he = hipGetLastError();
    if (he == hipSuccess) he = hipEventRecord(R.ev[slot], d->stream);
    if (he == hipSuccess) issued++;
  };
  /* the ring may be reused or freed only once nothing on the stream writes it */
  auto give_up = [&]() {
    hipStreamSynchronize(d->stream);
    return fail(RHIP_E_HIP, "read: %s", hipGetErrorString(he));
  };
  while (issued < std::min(pieces, kSlots) && he == hipSuccess) issue();
  if (he != hipSuccess) return give_up();

  Copiers *C = bytes > kParallelBytes ? copiers() : nullptr;
  std::unique_lock<std::mutex> own;
  if (C) own = std::unique_lock<std::mutex>(C->owner, std::try_to_lock);
  if (!C || !own.owns_lock()) {
    for (int c = 0; c < pieces; c++) {
      if ((he = hipEventSynchronize(R.ev[c % kSlots])) != hipSuccess) return give_up();
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
      he = hipEventSynchronize(R.ev[c % kSlots]);
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
  if (errors) memcpy(errors, R.errors(), kErrSlots * 4);
  return RHIP_OK;
}

}  // namespace

void readDeviceAdded() {
  Shared &s = shared();
  std::lock_guard<std::mutex> l(s.m);
  s.devices++;
}

void readDeviceGone() {
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

int readLevel(rhip_device d, const uint8_t *src, const TexLevel &lv, int layout, void *out, uint32_t *errors) {
  return readWords(d, src, &lv, layout, (size_t)lv.w * lv.h, out, errors);
}

int readLinear(rhip_device d, const void *src, size_t words, void *out, uint32_t *errors) {
  return readWords(d, src, nullptr, LAYOUT_LINEAR, words, out, errors);
}

}  // namespace rhip
