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

#include "rhip_host.h"
#include "rhip_kernels.h"
#include "rhip_ring.h"

namespace rhip {

static_assert(kErrSlots == kRingErrors, "error words of a read");

namespace {

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
  const TexLevel level = lv ? *lv : TexLevel{};
  const int rc = readPieces(d->hip_device, d->stream, words * 4, out, errors,
                            [&](size_t at, size_t bytes, char *slot, uint32_t *errors_out) {
                              const size_t n = bytes / 4;
                              const unsigned grid = std::max(1u, std::min(blocks(n, 1024), 256u));
                              k_read_words<<<grid, 256, 0, d->stream>>>((const uint32_t *)src, level, layout, at / 4, n,
                                                                        (uint32_t *)slot,
                                                                        errors_out ? d->errors : nullptr, errors_out);
                              return hipGetLastError();
                            });
  if (rc != kNoPinned) return rc;
  if (layout == LAYOUT_LINEAR) return readPageable(d->stream, src, words, out, d->errors, errors);
  return readPageable(d->stream, src, (size_t)level.inner_w * level.inner_h, level.w, level.h, out, d->errors, errors,
                      [&](int x, int y) { return hostTexelIndex(level, layout, x, y); });
}

}  // namespace

int readLevel(rhip_device d, const uint8_t *src, const TexLevel &lv, int layout, void *out, uint32_t *errors) {
  return readWords(d, src, &lv, layout, (size_t)lv.w * lv.h, out, errors);
}

int readLinear(rhip_device d, const void *src, size_t words, void *out, uint32_t *errors) {
  return readWords(d, src, nullptr, LAYOUT_LINEAR, words, out, errors);
}

}  // namespace rhip
