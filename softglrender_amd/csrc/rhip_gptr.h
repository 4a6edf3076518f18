/*
 * rhip_gptr.h -- pointers to device memory inside structures.
 */
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace rhip {

/* A pointer to device memory, for structures that kernels read from memory
 * (texture descriptors, the parameters of batched views): the compiler takes a
 * pointer it loads to point anywhere and reads through flat loads, which also
 * count as LDS accesses and are waited for with them; the cast says that it is
 * global. PBR shading of a full HD 4x frame took 137 us (now 125), the persistent
 * raster of 48 batched views 455 us (381, with its share of other changes). */
template <typename T>
struct GPtr {
  T *p;
  GPtr() = default;
  __host__ __device__ GPtr(T *q) : p(q) {}
  __host__ __device__ __forceinline__ operator T *() const {
#ifdef __HIP_DEVICE_COMPILE__
    /* through an integer: a cast there and back again would fold away */
    return (T *)(__attribute__((address_space(1))) T *)(uintptr_t)p;
#else
    return p;
#endif
  }
  __host__ __device__ __forceinline__ T *operator->() const { return *this; }
  template <typename U>
  __host__ __device__ __forceinline__ explicit operator U *() const {
    return (U *)(T *)*this;
  }
};

}  // namespace rhip
