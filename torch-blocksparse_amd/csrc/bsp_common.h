// Shared declarations for the gfx950 block-sparse kernels: status helpers, 16-bit types, MFMA wrappers.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <atomic>
#include "../../include/bsp.h"

#define BSP_HIP_CHECK(expr)                       \
  do {                                            \
    hipError_t e__ = (expr);                      \
    if (e__ != hipSuccess) return BSP_ERR_HIP;    \
  } while (0)

// Launch check: asynchronous launches only report configuration errors here.
#define BSP_LAUNCH_CHECK()                                 \
  do {                                                     \
    if (hipGetLastError() != hipSuccess) return BSP_ERR_HIP; \
  } while (0)

namespace bsp {

// A builder that allocates host memory, behind its C entry point: no exception may leave that
template <class F> int no_throw(F &&build) {
  try {
    return build();
  } catch (...) {
    return BSP_ERR_UNSUPPORTED;
  }
}

// Kernels that use more dynamic LDS than a launch may ask for by default: the limit of a kernel is raised once per device
// (a bit per device; devices past the 64th set it at every launch), from whichever thread gets there.
inline bool raise_lds_limit(const void *kernel, int bytes, std::atomic<uint64_t> &done) {
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) return false;
  const uint64_t bit = dev < 64 ? uint64_t(1) << dev : 0;
  if (bit && (done.load(std::memory_order_acquire) & bit)) return true;
  if (hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, bytes) != hipSuccess) return false;
  done.fetch_or(bit, std::memory_order_release);
  return true;
}

typedef _Float16 f16;
typedef __bf16 bf16;

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

static inline int cdiv(int64_t a, int64_t b) { return (int)((a + b - 1) / b); }
static inline hipStream_t as_stream(void *s) { return reinterpret_cast<hipStream_t>(s); }

// Workgroups are dealt round-robin to the 8 XCDs (each with its own L2).  Re-number them so that the
// workgroups that land on one XCD cover one contiguous range of work items.
__device__ __forceinline__ int64_t xcd_remap(int64_t wg, int64_t n_wg) {
  const int64_t per = n_wg >> 3;
  const int64_t full = per << 3;
  if (wg >= full) return wg;            // ragged tail keeps its position
  return (wg & 7) * per + (wg >> 3);
}

// n = q d + r.  The place of a workgroup in its launch, which has fewer than 2^31, is computed with these: a division of 64 bits is a
// hundred scalar instructions one after the other, a quarter of a microsecond before the first load (fp32 sdd of 213 blocks of 64,
// reduction 512: one such division more took it from 25.2 to 25.7 us).
struct Quotient {
  uint32_t q, r;
  __device__ __forceinline__ Quotient(uint32_t n, uint32_t d) : q(n / d), r(n - q * d) {}
};

// Look-up tables are read-only for every kernel that consumes them.  Reading them through the constant address
// space lets the compiler use scalar loads for wave-uniform entries even after a barrier (a plain global pointer
// falls back to vector loads there, and waiting for such a load means waiting for every prefetch issued before it).
typedef const int32_t __attribute__((address_space(4))) *table_ptr;
__device__ __forceinline__ table_ptr as_table(const int32_t *p) { return (table_ptr)p; }

template <typename T> struct TypeInfo;
template <> struct TypeInfo<f16> { static constexpr int kVec = 8; static constexpr bool k16 = true; };
template <> struct TypeInfo<bf16> { static constexpr int kVec = 8; static constexpr bool k16 = true; };
template <> struct TypeInfo<float> { static constexpr int kVec = 4; static constexpr bool k16 = false; };

__device__ __forceinline__ float to_float(f16 v) { return (float)v; }
__device__ __forceinline__ float to_float(bf16 v) { return (float)v; }
__device__ __forceinline__ float to_float(float v) { return v; }
template <typename T> __device__ __forceinline__ T from_float(float v) { return (T)v; }

}  // namespace bsp
