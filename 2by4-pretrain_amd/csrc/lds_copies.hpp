// What the kernels that stream operands through LDS into matrix instructions share: vector types, copies from memory straight
// into LDS, the waits that go with them, and the number of compute units that tiles are dealt to.
#pragma once
#include "tf24_common.hpp"
#include <atomic>

namespace tf24 {
namespace {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float float4v __attribute__((ext_vector_type(4)));
typedef float float16v __attribute__((ext_vector_type(16)));
typedef short short4v __attribute__((ext_vector_type(4)));
typedef int int4v __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) void* lds_ptr_t;
typedef __attribute__((address_space(3))) short4v* lds_short4_ptr;

// The copies are issued from inline assembly so that the compiler's wait-count insertion does not
// see them: it would otherwise drain all outstanding copies (vmcnt(0)) before every LDS read, because
// it cannot tell the stage buffers apart.  Ordering is enforced by hand with s_waitcnt vmcnt(N)
// before the stage barrier.  M0 carries the wave-uniform LDS base of the copy.
__device__ __forceinline__ uint32_t lds_offset(const void* p) {
  return (uint32_t)(uintptr_t)(lds_ptr_t)p;
}
// Lane l brings 16 bytes to LDS[base + 16*l].  The source address is a wave-uniform 64-bit base in scalar registers plus a
// 32-bit offset per lane: with a 64-bit address per lane the same copies hold up the matrix instructions issued around them (on an
// instruction mix like the products' main loop, 25 % more cycles than the matrix instructions alone against 3 %).
__device__ __forceinline__ void g2l16(const uint8_t* base, uint32_t lane_offset, uint32_t lds_base) {
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(lane_offset), "s"(base), "s"(lds_base) : "memory", "m0");
}
// the same with one dword per lane: lane l writes LDS[base + 4*l]
__device__ __forceinline__ void g2l4(const uint8_t* base, uint32_t lane_offset, uint32_t lds_base) {
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dword %0, %1" ::"v"(lane_offset), "s"(base), "s"(lds_base) : "memory", "m0");
}
// At most N of this wave's copies still in flight, then a workgroup barrier (a bare s_barrier: __syncthreads() would add
// a fence that drains every outstanding copy).  READS: this wave's LDS reads are complete as well, for rings whose next
// copies go into the stage just read.
template <int N, bool READS>
__device__ __forceinline__ void wait_copies_and_barrier() {
  if constexpr (READS) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(N) : "memory");
  else asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(N) : "memory");
}
// workgroup barrier behind this wave's LDS reads only: copies stay in flight
__device__ __forceinline__ void wait_reads_and_barrier() {
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}
// compute units of the current device (looked up once per device; the cache is a table of atomics: two threads
// that meet on an empty entry both look the value up and store the same number)
inline int compute_units() {
  static std::atomic<int> cached[64];
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
  int n = cached[dev].load(std::memory_order_relaxed);
  if (!n) {
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0) n = 256;
    cached[dev].store(n, std::memory_order_relaxed);
  }
  return n;
}

}  // namespace
}  // namespace tf24
