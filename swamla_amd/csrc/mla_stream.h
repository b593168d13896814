// mla_stream.h — pieces shared by the kernels whose waves copy their own
// tiles into LDS and count their memory operations themselves (the prompt
// pass's expansion product and attention).
//
// The LDS copies are inline assembly with a uniform base and 32-bit lane
// offsets: the compiler does not see them, so it neither drains the copies
// in flight before an LDS read of another buffer nor forms a 64-bit address
// per lane and copy.  They have no result registers; they set M0, which the
// compiler reserves, so a kernel that uses them uses no builtin that needs
// it.  Every use of a tile sits behind the kernel's own wait (vmcnt) and barrier.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "mla_device.h"

namespace swamla {

typedef unsigned int st_u32x4_t __attribute__((ext_vector_type(4)));
typedef unsigned int st_u32x2_t __attribute__((ext_vector_type(2)));
typedef float f32x16_t __attribute__((ext_vector_type(16)));

// 16 bytes per lane from base + off (bytes; off per lane) into LDS at
// dst + 16 lane (base and dst uniform).
__device__ __forceinline__ void st_copy16(uint32_t dst, uint32_t off, const void* base) {
#ifdef __HIP_DEVICE_COMPILE__
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
               :: "s"(dst), "v"(off), "s"(base) : "memory");
#endif
}
// The same with an address per lane, and 4 bytes per lane into dst + 4 lane.
__device__ __forceinline__ void st_copy16_at(uint32_t dst, const void* p) {
#ifdef __HIP_DEVICE_COMPILE__
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" :: "s"(dst), "v"(p) : "memory");
#endif
}
__device__ __forceinline__ void st_copy4_at(uint32_t dst, const void* p) {
#ifdef __HIP_DEVICE_COMPILE__
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, off" :: "s"(dst), "v"(p) : "memory");
#endif
}

// LDS operand reads at a byte address (compiler-visible: it counts them and
// waits before their uses; the kernels fix their order with scheduling
// barriers).
template <typename T>
__device__ __forceinline__ T st_read(uint32_t addr) {
  return *reinterpret_cast<const __attribute__((address_space(3))) T*>(addr);
}
template <typename T>
__device__ __forceinline__ void st_write(uint32_t addr, T v) {
  *reinterpret_cast<__attribute__((address_space(3))) T*>(addr) = v;
}
__device__ __forceinline__ s16x4_t st_read_tr(uint32_t addr) {
  return __builtin_amdgcn_ds_read_tr16_b64_v4i16(reinterpret_cast<__attribute__((address_space(3))) s16x4_t*>(addr));
}

// Everything this wave has in flight (copies, stores, LDS reads) is done,
// then the workgroup barrier: tiles copied before it are complete after it,
// and no wave still reads a buffer the next copies overwrite.
__device__ __forceinline__ void st_tile_barrier() {
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

// f(0) ... f(N - 1) with compile-time indices.
template <int I, int N, typename F>
__device__ __forceinline__ void st_for(F&& f) {
  if constexpr (I < N) {
    f(std::integral_constant<int, I>{});
    st_for<I + 1, N>(f);
  }
}
constexpr int st_min(int a, int b) { return a < b ? a : b; }

}  // namespace swamla
