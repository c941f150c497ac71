// Device helpers shared by the matrix-core conv kernels (conv_halo.hip,
// conv_ring.hip): vector types, raw buffer resources, direct global -> LDS
// loads.
#pragma once
#include "cf_common.h"

namespace {

typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef float f16v __attribute__((ext_vector_type(16)));
typedef _Float16 h4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));

// Raw buffer resource over [base, base + bytes) (gfx9 word 3).  Buffer
// loads outside the range return zeros and buffer stores outside it are
// dropped by the hardware, so the lean epilogue issues every load and store
// unconditionally (a fixed count per step, which lets the compiler wait for
// exactly the loads it needs instead of draining earlier stores).
__device__ __forceinline__ __amdgpu_buffer_rsrc_t halo_rsrc(const void* base, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), (short)0, (int)bytes,
                                           0x00020000);
}
constexpr uint32_t HALO_OOB = 0x80000000u;  // an offset beyond every range used here

// Sixteen zero bytes in device memory: absent route words (counts,
// descriptors) are read from here.
__device__ __attribute__((aligned(16))) u32x4 g_halo_zero;

// Returns x unchanged, hidden from the optimiser: per-element addresses
// derived from it are recomputed where they are used instead of being kept
// live (in registers or scratch) across the K loop.
__device__ __forceinline__ int opaque(int x) {
  asm volatile("" : "+v"(x));
  return x;
}

constexpr int KC = 32;  // channels per chunk: four 16-byte parts per staged pixel

// One direct global -> LDS load (buffer_load_dwordx4 ... lds): lane l
// copies the 16 bytes at byte offset voff of the buffer rsrc (zeros when
// voff is beyond its range) to LDS byte address lds + 16 l (lds
// wave-uniform); the buffer's base is in scalar registers, so a copy takes
// no vector address arithmetic.
// Issued through inline assembly so that the compiler does not track it:
// its own load counting then never waits for these copies (it only waits
// for loads it issued, which in-order completion makes safe: a copy issued
// after a load never delays the wait for that load).  The kernel waits for
// the copies itself (s_waitcnt vmcnt and a barrier) before reading them.
typedef int cf_v4i __attribute__((ext_vector_type(4)));
__device__ __forceinline__ void lds_buf_copy16(cf_v4i rsrc, unsigned voff, unsigned lds) {
  asm volatile(
      "s_mov_b32 m0, %2\n\t"
      "s_nop 0\n\t"
      "buffer_load_dwordx4 %0, %1, 0 offen lds"
      :
      : "v"(voff), "s"(rsrc), "s"(lds)
      : "memory", "m0");
}
// The same with a wave-uniform byte offset soff added to the address.
__device__ __forceinline__ void lds_buf_copy16_at(cf_v4i rsrc, unsigned voff, unsigned soff,
                                                  unsigned lds) {
  asm volatile(
      "s_mov_b32 m0, %2\n\t"
      "s_nop 0\n\t"
      "buffer_load_dwordx4 %0, %1, %3 offen lds"
      :
      : "v"(voff), "s"(rsrc), "s"(lds), "s"(soff)
      : "memory", "m0");
}
// Raw buffer resource words (as halo_rsrc) in scalar registers, for inline
// assembly.
__device__ __forceinline__ cf_v4i halo_rsrc_v4(const void* base, uint32_t bytes) {
  const uint64_t p = (uint64_t)(uintptr_t)base;
  cf_v4i r;
  r[0] = __builtin_amdgcn_readfirstlane((int)(uint32_t)p);
  r[1] = __builtin_amdgcn_readfirstlane((int)((uint32_t)(p >> 32) & 0xffffu));
  r[2] = (int)bytes;
  r[3] = 0x00020000;
  return r;
}
__device__ __forceinline__ unsigned lds_addr(const void* p) {
  return (unsigned)(uintptr_t)(const __attribute__((address_space(3))) void*)p;
}

// EPI_POOL: BN -> AvgPool2d(2, 2) -> LIF, the pooled spikes as the fp16
// NHWC copy, the pooled membrane state.
enum { EPI_LIF = 0, EPI_Z = 1, EPI_POOL = 2 };
enum { ID_ADD_SPIKE = 1, ID_ADD_Z = 2 };

}  // namespace
