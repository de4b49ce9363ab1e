// Pieces that the MFMA kernels whose K loops load by LDS DMA share (hn_gemm.hip,
// hn_mid.hip): buffer descriptors, loads from memory straight to LDS, the explicit
// waits on them, and the constants of the in-register INT4 unpack.
#pragma once
#include "hn_common.h"

namespace {

typedef __attribute__((address_space(3))) void lds_void_t;

__device__ __forceinline__ __amdgpu_buffer_rsrc_t rsrc(const void* p, int bytes) {
  return __builtin_amdgcn_make_buffer_rsrc((void*)p, (short)0, bytes, 0x00020000);
}

// ---------------------------------------------------------------------------
// Loads.  What a K loop stages through LDS (the prefill GEMM everything that it
// reads, the middle-size kernels their activations) goes from memory to LDS directly
// (buffer_load ... lds: lane i's bytes land at m0 + size * i) through the
// compiler's LDS-DMA builtin, which sets M0 and places the wait states gfx9
// needs between a VALU or SALU write of an SGPR operand (M0, soffset, the
// descriptor) and the load that reads it.  The compiler does not wait on
// these loads before the K loop's LDS reads: every wait on them is explicit
// (s_waitcnt vmcnt below), and loads return in issue order.  Offsets: the
// per-lane part is in voffset (the buffer range check covers voffset only, so
// rows past N carry an offset past the descriptor's range and read as 0
// without touching memory); the per-group part is in soffset.
// ---------------------------------------------------------------------------
__device__ __forceinline__ lds_void_t* lds_ptr(uint32_t addr) {
  return (lds_void_t*)((__attribute__((address_space(3))) char*)nullptr + addr);
}

__device__ __forceinline__ void dma_b128(__amdgpu_buffer_rsrc_t r, uint32_t voff, uint32_t soff,
                                         uint32_t lds) {
  // soffset and the LDS address are uniform by construction
  __builtin_amdgcn_raw_ptr_buffer_load_lds(r, lds_ptr(__builtin_amdgcn_readfirstlane(lds)), 16,
                                           voff, __builtin_amdgcn_readfirstlane(soff), 0, 0);
}

template <int N>
__device__ __forceinline__ void wait_vmcnt() {
  static_assert(N >= 0 && N < 64, "vmcnt range");
  asm volatile("s_waitcnt vmcnt(%0)" :: "n"(N) : "memory");
}

// The K loop's barrier: this wave's LDS reads have returned (another wave's
// loads may overwrite what they read right after it), LDS accesses stay on
// their side of it, and the loads of later stages stay in flight.  (A
// __syncthreads is also a release fence, for which the compiler waits until
// every LDS-DMA load of the wave has landed: the loads of stage t + 2, issued
// at the start of stage t, then had to arrive before stage t could end.  4096
// rows over eight Mixtral experts by the prefill GEMM on MI355X, with
// __syncthreads and with this: 1571 to 102 rows each, gate/up 1012 -> 994 us,
// down 548 -> 536; 512 each, 877 -> 872 and 428 -> 424.)
__device__ __forceinline__ void stage_barrier() {
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

template <typename T>
__device__ __forceinline__ T lds_read(uint32_t addr) {
  return *reinterpret_cast<const __attribute__((address_space(3))) T*>(
      (__attribute__((address_space(3))) char*)nullptr + addr);
}

// Unpack constants (gfx9 VOP3 takes no literals): mask in an SGPR, the rest
// in VGPRs.
struct DeqRegs {
  uint32_t m_pair;  // SGPR 0x00F0000F: low nibble of byte 0, high nibble of byte 2
  uint32_t magic;   // 0x64006400
  uint32_t mul;     // half2(1, 1/16)
  uint32_t add;     // half2(-1032, -72)
};

}  // namespace
