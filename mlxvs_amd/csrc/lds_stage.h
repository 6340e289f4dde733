// Staging rows in LDS for the MFMA kernels: direct loads and the waits around
// them.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace mlxvs::kern {

// Buffer loads of 16 / 4 bytes per lane straight into LDS: lane l writes at
// lds + 16 l (4 l); lds is wavefront-uniform; out-of-range lanes write
// zeros.  (The builtin exists only for the device target.)
__device__ __forceinline__ void load16_to_lds(__amdgpu_buffer_rsrc_t r, void* lds, uint32_t voff) {
#if defined(__HIP_DEVICE_COMPILE__)
  __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (__attribute__((address_space(3))) void*)lds, 16,
                                           voff, 0, 0, 0);
#else
  (void)r, (void)lds, (void)voff;
#endif
}
__device__ __forceinline__ void load4_to_lds(__amdgpu_buffer_rsrc_t r, void* lds, uint32_t voff) {
#if defined(__HIP_DEVICE_COMPILE__)
  __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (__attribute__((address_space(3))) void*)lds, 4,
                                           voff, 0, 0, 0);
#else
  (void)r, (void)lds, (void)voff;
#endif
}

// A workgroup barrier after this wavefront's outstanding vector-memory
// operations -- its LDS-direct loads among them -- have completed: an LDS
// buffer that every wavefront fills with LDS-direct loads is whole once all
// have passed it.  (The barrier's own workgroup-scope fence does not wait
// for loads, so the wait is explicit.)
__device__ __forceinline__ void dma_barrier() {
  __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0), no other counter
  __syncthreads();
}

// Wait states between a barrier and the first read of MFMA results issued
// before it.  The compiler's MFMA-to-VALU dependency count includes the
// barrier and the wait in front of it, which need not take a cycle (a
// wavefront that arrives last passes both at once): reading the last
// accumulator registers first, at the count it derived, gave stale values
// now and then (lists that lost a candidate, measured on the GPU: gone with
// 8 more wait states, not with 1).  Twenty-four, fenced so that nothing is
// scheduled across them: more than the longest MFMA here needs (16 passes
// + 2) whether or not the compiler counts them towards its own.
__device__ __forceinline__ void mfma_settle() {
  __builtin_amdgcn_sched_barrier(0);
  asm volatile("s_nop 7\n\ts_nop 7\n\ts_nop 7");
  __builtin_amdgcn_sched_barrier(0);
}

}  // namespace mlxvs::kern
