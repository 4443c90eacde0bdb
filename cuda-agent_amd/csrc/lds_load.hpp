// Loads of 64 lanes x 16 bytes from global memory straight into LDS: lane l's bytes land at lds_base + 16*l (M0 carries
// lds_base). They are asm statements, so that they stay outside the compiler's bookkeeping of outstanding memory operations, which
// would make every later LDS read wait for them: a kernel awaits their completion itself (vmcnt).
//
// What the compiler puts in front of its own loads is then missing as well. The hardware doesn't wait for a scalar write of M0:
// one wait state (s_nop 0) has to lie between it and the load that reads M0. Nor does it wait for a vector instruction's write
// of the scalar registers of the address: five have to, of which the write of M0 is one and s_nop 3 four. (Where a kernel holds more
// base addresses than there are scalar registers, they come back through v_readlane right in front of their load.)
// tests/test_lds_loads.py looks at the built kernels.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace lds {

// from base + the lane's offset (bytes)
__device__ __forceinline__ void dma16(const void* base, uint32_t lane_byte_offset, uint32_t lds_base) {
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 3\n\tglobal_load_lds_dwordx4 %0, %1"
                 :
                 : "v"(lane_byte_offset), "s"(base), "s"(lds_base)
                 : "memory", "m0");
}

// the same with the non-temporal hint, for bytes that a launch reads once
__device__ __forceinline__ void dma16_once(const void* base, uint32_t lane_byte_offset, uint32_t lds_base) {
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 3\n\tglobal_load_lds_dwordx4 %0, %1 nt"
                 :
                 : "v"(lane_byte_offset), "s"(base), "s"(lds_base)
                 : "memory", "m0");
}

// from the lane's own address
__device__ __forceinline__ void dma16_ptr(const void* lane_ptr, uint32_t lds_base) {
    asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off"
                 :
                 : "v"(lane_ptr), "s"(lds_base)
                 : "memory", "m0");
}

}  // namespace lds
