// Global -> LDS copies that pass no registers (buffer loads with the LDS modifier), for kernels that count them themselves.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace gq {

namespace {

typedef int i32x4 __attribute__((ext_vector_type(4)));

// One 16-byte-per-lane buffer load whose data goes to LDS at lds_addr + 16 * lane.  The compiler
// does not see that the instruction writes LDS or that it is counted by vmcnt: the kernel orders
// these loads against its LDS reads with explicit waits and barriers.  (The s_nop is the wait
// state the hardware wants between a write of M0 and an LDS DMA; the assembler does not add it
// inside inline assembly.)
__device__ __forceinline__ void dma16(uint32_t lds_addr, i32x4 rsrc, uint32_t voff, uint32_t soff) {
    lds_addr = __builtin_amdgcn_readfirstlane(lds_addr);  // both are uniform by construction
    soff = __builtin_amdgcn_readfirstlane(soff);
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds" ::"s"(lds_addr), "v"(voff), "s"(rsrc), "s"(soff) : "memory");
}

// Raw buffer over `bytes` bytes from `base` (reads past the end return zero and touch no memory).
__device__ __forceinline__ i32x4 make_rsrc(const void *base, uint64_t bytes) {
    const uint64_t b = reinterpret_cast<uint64_t>(base);
    i32x4 r;
    r.x = __builtin_amdgcn_readfirstlane((int)(uint32_t)b);
    r.y = __builtin_amdgcn_readfirstlane((int)(uint32_t)(b >> 32));  // stride 0: raw buffer, byte offsets
    r.z = __builtin_amdgcn_readfirstlane((int)(uint32_t)(bytes > 0xFFFFFFFFull ? 0xFFFFFFFFull : bytes));
    r.w = 0x00020000;  // 32-bit data format, no swizzle
    return r;
}

}  // namespace

}  // namespace gq
