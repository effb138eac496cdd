// Loads from global memory straight into LDS.  The caller waits (s_waitcnt vmcnt) before the barrier behind which it reads.
#pragma once
#include <cstdint>

// 64 lanes x 16 (4) bytes: base + off_lane of every lane to lds, lane after lane.  Inline assembly: with the compiler's form of
// these loads every later wait on an LDS read is a wait for all loads in flight.  Behind m0's write, and for a base that a
// vector instruction has put into scalar registers (readfirstlane, a reload of a spilled one: five wait states), the waits
// stand in the block, since the compiler does not look into it.
__device__ __forceinline__ void lds_dma_1k(const void* base, uint32_t off_lane, uint32_t lds) {
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 4\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(off_lane), "s"(base), "s"(lds) : "memory", "m0");
}
__device__ __forceinline__ void lds_dma_256(const void* base, uint32_t off_lane, uint32_t lds) {
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 4\n\tglobal_load_lds_dword %0, %1" ::"v"(off_lane), "s"(base), "s"(lds) : "memory", "m0");
}
__device__ __forceinline__ uint32_t lds_addr(const void* p) {
    return static_cast<uint32_t>(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) void*)(p)));
}
// a pointer that is the same in all lanes, in scalar registers (readfirstlane is signed: the low half must not spread its sign)
__device__ __forceinline__ const uint8_t* lds_dma_base(const uint8_t* p) {
    const uint64_t v = reinterpret_cast<uint64_t>(p);
    const uint32_t lo = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(static_cast<uint32_t>(v)))),
                   hi = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(static_cast<uint32_t>(v >> 32))));
    return reinterpret_cast<const uint8_t*>(static_cast<uint64_t>(hi) << 32 | lo);
}
