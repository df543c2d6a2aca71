// Loads from a buffer straight into LDS, written in assembly: behind the builtin the compiler orders every transposing
// LDS read (ds_read_b64_tr_b16) after all loads in flight. They have no output register; the caller waits (vmcnt)
// before the bytes are read.
#pragma once
#include "common.cuh"

namespace w8a8 {

// A raw buffer descriptor in scalar registers, as lds_dma16's assembly takes it (see make_rsrc). Its words leave vector
// instructions, and five wait states pass until a load may read them; the compiler does not insert them into assembly,
// so they stand here.
__device__ __forceinline__ u32x4 make_desc(const void* p, uint32_t bytes) {
    const uint64_t addr = (uint64_t)p;
    u32x4 desc = {(uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)addr),
                  (uint32_t)__builtin_amdgcn_readfirstlane((int)((uint32_t)(addr >> 32) & 0xffffu)),
                  (uint32_t)__builtin_amdgcn_readfirstlane((int)bytes), 0x00020000u};
    __asm__ volatile("s_nop 4" : "+s"(desc));
    return desc;
}

// 16 bytes per lane into LDS at lds_addr + 16 * lane (lds_addr the same for the whole wave), with a descriptor of
// make_desc. Out-of-range lanes write zeros. One wait state after m0 is written; SPILLS, for kernels that keep scalar
// registers in lanes of vector ones, where a word may be restored right before: the five (1 x 4096 tokens of
// attn_prefill.hip, which spills none, 0.5% slower with them). (m0 is reserved and cannot be declared as clobbered:
// kernels with these loads use it for nothing else.)
template <bool SPILLS>
__device__ __forceinline__ void lds_dma16(u32x4 desc, uint32_t lds_addr, uint32_t voff) {
    __asm__ volatile(
        "s_mov_b32 m0, %0\n\t"
        "s_nop %3\n\t"
        "buffer_load_dwordx4 %1, %2, 0 offen lds"
        :
        : "s"(lds_addr), "v"(voff), "s"(desc), "n"(SPILLS ? 3 : 0)
        : "memory");
}

// The same at lds_addr + AT, soff (a scalar register) further on in memory: range-checked as part of the offset
template <int AT>
__device__ __forceinline__ void lds_dma16_at(u32x4 desc, uint32_t lds_addr, uint32_t voff, uint32_t soff) {
    __asm__ volatile(
        "s_add_u32 m0, %0, %4\n\t"
        "s_nop 0\n\t"
        "buffer_load_dwordx4 %1, %2, %3 offen lds"
        :
        : "s"(lds_addr), "v"(voff), "s"(desc), "s"(soff), "n"(AT)
        : "memory", "scc");
}

}  // namespace w8a8
