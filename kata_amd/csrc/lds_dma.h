// Copies from memory straight into LDS, shared by the GEMV (gemv_ptq1.hip) and every prefill GEMM.
// Through inline assembly so that the compiler does not make later LDS accesses wait for every copy
// in flight (it cannot tell which LDS bytes one writes); the kernels wait for these copies
// explicitly.  lds (wave-uniform) is the LDS byte address of lane 0 and goes through M0, which is
// restored.  The s_nop is the wait state that gfx950 wants between a write of M0 and a copy that
// uses it: the hazard recogniser inserts it between instructions of its own and does not look in
// here.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace kata {

#define KATA_LDS_COPY(op, addr) \
    "s_mov_b32 %0, m0\n\ts_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_" op " " addr "\n\ts_mov_b32 m0, %0"

// 16 bytes per lane from g to lds + 16 * lane
__device__ inline void dma16(const void* g, uint32_t lds) {
    uint32_t saved;
    asm volatile(KATA_LDS_COPY("dwordx4", "%2, off") : "=&s"(saved) : "s"(lds), "v"(g) : "memory");
}
// the same from base + voff (base wave-uniform)
__device__ inline void dma16(const void* base, uint32_t voff, uint32_t lds) {
    uint32_t saved;
    asm volatile(KATA_LDS_COPY("dwordx4", "%2, %3") : "=&s"(saved) : "s"(lds), "v"(voff), "s"(base) : "memory");
}
// one dword per lane to lds + 4 * lane
__device__ inline void dma4(const void* g, uint32_t lds) {
    uint32_t saved;
    asm volatile(KATA_LDS_COPY("dword", "%2, off") : "=&s"(saved) : "s"(lds), "v"(g) : "memory");
}
__device__ inline void dma4(const void* base, uint32_t voff, uint32_t lds) {
    uint32_t saved;
    asm volatile(KATA_LDS_COPY("dword", "%2, %3") : "=&s"(saved) : "s"(lds), "v"(voff), "s"(base) : "memory");
}
#undef KATA_LDS_COPY

// the LDS byte address of p (wave-uniform)
__device__ inline uint32_t lds_addr(const void* p) {
    return __builtin_amdgcn_readfirstlane((uint32_t)(size_t)(__attribute__((address_space(3))) const void*)p);
}

}  // namespace kata
