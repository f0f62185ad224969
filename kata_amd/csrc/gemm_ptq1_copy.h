// Copies of PTQ1_0 weight blocks into LDS, shared by the prefill GEMMs that decode them into
// registers (gemm_f16.hip, gemm_i8.hip): groups of two 28-byte blocks of each of a tile's BN rows.
// The 56 bytes of a row's group are four 16-byte pieces at 0, 16, 32, 40 (a last group of one block:
// 0, 12), so no copy reads past the row; row r's piece p sits in slot p ^ ((r >> 2) & 3) of its 64
// LDS bytes.
#pragma once
#include "gemm_reg.h"

namespace kata {

struct Ptq1Copy {
    static constexpr int kBlockB = kBlockBytes;   // bytes of 128 k of a row
    static constexpr int GROUP = 2;               // blocks per copied group
    template <class C>
    static constexpr int copies() {
        static_assert(C::BN * 4 % C::THREADS == 0, "whole weight copies per thread");
        return C::BN * 4 / C::THREADS;
    }
    template <class C>
    static constexpr int slot_bytes() { return C::BN * 64; }

    const uint8_t* wbase[4];                      // copy sources: per instruction a uniform row base
    uint32_t wvo[4];                              // and this lane's offset (full group)
    uint32_t wsingle;                             // added to it in a group of one block
    uint32_t w_lds;
    int nblk;
    uint32_t rd;                                  // LDS address of this lane's row (tile 0) in slot 0
    uint32_t f16_;                                // 16 times the row's slot swizzle

    template <class C>
    __device__ inline void init_copy(const uint8_t* W, int nbk, int kb0, int nb, int n0, int N, int tid, int wave, int wc,
                                     int l32, uint32_t Ws) {
        const uint32_t row_bytes = (uint32_t)nbk * kBlockBytes;
        constexpr int RPI = C::THREADS / 4;
        nblk = nb;
#pragma unroll
        for (int i = 0; i < copies<C>(); i++) {
            const int r0 = min(n0 + i * RPI, N - 1), r = tid / 4;
            const int p = (tid & 3) ^ (((i * RPI + r) >> 2) & 3);
            wbase[i] = W + (size_t)r0 * row_bytes + (size_t)kb0 * kBlockBytes;
            wvo[i] = (uint32_t)min(r, N - 1 - r0) * row_bytes + (p < 3 ? 16u * p : 40u);
        }
        const int p = (tid & 3) ^ ((tid >> 4) & 3);
        wsingle = p == 0 ? 0u : (uint32_t)(12 - (p < 3 ? 16 * p : 40));
        w_lds = Ws + 1024u * wave;
        rd = Ws + (wc * 32 * C::NT + l32) * 64;
        f16_ = ((uint32_t)(l32 >> 2) & 3u) << 4;
    }
    // LDS offset of piece p in this lane's row
    __device__ inline uint32_t piece(uint32_t p) const { return (p << 4) ^ f16_; }
    template <class C>
    __device__ inline void issue(int g, int slot, int i0, int i1) {
        const uint32_t add = 2 * g + 1 == nblk ? wsingle : 0u;
#pragma unroll
        for (int i = i0; i < i1; i++)
            dma16(wbase[i] + (size_t)g * (2 * kBlockBytes), wvo[i] + add,
                      w_lds + slot * slot_bytes<C>() + i * (C::THREADS * 16));
    }
};

__host__ __device__ constexpr uint32_t p3x2(int n) {
    return n == 0 ? 0x00010001u : n == 1 ? 0x00030003u : n == 2 ? 0x00090009u : n == 3 ? 0x001b001bu : 0x00510051u;
}
// the bytes (b0, b1) / (b2, b3) of w in 16-bit lanes (v_perm selector 0x0c is a zero byte)
__device__ inline rg::u16x2 bytes01(uint32_t w) { return __builtin_bit_cast(rg::u16x2, __builtin_amdgcn_perm(0u, w, 0x0c010c00u)); }
__device__ inline rg::u16x2 bytes23(uint32_t w) { return __builtin_bit_cast(rg::u16x2, __builtin_amdgcn_perm(0u, w, 0x0c030c02u)); }

}  // namespace kata
