// LDS tiles and copies of the tall int8 prefill GEMM (gemm_i8.hip): a workgroup of
// producer and consumer waves computes a 256 x 128 tile of C in stages of 128 bytes of k per
// row.  The producers copy A tiles into LDS by DMA two stages ahead (three A buffers) and write
// the decoded weights of the next stage into one of two B buffers; a stage is released by a
// workgroup barrier.
//
// LDS: [kABuf][BM rows][ROWB] A tiles, then [2][BN rows][ROWB] B tiles, then what the producers
// stage besides.  Rows are 128 B in 8 chunks of 16 B; chunk c of row r is stored at
// c ^ ((r >> 1) & 7) (conflict-free fragment reads).
#pragma once
#include "common.h"
#include "gemm_sched.h"
#include "lds_dma.h"

namespace kata {
namespace gemm {

constexpr int BM = 256;          // rows of A / C per workgroup
constexpr int BKS = 64;          // k per stage (halves)
constexpr int ROWB = BKS * 2;    // LDS bytes per tile row
constexpr int NT = 4;            // 32-column MFMA tiles per workgroup
constexpr int BN = 32 * NT;      // columns per tile (128)
constexpr int kABuf = 3;         // A stage buffers (DMA two stages ahead)
constexpr int kTileBytes = kABuf * BM * ROWB + 2 * BN * ROWB;   // LDS before the producers' staging

typedef float v16f __attribute__((ext_vector_type(16)));

__device__ inline uint32_t swz(int row, int chunk) { return (uint32_t)(row * ROWB + ((chunk ^ ((row >> 1) & 7)) << 4)); }
__device__ inline uint8_t* tile_a(uint8_t* smem, int buf) { return smem + buf * (BM * ROWB); }
__device__ inline uint8_t* tile_b(uint8_t* smem, int buf) { return smem + kABuf * BM * ROWB + buf * (BN * ROWB); }

// Producer A copies: DMA instruction i of producer pw copies LDS bytes [1024 (4i + pw), +1024)
// of stage st's A tile: lane l -> tile row r = 8 (4i + pw) + l / 8, LDS slot l % 8, which
// holds global chunk (l % 8) ^ ((r >> 1) & 7) of that row (rows >= M read row M - 1); stages
// past the end copy the last one.  8 vector-memory instructions per call.
__device__ inline void issue_a(uint8_t* smem, int pw, int lane, const _Float16* A, int lda, int M, int m0, int st,
                               int nst) {
    const int ar_lo = 8 * pw + (lane >> 3);      // row for i = 0; + 32 i
    const int aslot = lane & 7;
    const int s2 = min(st, nst - 1);
    const uint32_t base = lds_addr(tile_a(smem, st % kABuf)) + 1024 * pw;
#pragma unroll
    for (int i = 0; i < 8; i++) {
        const int r = ar_lo + 32 * i;
        const int chunk = aslot ^ ((r >> 1) & 7);
        const _Float16* src = A + (size_t)min(m0 + r, M - 1) * lda + (size_t)s2 * BKS + chunk * 8;
        dma16(src, base + 4096 * i);
    }
}

}  // namespace gemm
}  // namespace kata
