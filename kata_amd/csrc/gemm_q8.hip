// Exact fp16 prefill GEMM over a Q8_0 matrix, the quants decoded into the MFMA's registers: the
// MTP head's K/V catch-up (Engine::encMtpKv, src/engine.cpp:392-401: k_expand_q8 then
// dGemm, shaders/mtp.metal:24-33).
//
// Semantics: C[m][n] = sum_k A[m][k] * half(d[n][k/32] * q[n][k]),  fp16 x fp16 -> fp32,
// with half() round-to-nearest-even as the reference's expansion.  Every product term equals
// the reference's; only the fp32 summation order differs (tolerance-based parity).
//
// Design: the skeleton of gemm_reg.h (tiles of 64, 128 or 256 rows by 256 columns, weights
// decoded straight into MFMA registers) with a Q8_0 decode:
//  * Copies: a 128-k block is four 34-byte blocks of each of the tile's 256 weight rows (136 bytes,
//    dword-aligned), copied into LDS by DMA one or two blocks ahead as nine 16-byte pieces (at
//    bytes 0, 16, .. 112 and 120, the last overlapping so that no copy reads past the block).
//  * Decode: lane half lh of a column takes 8 consecutive quants per 16-k step.  An int8 q
//    becomes an exact fp16 through its bits: byte q ^ 0x80 as the low byte under a 0x66 high
//    byte is the fp16 1536 + (q + 128), minus 1664 is q; one packed fp16 multiply by d then
//    rounds d * q once, to nearest even, as half(d * float(q)) does (the fp32 product of an
//    fp16 and a 7-bit integer is exact).
// What bounds it: up to a few hundred rows the packed bytes' way into LDS (36 KB a block, 5 DMA
// instructions per wave, spread over the stages: 74.7 -> 66.7 us at 333 rows), bank conflicts (half the
// LDS cycles: rows are 144 bytes apart) and the 3 us to the first MFMA; many rows the matrix cores and
// the vector instructions beside them.  10240 -> 5120 / 5120 ->
// 1024 before (256 x 128 tiles, decoded weights through LDS) -> now, us: 28 rows 45.9 / 16.4 ->
// 23.1 / 11.9, 333 rows 77.5 / 23.1 -> 60.9 / 19.3, 512 rows 78.8 / 22.9 -> 77.5 / 21.7, 4000 rows
// 491 / 64 -> 428 / 61.
#include "common.h"
#include "launch.h"

#include "gemm_reg.h"

namespace kata {

namespace {

struct Q8F16 {
    static constexpr bool TWO_FORMS = false;
    static constexpr int GROUP = 1;
    static constexpr int kBlockB = 4 * kQ8BlockBytes;
    static constexpr int kPieces = 9, kRowB = 16 * kPieces;
    template <class C>
    static constexpr int copies() { return (C::BN * kPieces + C::THREADS - 1) / C::THREADS; }
    template <class C>
    static constexpr int slot_bytes() { return C::BN * kRowB; }

    const uint8_t* wbase;                         // block kb0 of the tile's first row
    uint32_t wvo[9];                              // this lane's copy sources from there
    uint32_t w_lds;
    int wave;
    uint32_t rd;                                  // LDS address of this lane's row (tile 0) in slot 0, plus 8 lh
    uint32_t last;                                // 8 for lh = 1: the last quants sit in the overlapping piece
    uint32_t w[2][2][3], dw[2][2];                // words of steps kk % 2; scale words of blocks (kk / 2) % 2

    template <class C>
    __device__ inline void init(const uint8_t* W, int nbk, int kb0, int, int n0, int N, int tid, int wave_, int wc,
                                int l32, int lh, uint32_t Ws) {
        const uint32_t row_bytes = (uint32_t)nbk * 136u;
        wbase = W + (size_t)n0 * row_bytes + (size_t)kb0 * 136;
        wave = wave_;
#pragma unroll
        for (int i = 0; i < copies<C>(); i++) {
            // pieces past the tile's last repeat the wave's previous ones
            const int idx = (i * C::THREADS + wave * 64 < C::BN * kPieces ? i : i - 1) * C::THREADS + tid;
            const int r = idx / kPieces, p = idx % kPieces;
            wvo[i] = (uint32_t)min(r, N - 1 - n0) * row_bytes + (p < 8 ? 16u * p : 120u);
        }
        w_lds = Ws + 1024u * wave;
        rd = Ws + (wc * 32 * C::NT + l32) * kRowB + 8 * lh;
        last = 8u * lh;
    }
    template <class C>
    __device__ inline void issue(int g, int slot, int i0, int i1) {
#pragma unroll
        for (int i = i0; i < i1; i++) {
            const int at = i * C::THREADS + wave * 64 < C::BN * kPieces ? i : i - 1;
            dma16(wbase + (size_t)g * 136, wvo[i],
                      __builtin_amdgcn_readfirstlane(w_lds + slot * slot_bytes<C>() + at * (C::THREADS * 16)));
        }
    }
    template <class C, int J>
    __device__ inline void read(int, int, int) {}
    template <class C>
    __device__ inline bool begin() { return false; }
    // the words of step kb + 2 (of the next block for kb = 6, 7): its 8 quants, whose first byte
    // is 2 bytes into a word in even blocks, and the scale with a block's first step
    template <class C, int kb>
    __device__ inline void look(int g) {
        constexpr int kk = (kb + 2) % 8, b = kk / 2, q0 = (34 * b + 2 + 16 * (kk & 1)) & ~3;
        const uint32_t s = rd + (uint32_t)((kb >= 6 ? g + 1 : g) % (C::DW + 1)) * slot_bytes<C>();
#pragma unroll
        for (int t = 0; t < C::NT; t++) {
            const uint32_t a = s + t * (32 * kRowB);
            const uint32_t e = kk == 7 ? a + last : a;
            w[kk & 1][t][0] = rg::lds_ld<uint32_t>(e + q0);
            w[kk & 1][t][1] = rg::lds_ld<uint32_t>(e + q0 + 4);
            if constexpr (b % 2 == 0) w[kk & 1][t][2] = rg::lds_ld<uint32_t>(a + q0 + 8);
            if constexpr (kk % 2 == 0) dw[b & 1][t] = rg::lds_ld<uint32_t>(a - last + ((34 * b) & ~3));
        }
    }
    template <int kk, bool>
    __device__ inline v8h chunk(int t) {
        constexpr int b = kk / 2;
        const uint32_t(&x)[3] = w[kk & 1][t];
        const uint32_t q[2] = {b % 2 ? x[0] : __builtin_amdgcn_alignbyte(x[1], x[0], 2),
                               b % 2 ? x[1] : __builtin_amdgcn_alignbyte(x[2], x[1], 2)};
        const v2h d = __builtin_bit_cast(v2h, __builtin_amdgcn_perm(0u, dw[b & 1][t], b % 2 ? 0x03020302u : 0x01000100u));
        const v2h off = {(_Float16)1664.0f, (_Float16)1664.0f};
        uint32_t o[4];
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const uint32_t u = q[j / 2] ^ 0x80808080u;
            const v2h v = __builtin_bit_cast(v2h, __builtin_amdgcn_perm(0x66666666u, u, j & 1 ? 0x04030402u : 0x04010400u)) - off;
            o[j] = __builtin_bit_cast(uint32_t, v * d);
        }
        return __builtin_bit_cast(v8h, make_uint4(o[0], o[1], o[2], o[3]));
    }
};

//               MT NT WR WC  KS DA DW waves per SIMD
typedef rg::Cfg<2, 1, 1, 8, 64, 2, 2, 2> Cfg64;      // 64 x 256
typedef rg::Cfg<4, 1, 1, 8, 32, 3, 2, 2> Cfg128;     // 128 x 256
typedef rg::Cfg<8, 2, 1, 4, 32, 3, 1, 1> Cfg256;     // 256 x 256
// us of a round and a 128-k block (rg::Shape), fitted to 28..2000 rows of 10240 -> 5120, 5120 -> 1024
// and 17408: over 1086 sizes (K 1024..17408, N 300..34816, 9..3000 rows) what they choose takes 0.6 %
// longer than the best schedule on average, at one size in a hundred 9 % or more (a 32 row tile takes
// longer than a 64 row one here: its stages leave LDS for one ahead)
constexpr rg::Shape kShapes[3] = {{64, 256, 3.0f, 1.5f, 1.55f, 1.0f}, {128, 256, 3.0f, 1.85f, 1.95f, 1.0f}, {256, 256, 3.0f, 3.3f, 3.5f, 1.0f}};

}  // namespace

PrefillPlan plan_gemm_q8(int M, int K, int N, int n_cu, bool pieces) {
    return rg::prefill_plan(kShapes, M, K, 1, &N, n_cu, pieces);
}

hipError_t launch_gemm_q8(const uint16_t* A, int lda, const uint8_t* W, void* C, int c_dtype, int ldc, int M, int K,
                          int N, hipStream_t s) {
    return rg::launch<Q8F16, Cfg64, Cfg128, Cfg256>(kShapes, (const _Float16*)A, lda, 1, &W, &C, c_dtype, &ldc, M, K, &N, s);
}

}  // namespace kata
