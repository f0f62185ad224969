// Exact fp16 prefill GEMM, the PTQ1_0 weights decoded into the MFMA's registers.
//
// Semantics (shaders/prefill.metal:31-41 after k_expand_ptq1_v2, :472-479):
//   C[m][n] = sum_k A[m][k] * half(trit[n][k] * d[n][k/128]),  fp16 x fp16 -> fp32.
// half(trit*d) is exact, so every product term equals the reference's; only the fp32
// summation order differs (tolerance-based parity).
//
// Design (MI355X-first; the reference expands every matrix to a 178 MB fp16 stage first): the
// skeleton of gemm_reg.h with the PTQ1_0 decode below.  No fp16 weight copy exists, in HBM or in
// LDS: a lane turns the packed bytes of its own column into the MFMA's B registers.
//
// What bounds it (K = 5120, N = 17408; before: 256 x 128 tiles whose producer waves wrote decoded
// weights into LDS):
//  * Many rows: at 7300 every CU runs 256 x 256 tiles, the clock falls to 1.7 - 2.0 of 2.4 GHz, and of
//    a busy CU's cycles 62 - 65 % are MFMAs and 23 % other vector instructions, which with one wave per
//    SIMD hardly overlap: instructions and LDS bytes per MFMA count, not their latency.  One wave per
//    SIMD with 256 x 64 of C (2.8 vector instructions and half an LDS fragment read per MFMA) 1337 ->
//    1100 us (1.18 PFLOP/s); a plain fp16 library product of the shape takes 1150.  Two waves per
//    SIMD of 128 x 64: 1118; of 128 x 32: 1220.
//  * A hundred to a few hundred rows: vector instructions and MFMAs of the two waves of a SIMD
//    overlap only in part (the stage barrier keeps them in step): 128 x 256 tiles, 200 rows
//    80 -> 61 us.
//  * Up to 64 rows: the decode (3 vector instructions per weight, each weight once per launch),
//    waits (a third of the waves' time) and the fixed 3 us to the first MFMA; short tiles instead of rows of padding: 41
//    rows 78 -> 28 us, 28 rows 78 -> 24 us.
// Measured and not kept: trits from a conflict-free LDS table (half the vector instructions,
// as many LDS cycles more: equal at 41 rows, 1.2x slower at 7300); waves of a SIMD in opposite
// decode / multiply phases (1.1 - 1.3x slower: two barriers a unit); fragments read three or
// seven steps ahead (equal).
#include "common.h"
#include "launch.h"

#include <algorithm>
#include <type_traits>

#include "gemm_ptq1_copy.h"

namespace kata {

namespace {

using rg::u16x2;

// PTQ1_0 weights as B operand registers.  Lane half lh of column c takes chunk 2 kk + lh (8
// consecutive k) of every 16-k step kk of a block: for kk < 5 digit kk of qs bytes 8 lh .. 8 lh
// + 7; for kk = 5, 6 digit 2 (kk - 5) + lh of bytes 16..23; for kk = 7 digit 4 of those (lh = 0)
// or the qh bytes, digit j for pair j (lh = 1).
struct Ptq1F16 : Ptq1Copy {
    static constexpr bool TWO_FORMS = true;

    uint32_t o_own0, o_p1, o_own10, o_own11, o_p2, o_p3;
    int lh;
    uint32_t wn[2][5];                            // next block's words: own half, bytes 16..27
    u16x2 m[2][4];                                // remainders of the digits taken so far
    uint32_t w4[2], w5[2], w6[2];
    v2h dd[2], S[2];

    template <class C>
    __device__ inline void init(const uint8_t* W, int nbk, int kb0, int nb, int n0, int N, int tid, int wave, int wc,
                                int l32, int lh_, uint32_t Ws) {
        init_copy<C>(W, nbk, kb0, nb, n0, N, tid, wave, wc, l32, Ws);
        lh = lh_;
        o_own0 = piece(0) + 8u * lh;
        o_p1 = piece(1);
        o_p2 = piece(2) + 12u;
        o_p3 = piece(3) + 8u;
        o_own10 = lh ? piece(2) + 4u : piece(1) + 12u;
        o_own11 = piece(2) + (lh ? 8u : 0u);
    }
    template <class C, int J>
    __device__ inline void read(int g, int slot, int nb) {
        const uint32_t p = rd + slot * slot_bytes<C>();
        auto word = [](uint32_t a) { return rg::lds_ld<uint32_t>(a); };
#pragma unroll
        for (int t = 0; t < C::NT; t++) {
            if constexpr (J == 0) {
                const uint32_t q = p + o_p1 + (2 * g + 1 == nb ? 4u : 0u) + t * 2048;
                const rg::u32x2 a = rg::lds_ld<rg::u32x2>(p + o_own0 + t * 2048);
                wn[t][0] = a.x;
                wn[t][1] = a.y;
                wn[t][2] = word(q);
                wn[t][3] = word(q + 4);
                wn[t][4] = word(q + 8);
            } else {
                wn[t][0] = word(p + o_own10 + t * 2048);
                wn[t][1] = word(p + o_own11 + t * 2048);
                wn[t][2] = word(p + o_p2 + t * 2048);
                wn[t][3] = word(p + o_p3 + t * 2048);
                wn[t][4] = word(p + o_p3 + 4 + t * 2048);
            }
        }
    }
    template <class C, int kb>
    __device__ inline void look(int) {}
    // Unpack the block read ahead.  True if a scale of the wave's columns is not below 1 in
    // magnitude (or not finite): the fast form of `value` needs d * 2^16 in fp16.
    template <class C>
    __device__ inline bool begin() {
        bool big = false;
#pragma unroll
        for (int t = 0; t < C::NT; t++) {
            m[t][0] = bytes01(wn[t][0]);
            m[t][1] = bytes23(wn[t][0]);
            m[t][2] = bytes01(wn[t][1]);
            m[t][3] = bytes23(wn[t][1]);
            w4[t] = wn[t][2];
            w5[t] = wn[t][3];
            w6[t] = wn[t][4];
            const uint32_t d2 = __builtin_amdgcn_perm(0u, w6[t], 0x03020302u);
            dd[t] = __builtin_bit_cast(v2h, d2);
            const v2h k = {(_Float16)256.0f, (_Float16)256.0f};
            S[t] = dd[t] * k * k;
            big |= (d2 & 0x7fffu) >= 0x3c00u;
        }
        return __any(big);
    }
    // fp16 of (digit - 1) * d for X = 3 m in 16-bit lanes, digit = X >> 8.  The digit's bits are
    // the subnormal digit * 2^-16, so one fma with d * 2^16 and -d is exact (4 vector
    // instructions per pair with the remainder update); with a scale of 1 or more the
    // value is picked by a byte permute.
    template <bool BIG>
    __device__ inline uint32_t value(u16x2 X, int t) {
        if constexpr (BIG) {
            const uint32_t db = __builtin_bit_cast(uint32_t, dd[t]);
            const u16x2 sel = (X >> (u16x2){8, 8}) * (u16x2){0x0202, 0x0202} + (u16x2){0x0100, 0x0100};
            return __builtin_amdgcn_perm(db, (db & 0xffffu) ^ 0x8000u, __builtin_bit_cast(uint32_t, sel));
        } else {
            const v2h dg = __builtin_bit_cast(v2h, X & (u16x2){0x300, 0x300});
            return __builtin_bit_cast(uint32_t, __builtin_elementwise_fma(dg, S[t], -dd[t]));
        }
    }
    // chunk of 16-k step kk of the block, column tile t; steps in order
    template <int kk, bool BIG>
    __device__ inline v8h chunk(int t) {
        const u16x2 three = {3, 3}, lo8 = {0xff, 0xff};
        uint32_t o[4];
#pragma unroll
        for (int j = 0; j < 4; j++) {
            u16x2 X;
            if constexpr (kk < 5) {
                X = m[t][j] * three;
                if constexpr (kk < 4) m[t][j] = X & lo8;
            } else if constexpr (kk == 5) {
                const u16x2 mul = __builtin_bit_cast(u16x2, lh ? p3x2(1) : p3x2(0));
                const uint32_t w = j < 2 ? w4[t] : w5[t];
                m[t][j] = ((j & 1 ? bytes23(w) : bytes01(w)) * mul) & lo8;
                X = m[t][j] * three;
            } else if constexpr (kk == 6) {
                m[t][j] = (m[t][j] * (u16x2){9, 9}) & lo8;
                X = m[t][j] * three;
            } else {
                const uint32_t src = lh ? __builtin_bit_cast(uint32_t, bytes01(w6[t])) : __builtin_bit_cast(uint32_t, m[t][j]);
                const u16x2 mul = __builtin_bit_cast(u16x2, lh ? p3x2(j) : p3x2(2));
                X = ((__builtin_bit_cast(u16x2, src) * mul) & lo8) * three;
            }
            o[j] = value<BIG>(X, t);
        }
        return __builtin_bit_cast(v8h, make_uint4(o[0], o[1], o[2], o[3]));
    }
};

//               MT NT WR WC  KS DA DW waves per SIMD
typedef rg::Cfg<8, 2, 1, 4, 64, 2, 1, 1> Cfg256;     // 256 x 256
typedef rg::Cfg<4, 1, 1, 8, 64, 2, 1, 2> Cfg128;     // 128 x 256
typedef rg::Cfg<2, 1, 1, 8, 128, 2, 2, 2> Cfg64;     // 64 x 256
typedef rg::Cfg<1, 1, 1, 8, 128, 2, 2, 2> Cfg32;     // 32 x 256
// us of a round and a 128-k block (rg::Shape), fitted to 1405 sizes (K 1024..17408, N 300..34816, 9..3000
// rows): what they choose takes 0.9 % longer than the best schedule on average, and 13 % or more at one
// size in a hundred.  Before, fitted to the model's shapes with tiles of 128 and 256 rows at 1.42 - 2.05
// and 2.85 - 3.5 us by the busy CUs: 2.0 % and 19 % (1000 rows of 4096 -> 17408 173 us in 2.1 rounds of
// 128-row tiles, against 149 in two and a split rest).
// Pieces of fewer than 8 blocks only from 10 % by the model (from any gain: 0.7 % and 8 %): of a gain that
// it has, up to 13 % of the time does not come (64 rows of 4096 -> 4096 17.2 us with them, 17.0 without,
// by the model 15.4 / 17.4), and below that the sums stay in longer pieces.  With / without, us: 25
// rows of 1920 -> 1500 9.5 / 17.7, of 5120 -> 1024 10.0 / 13.7.
constexpr int kBN = 256;
constexpr float kShort = 0.9f;
constexpr rg::Shape kShapes[4] = {{32, kBN, 3.0f, 1.04f, 1.04f, kShort}, {64, kBN, 3.0f, 1.15f, 1.15f, kShort},
                                  {128, kBN, 3.0f, 1.48f, 1.48f, kShort}, {256, kBN, 7.0f, 2.6f, 2.6f, kShort}};

}  // namespace

hipError_t gemm_device(bool need_ws, hipStream_t s, int* n_cu, float** ws) {
    hipError_t e = device_cu_count(n_cu);
    if (e != hipSuccess) return e;
    *ws = nullptr;
    if (!need_ws) return hipSuccess;
    void* p = nullptr;
    e = stream_buffer(kBufGemmPieces, (size_t)*n_cu * rg::kPieceFloats * sizeof(float), s, &p);
    *ws = (float*)p;
    return e;
}

PrefillPlan plan_gemm_f16(int M, int K, int count, const int* N, int n_cu, bool pieces) {
    return rg::prefill_plan(kShapes, M, K, count, N, n_cu, pieces);
}

hipError_t launch_gemm_f16_multi(const uint16_t* A, int lda, int count, const uint8_t* const* W, void* const* C, int c_dtype,
                                 const int* ldc, int M, int K, const int* N, hipStream_t s) {
    return rg::launch<Ptq1F16, Cfg32, Cfg64, Cfg128, Cfg256>(kShapes, (const _Float16*)A, lda, count, W, C, c_dtype, ldc, M, K, N, s);
}

hipError_t launch_gemm_f16(const uint16_t* A, int lda, const uint8_t* W, void* C, int c_dtype, int ldc,
                           int M, int K, int N, hipStream_t s) {
    return launch_gemm_f16_multi(A, lda, 1, &W, &C, c_dtype, &ldc, M, K, &N, s);
}

}  // namespace kata
