// int8 prefill path: activation quantisation and the int8 x trit GEMM with the per-group
// scale epilogue, ternary decode fused into the LDS tile load.
//
// quant_rows (shaders/prefill.metal:369-381): per (token m, group g of 128):
//   scale = amax > 0 ? amax/127 : 1; q = clamp(rint(x * (1/scale)), -127, 127);
//   SX[g*ldS + m] = scale.   IEEE fp32 division and round-half-even, bit-exact.
// gemm (shaders/prefill.metal:382-415): I = sum_{k in g} A8[m][k]*trit[n][k] (exact int32),
//   C[m][n] = sum_g float(I) * (d[n][g] * SX[g][m]) in fp32, groups ascending.
//
// Two kernels.  Tall (256 x 128 C tiles): 12 waves, 8 consumers on v_mfma_i32_32x32x32_i8, two
// per SIMD, and 4 producers that copy A by DMA and decode weights into LDS (gemm_tile.h), whole
// tiles per CU, then K pieces summed by a second kernel.  A stage is one 128-group; the
// producers also stage the group's row scales (A side) and column scales (decoded weights) in
// LDS, and consumers fold each 32 x 32 tile's exact group sum into fp32 right after its four
// MFMAs, groups ascending.  Short (32, 64 and 128 rows): every wave decodes its weights into
// MFMA registers on the skeleton of the fp16 GEMM (gemm_reg.h); launch_gemm_i8 has the rule.
#include "common.h"
#include "launch.h"
#include "gemm_ptq1_copy.h"
#include "gemm_tile.h"
#include <utility>

namespace kata {

namespace {

// max over the 16 lanes of a DPP row
__device__ inline float row16_max(float a) {
    a = fmaxf(a, __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, a), 0xb1, 0xf, 0xf, false)));
    a = fmaxf(a, __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, a), 0x4e, 0xf, 0xf, false)));
    a = fmaxf(a, __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, a), 0x141, 0xf, 0xf, false)));
    a = fmaxf(a, __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, a), 0x140, 0xf, 0xf, false)));
    return a;
}

// One (token, group) per 16 lanes (a DPP row), 8 elements per lane from one 16-byte load;
// groups numbered token-major, 16 per 256-thread workgroup.
__global__ __launch_bounds__(256) void k_quant_rows(const _Float16* __restrict__ X, int8_t* __restrict__ Q,
                                                    float* __restrict__ SX, int M, int K, int ldS) {
    const int G = K / kGroup;
    const int gi = blockIdx.x * 16 + (threadIdx.x >> 4), sub = threadIdx.x & 15;
    if (gi >= M * G) return;                     // whole DPP rows drop out together
    const int m = gi / G, g = gi - m * G;
    const size_t o = (size_t)m * K + (size_t)g * kGroup + 8 * sub;
    const uint4 raw = *(const uint4*)(X + o);
    const uint32_t rw[4] = {raw.x, raw.y, raw.z, raw.w};
    float v[8];
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const v2h h = __builtin_bit_cast(v2h, rw[i]);
        v[2 * i] = (float)h[0];
        v[2 * i + 1] = (float)h[1];
    }
    float mx = 0.0f;
#pragma unroll
    for (int i = 0; i < 8; i++) mx = fmaxf(mx, fabsf(v[i]));
    mx = row16_max(mx);
    const float scale = mx > 0.0f ? mx / 127.0f : 1.0f;
    const float inv = 1.0f / scale;
    uint32_t q[2] = {0u, 0u};
#pragma unroll
    for (int i = 0; i < 8; i++) {
        const float qf = fminf(fmaxf(rintf(v[i] * inv), -127.0f), 127.0f);
        q[i >> 2] |= (uint32_t)(uint8_t)(int8_t)qf << (8 * (i & 3));
    }
    *(uint2*)(Q + o) = make_uint2(q[0], q[1]);
    if (sub == 0) SX[(size_t)g * ldS + m] = scale;
}

// int8 trits (digit - 1) of the 4 bytes of w, in byte order: bytes 0, 1 at the digit of
// multiplier p3lo, bytes 2, 3 at p3hi.  The bytes go to 16-bit lanes (v_perm selector 0x0c is
// a zero byte); ((b * 3^n) mod 256) * 3 - 256 has the trit in its high byte (0xff, 0x00, 0x01).
__device__ inline uint32_t trits4(uint32_t w, uint32_t p3lo, uint32_t p3hi) {
    typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));
    u16x2 e = __builtin_bit_cast(u16x2, __builtin_amdgcn_perm(0u, w, 0x0c010c00u));
    u16x2 o = __builtin_bit_cast(u16x2, __builtin_amdgcn_perm(0u, w, 0x0c030c02u));
    e = (e * __builtin_bit_cast(u16x2, p3lo)) & (u16x2){0xff, 0xff};
    o = (o * __builtin_bit_cast(u16x2, p3hi)) & (u16x2){0xff, 0xff};
    e = e * (u16x2){3, 3} + (u16x2){0xff00, 0xff00};
    o = o * (u16x2){3, 3} + (u16x2){0xff00, 0xff00};
    return __builtin_amdgcn_perm(__builtin_bit_cast(uint32_t, o), __builtin_bit_cast(uint32_t, e), 0x07050301u);
}

using namespace gemm;
using rg::barrier_lds;
constexpr int kWStage = BN * 32;                     // staged packed bytes of one block of the tile rows
constexpr int kSxOff = kTileBytes + 2 * kWStage;     // [kABuf][BM] fp32 row scales (with the A buffers)
constexpr int kSwOff = kSxOff + kABuf * BM * 4;      // [2][BN] fp32 column scales (with the B buffers)
constexpr int kLdsBytes = kSwOff + 2 * BN * 4;

typedef int v16i __attribute__((ext_vector_type(16)));
// the value v of lane Q of the caller's 16-lane row (DPP row_newbcast)
template <int Q>
__device__ inline float row_bcast(float v) {
    return __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), 0x150 + Q, 0xf, 0xf, true));
}
// acc[q] += float(I[q]) * (w * sx[row of output q]), where lane 16 R + Q of the caller's
// 16-lane row R holds the row scale of output q = Q
// (the empty asm gives each call its own copy of sxv, so every broadcast is used once and
// becomes the DPP operand of its multiply instead of a move held across the column tiles)
template <int... Q>
__device__ inline void fold_tile(v16f& acc, const v16i& I, float w, float sxv, std::integer_sequence<int, Q...>) {
    asm volatile("" : "+v"(sxv));
    ((acc[Q] += (float)I[Q] * (w * row_bcast<Q>(sxv))), ...);
}

// Consumer waves (wave < kCW): wave w owns rows 32w..32w+31 and all 128 columns, 4 tiles of
// 32 x 32.  Per stage (one group of 128 k) the A fragments stay in registers; for each column
// tile j the int32 sum is 4 dependent v_mfma_i32_32x32x32_i8, then folded: acc += float(I) *
// (sw[n] * sx[m]), the row scale spread across the lanes by DPP.  The fold of tile j follows
// the MFMAs of tile j + 1.  A wave's VALU does not overlap its own MFMAs; with two consumers
// on each SIMD one's fold can run under the other's MFMAs (2.5 % faster than four consumers
// of 64 rows; 64 x 64 per wave, fewer LDS reads, gains nothing over it).
// Barriers: two before the first stage (the producers' first copies landed, stage 0 produced), one
// per stage (after the stage's last LDS read).
constexpr int kCW = 8;                   // consumer waves; each owns BM / kCW rows
constexpr int kRH = BM / kCW;             // rows per consumer wave
constexpr int kRT = kRH / 32;             // 32-row MFMA tiles per consumer wave
template <bool C_F16>
__device__ inline void consume_i8(uint8_t* smem, int wave, int lane, int nb, int job, const GemmJobs& J, float* ws,
                                  void* C, int ldc, int M, int m0, int n0, int R) {
    const int l32 = lane & 31, lh = lane >> 5;
    v16f acc[kRT][NT];
#pragma unroll
    for (int i = 0; i < kRT; i++)
#pragma unroll
        for (int j = 0; j < NT; j++)
#pragma unroll
            for (int q = 0; q < 16; q++) acc[i][j][q] = 0.0f;
    const int xs = (l32 >> 1) & 7;
    const uint32_t a_row = (uint32_t)(wave * kRH + l32) * ROWB, b_row = (uint32_t)l32 * ROWB;
    const float* sxs = (const float*)(smem + kSxOff) + wave * kRH + 8 * ((lane & 15) >> 2) + 4 * lh + (lane & 3);
    const float* sws = (const float*)(smem + kSwOff) + l32;
    barrier_lds();                           // the producers' first copies landed
    barrier_lds();                           // stage 0 produced
    for (int st = 0; st < nb; st++) {
        const uint8_t* at = tile_a(smem, st % kABuf) + a_row;
        const uint8_t* bt = tile_b(smem, st & 1) + b_row;
        v4i af[kRT][4];
#pragma unroll
        for (int i = 0; i < kRT; i++)
#pragma unroll
            for (int kk = 0; kk < 4; kk++) af[i][kk] = *(const v4i*)(at + i * 32 * ROWB + (((2 * kk + lh) ^ xs) << 4));
        float sxv[kRT];
#pragma unroll
        for (int i = 0; i < kRT; i++) sxv[i] = sxs[(st % kABuf) * BM + i * 32];
        float sw[NT];
#pragma unroll
        for (int j = 0; j < NT; j++) sw[j] = sws[(st & 1) * BN + j * 32];
        v16i I[2];
        v4i bfA[4], bfB[4];
        auto ldb = [&](int j, v4i (&bf)[4]) {
#pragma unroll
            for (int kk = 0; kk < 4; kk++) bf[kk] = *(const v4i*)(bt + j * 32 * ROWB + (((2 * kk + lh) ^ xs) << 4));
            if (j == NT - 1) barrier_lds();  // stage st + 1 produced; stage st's buffers free
        };
        auto mmi = [&](int i, int slot, v4i (&bf)[4]) {
#pragma unroll
            for (int q = 0; q < 16; q++) I[slot][q] = 0;
#pragma unroll
            for (int kk = 0; kk < 4; kk++)
                I[slot] = __builtin_amdgcn_mfma_i32_32x32x32_i8(af[i][kk], bf[kk], I[slot], 0, 0, 0);
        };
        auto fold = [&](int i, int j, int slot) {
            fold_tile(acc[i][j], I[slot], sw[j], sxv[i], std::make_integer_sequence<int, 16>());
        };
        // one 32-row tile: the fold of column tile j follows the MFMAs of tile j + 1
        auto step = [&](int j, v4i (&bn)[4]) {
            if (j + 1 < NT) {
                ldb(j + 1, bn);
                mmi(0, (j + 1) & 1, bn);
            }
            fold(0, j, j & 1);
        };
        static_assert(NT == 4, "the steps below cover four column tiles");
        ldb(0, bfA);
        mmi(0, 0, bfA);
        step(0, bfB);
        step(1, bfA);
        step(2, bfB);
        step(3, bfA);
    }
    // store: lane holds D[8(q/4) + 4(l/32) + q%4][l % 32] of each 32x32 tile
    if (job >= J.n_full) {
        float* P = ws + (size_t)(job - J.n_full) * (BM * BN);
#pragma unroll
        for (int i = 0; i < kRT; i++)
#pragma unroll
            for (int j = 0; j < NT; j++)
#pragma unroll
                for (int q = 0; q < 16; q++)
                    P[(wave * kRH + i * 32 + 8 * (q >> 2) + 4 * lh + (q & 3)) * BN + j * 32 + l32] = acc[i][j][q];
        return;
    }
#pragma unroll
    for (int i = 0; i < kRT; i++)
#pragma unroll
        for (int j = 0; j < NT; j++) {
            const int gc = j * 32 + l32;
            const int gn = n0 + gc;
#pragma unroll
            for (int q = 0; q < 16; q++) {
                const int gm = m0 + wave * kRH + i * 32 + 8 * (q >> 2) + 4 * lh + (q & 3);
                if (gm < M && gc < R) {
                    if (C_F16) ((_Float16*)C)[(size_t)gm * ldc + gn] = (_Float16)acc[i][j][q];
                    else ((float*)C)[(size_t)gm * ldc + gn] = acc[i][j][q];
                }
            }
        }
}

// Stage = one PTQ1_0 block (128 k).  Producer waves kCW..kCW+3: A stage copies (8 DMA per wave)
// plus the stage's row scales (one dword DMA per wave, rows 64 pw .. +63, clamped to M - 1),
// two stages ahead into three buffers; packed weight bytes of a block staged by DMA two
// blocks ahead; decode of the next stage into one of two B buffers.  Producer lane decodes
// half q = pw & 1 of tile row 64 (pw >> 1) + lane: chunks 0..3 (q = 0: dwords 0..3 at digits
// 0..3) or chunks 4..7 (q = 1: digit 4 of dwords 0..3, dwords 4, 5, the qh bytes).
template <bool C_F16>
__global__ __launch_bounds__(64 * (kCW + 4)) void k_gemm_ptq1_i8(const int8_t* __restrict__ A8, const float* __restrict__ SX,
                                                      int ldS, const uint8_t* __restrict__ W, void* __restrict__ C,
                                                      int ldc, float* __restrict__ ws, int M, int K, int N,
                                                      GemmJobs J) {
    extern __shared__ __align__(16) uint8_t smem[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int nbk = K >> 7;
    int job, tile, kb0, nb;
    gemm_job(J, nbk, job, tile, kb0, nb);
    const int m0 = (tile / J.G) * BM;
    const int n0 = (tile % J.G) * BN;
    const int R = min(BN, N - n0);
    const uint32_t row_bytes = (uint32_t)nbk * kBlockBytes;

    if (wave < kCW) {
        consume_i8<C_F16>(smem, wave, lane, nb, job, J, ws, C, ldc, M, m0, n0, R);
        return;
    }

    // ================= producers =================
    const int pw = wave - kCW;
    // an int8 row of 128 k has the byte layout of an fp16 stage row of 64 k
    const _Float16* Ah = (const _Float16*)(A8 + (size_t)kb0 * kGroup);
    const float* sxsrc = SX + (size_t)kb0 * ldS + min(m0 + 64 * pw + lane, M - 1);
    const uint32_t sx_lds = lds_addr(smem + kSxOff) + 256 * pw;
    auto issue_a = [&](int st) {
        gemm::issue_a(smem, pw, lane, Ah, K >> 1, M, m0, st, nb);
        dma4(sxsrc + (size_t)min(st, nb - 1) * ldS, sx_lds + (st % kABuf) * (BM * 4));
    };
    const int wrow = 64 * (pw >> 1) + lane, q = pw & 1;
    const bool wactive = wrow < R;
    uint8_t* Ws = smem + kTileBytes;                                  // [2 slots][2][BN][16 B]
    float* sws = (float*)(smem + kSwOff);
    const uint8_t* wsrc = W + (size_t)min(n0 + min(wrow, R - 1), N - 1) * row_bytes + (size_t)kb0 * kBlockBytes + 12 * q;
    auto issue_w = [&](int blk) {
        dma16(wsrc + (size_t)min(blk, nb - 1) * kBlockBytes,
              lds_addr(Ws + (blk & 1) * kWStage + q * (BN * 16) + (pw >> 1) * 1024));
    };
    uint32_t w[7];
    auto read_w = [&](int blk) {
        const uint8_t* slot = Ws + (blk & 1) * kWStage;
        const uint4 a = *(const uint4*)(slot + wrow * 16);           // bytes 0..15
        const uint4 c = *(const uint4*)(slot + BN * 16 + wrow * 16); // bytes 12..27
        w[0] = a.x; w[1] = a.y; w[2] = a.z; w[3] = a.w;
        w[4] = c.y; w[5] = c.z; w[6] = c.w;
    };
    auto decode = [&](int buf) {
        uint8_t* bt = tile_b(smem, buf);
        auto put = [&](int chunk, uint32_t x0, uint32_t x1, uint32_t x2, uint32_t x3) {
            *(uint4*)(bt + swz(wrow, chunk)) = make_uint4(x0, x1, x2, x3);
        };
        if (!wactive) {
            if (q == 0) sws[buf * BN + wrow] = 0.0f;
            return;
        }
        if (q == 0) {
#pragma unroll
            for (int c = 0; c < 4; c++)
                put(c, trits4(w[0], p3x2(c), p3x2(c)), trits4(w[1], p3x2(c), p3x2(c)), trits4(w[2], p3x2(c), p3x2(c)),
                    trits4(w[3], p3x2(c), p3x2(c)));
            sws[buf * BN + wrow] = half_bits_to_float(w[6] >> 16);
        } else {
            put(4, trits4(w[0], p3x2(4), p3x2(4)), trits4(w[1], p3x2(4), p3x2(4)), trits4(w[2], p3x2(4), p3x2(4)),
                trits4(w[3], p3x2(4), p3x2(4)));
            put(5, trits4(w[4], p3x2(0), p3x2(0)), trits4(w[5], p3x2(0), p3x2(0)), trits4(w[4], p3x2(1), p3x2(1)),
                trits4(w[5], p3x2(1), p3x2(1)));
            put(6, trits4(w[4], p3x2(2), p3x2(2)), trits4(w[5], p3x2(2), p3x2(2)), trits4(w[4], p3x2(3), p3x2(3)),
                trits4(w[5], p3x2(3), p3x2(3)));
            const uint32_t qh = __builtin_amdgcn_perm(0u, w[6], 0x01000100u);   // (qh0, qh1, qh0, qh1)
            put(7, trits4(w[4], p3x2(4), p3x2(4)), trits4(w[5], p3x2(4), p3x2(4)), trits4(qh, p3x2(0), p3x2(1)),
                trits4(qh, p3x2(2), p3x2(3)));
        }
    };
    // Vector-memory order of a producer (all LDS copies, counted by the waits below):
    // W(b+2) then A(b+2) (9 copies) per iteration; the wait before the barrier that ends
    // iteration b leaves only A(b+2) in flight, so batch b+1 and block b+2 have landed.
    issue_w(0);
    issue_w(1);
    issue_a(0);
    issue_a(1);
    __builtin_amdgcn_s_waitcnt((9 & 15) | ((9 >> 4) << 14) | (7 << 4) | (15 << 8));       // blocks 0, 1, batch 0
    barrier_lds();
    read_w(0);
    decode(0);
    barrier_lds();
    for (int b = 0; b < nb; b++) {
        // consumers on stage b; produce stage b + 1 into B buffer (b + 1) & 1
        if (b + 1 < nb) read_w(b + 1);
        issue_w(b + 2);                          // into the slot read_w(b) freed
        issue_a(b + 2);
        if (b + 1 < nb) decode((b + 1) & 1);
        __builtin_amdgcn_s_waitcnt((9 & 15) | ((9 >> 4) << 14) | (7 << 4) | (15 << 8));   // batch b+1, block b+2
        barrier_lds();
    }
}

// ---------------------------------------------------------------------------------------
// Short tiles (32, 64 or 128 rows by 256 columns), on the skeleton of the fp16 GEMM
// (gemm_reg.h): wave w owns all rows and columns 32w..32w+31, and each lane decodes the trits
// of its own column straight into the MFMA's B registers.  A stage is one 128-group: its A
// rows (128 bytes, the byte layout of an fp16 stage of 64 k), its row scales, and four
// 32-k steps of v_mfma_i32_32x32x32_i8; the finished int32 tiles are folded into fp32 (groups
// ascending, the tall kernel's expression) after the next group's first decode.  The tall kernel computes 256 rows whatever their
// number: 28 / 41 / 100 rows of 5120 -> 17408 54.5 / 54.6 / 56.2 -> 25.4 / 29.8 / 40.0 us, of 17408 -> 5120
// 42.0 / 42.5 / 43.4 -> 23.9 / 26.9 / 37.  From about 150 rows it is the faster one (200 rows 57.8
// against 64): here every 128-row tile decodes its weights and folds 3 instructions per output
// and group beside them (about 330 vector instructions per 16 MFMAs).
namespace short_i8 {

using rg::lds_ld;
using rg::u16x2;
using rg::u32x2;
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

template <int MT_>
struct Cfg {
    static constexpr int MT = MT_, NT = 1, NWR = 1, NWC = 8, WAVES = 8, THREADS = 512;
    static constexpr int BM = 32 * MT, BN = 256, DA = 2, DW = 2, ABUF = DA + 1;
    static constexpr int ASTAGE = BM * 128;                      // A bytes of a stage
    static constexpr int SXROWS = BM < 64 ? 64 : BM;             // row scales of a stage
    static constexpr int NA = BM * 8 >= THREADS ? BM * 8 / THREADS : 1;
    static constexpr int kSx = ABUF * ASTAGE, kW = kSx + ABUF * SXROWS * 4;
    static constexpr int kLds = kW + (DW + 1) * BN * 64;
};

// B operand of 32-k step kk (16 consecutive k per lane: chunk 2 kk + lh of the block): digit 2 kk +
// lh of qs bytes 0..15 for kk < 2; then digit 4 of those (lh = 0) or digits 0, 1 of bytes 16..23;
// then digits 2, 3 of bytes 16..23 (lh = 0) or their digit 4 and the qh bytes.
struct Trits : Ptq1Copy {
    int lh;
    uint32_t wn[7], w4, w5, w6;
    u16x2 m[8];                                    // remainders of bytes 0..15
    float d;

    template <class C, int J>
    __device__ inline void read(int g, int slot, int nb) {
        const uint32_t p = rd + slot * slot_bytes<C>();
        if constexpr (J == 0) {
            const u32x4 a = lds_ld<u32x4>(p + piece(0));
            const uint32_t q = p + piece(1) + (2 * g + 1 == nb ? 4u : 0u);
#pragma unroll
            for (int i = 0; i < 4; i++) wn[i] = a[i];
#pragma unroll
            for (int i = 0; i < 3; i++) wn[4 + i] = lds_ld<uint32_t>(q + 4 * i);
        } else {
            wn[0] = lds_ld<uint32_t>(p + piece(1) + 12);
            const u32x4 a = lds_ld<u32x4>(p + piece(2));
            const u32x2 b = lds_ld<u32x2>(p + piece(3) + 8);
#pragma unroll
            for (int i = 0; i < 4; i++) wn[1 + i] = a[i];
            wn[5] = b[0];
            wn[6] = b[1];
        }
    }
    // unpack the block read ahead; its scale
    __device__ inline float begin() {
        const u16x2 mul = __builtin_bit_cast(u16x2, lh ? p3x2(1) : p3x2(0));
#pragma unroll
        for (int i = 0; i < 4; i++) {
            m[2 * i] = (bytes01(wn[i]) * mul) & (u16x2){0xff, 0xff};
            m[2 * i + 1] = (bytes23(wn[i]) * mul) & (u16x2){0xff, 0xff};
        }
        w4 = wn[4];
        w5 = wn[5];
        w6 = wn[6];
        return half_bits_to_float(w6 >> 16);
    }
    template <int kk>
    __device__ inline v4i chunk() {
        const u16x2 lo8 = {0xff, 0xff}, nine = {9, 9};
        u16x2 r[8];                                // the digits' remainders, four bytes per dword pair
#pragma unroll
        for (int j = 0; j < 8; j++) {
            const uint32_t w = j & 2 ? w5 : w4;
            const u16x2 n = j & 1 ? bytes23(w) : bytes01(w);
            auto pick = [&](u16x2 a, u16x2 b) {    // a for lh = 0, b for lh = 1
                return __builtin_bit_cast(u16x2, lh ? __builtin_bit_cast(uint32_t, b) : __builtin_bit_cast(uint32_t, a));
            };
            auto mulc = [&](int a, int b) { return __builtin_bit_cast(u16x2, lh ? p3x2(b) : p3x2(a)); };
            if constexpr (kk < 2) {
                if constexpr (kk == 1) m[j] = (m[j] * nine) & lo8;
                r[j] = m[j];
            } else if constexpr (kk == 2) {
                r[j] = (pick(m[j], n) * mulc(2, j < 4 ? 0 : 1)) & lo8;
            } else {
                r[j] = j < 4 ? (n * mulc(2, 4)) & lo8 : (pick(n, bytes01(w6)) * mulc(3, j - 4)) & lo8;
            }
        }
        v4i o;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            // 3 m - 256 has the trit (digit - 1) in its high byte
            const u16x2 a = r[2 * i] * (u16x2){3, 3} + (u16x2){0xff00, 0xff00};
            const u16x2 b = r[2 * i + 1] * (u16x2){3, 3} + (u16x2){0xff00, 0xff00};
            o[i] = (int)__builtin_amdgcn_perm(__builtin_bit_cast(uint32_t, b), __builtin_bit_cast(uint32_t, a), 0x07050301u);
        }
        return o;
    }
};

template <class C, bool C_F16>
__global__ __launch_bounds__(512, 2) void k_gemm_i8_short(const int8_t* __restrict__ A8, const float* __restrict__ SX,
                                                          int ldS, rg::Mats P, float* __restrict__ ws, int M, int K,
                                                          GemmJobs J) {
    constexpr int MT = C::MT, DA = C::DA, DW = C::DW, NA = C::NA, ABUF = C::ABUF, SPG = 2;
    constexpr int NW = Ptq1Copy::copies<C>();
    static_assert((DW - 1) * SPG >= DA, "a group's copies, spread over two stages, land in time");
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l32 = lane & 31, lh = lane >> 5;
    const int nbk = K >> 7;
    int job, tile, kb0, nb;
    gemm_job(J, nbk, job, tile, kb0, nb);
    const int m0 = (tile / J.G) * C::BM, mi = rg::mat_of(P, tile % J.G), n0 = (tile % J.G - P.g0[mi]) * C::BN;
    const int N = P.N[mi];
    const int ng = (nb + 1) / 2;

    // A copies: instruction i copies rows 64 i .. + 63 of a stage (32-row tiles: the upper waves
    // repeat the lower ones'), chunk c of row r at c ^ ((r >> 1) & 7); limited to row M - 1
    const int arow = (tid >> 3) & (C::BM < 64 ? 31 : 63);
    const uint32_t avo = (uint32_t)arow * (uint32_t)K + (uint32_t)(((tid & 7) ^ ((arow >> 1) & 7)) << 4);
    const uint32_t a_lds = 1024u * (C::BM < 64 ? wave & 3 : wave);
    auto issue_a = [&](int st) {
        const int buf = st % ABUF;
        const int8_t* ko = A8 + (size_t)(kb0 + min(st, nb - 1)) * 128;
#pragma unroll
        for (int i = 0; i < NA; i++) {
            const int r0 = min(m0 + i * 64, M - 1);
            const uint32_t lim = M - 1 - r0 < 64 ? (uint32_t)(M - 1 - r0) * (uint32_t)K + 112u : 0xffffffffu;
            dma16(ko + (size_t)r0 * K, min(avo, lim), a_lds + buf * C::ASTAGE + i * 8192);
        }
        // the stage's row scales, one dword per lane: wave w rows 64 (w % (SXROWS / 64)) + lane
        const int rg64 = wave & (C::SXROWS / 64 - 1);
        dma4(SX + (size_t)(kb0 + min(st, nb - 1)) * ldS, 4u * (uint32_t)min(m0 + 64 * rg64 + lane, M - 1),
                 C::kSx + buf * (C::SXROWS * 4) + 256u * rg64);
    };
    Trits dec;
    dec.lh = lh;
    dec.template init_copy<C>(P.W[mi], nbk, kb0, nb, n0, N, tid, wave, wave, l32, C::kW);
    auto issue_w = [&](int g, int i0, int i1) { dec.template issue<C>(min(g, ng - 1), g % (DW + 1), i0, i1); };

    v16f acc[MT];
#pragma unroll
    for (int i = 0; i < MT; i++)
#pragma unroll
        for (int q = 0; q < 16; q++) acc[i][q] = 0.0f;
    // copies that may fly when stage sp is awaited: the DA - 1 stages after it and the weight parts
    // issued with them
    auto vm_of = [](int sp) constexpr {
        int n = (DA - 1) * (NA + 1);
        for (int j = sp - DA + 1; j < sp; j++) n += ((j + SPG) % SPG + 1) * NW / SPG - (j + SPG) % SPG * NW / SPG;
        return n;
    };
    rg::unroll<DW * SPG>([&](auto ic) {
        constexpr int j = decltype(ic)::value - DW * SPG, sp = (j + DW * SPG) % SPG;
        issue_w((j - sp) / SPG + DW, sp * NW / SPG, (sp + 1) * NW / SPG);
        if constexpr (j >= -DA) issue_a(j + DA);
    });
    const uint32_t a_row = (uint32_t)l32 * 128u + (uint32_t)((lh ^ ((l32 >> 1) & 7)) << 4);
    const uint32_t sx_row = C::kSx + 4u * (8 * ((lane & 15) >> 2) + 4 * lh + (lane & 3));
    v4i af[2][MT], bf[2];
    auto frags = [&](int kk, int buf, v4i (&f)[MT]) {
        const uint32_t at = buf * C::ASTAGE + (a_row ^ (uint32_t)(kk << 5));
#pragma unroll
        for (int i = 0; i < MT; i++) f[i] = lds_ld<v4i>(at + i * 4096);
    };
    rg::wait_vm<vm_of(0)>();
    rg::barrier_lds();
    dec.template read<C, 0>(0, 0, nb);
    frags(0, 0, af[0]);
    float d = dec.begin();
    bf[0] = dec.template chunk<0>();
    int s = 0, abuf = 0;
    v16i I[MT];
    float sx[MT];
    static_assert(NW == 2 && vm_of(0) == vm_of(1), "one weight copy per stage: every stage waits alike");
    for (int b = 0; b < nb; b++) {
        const int g = b >> 1;
        if (b & 1) dec.template read<C, 0>(g + 1, (g + 1) % (DW + 1), nb);      // the next block's words
        else dec.template read<C, 1>(g, g % (DW + 1), nb);
        rg::unroll<4>([&](auto kc) {
            constexpr int kk = decltype(kc)::value, cur = kk & 1, nxt = cur ^ 1;
            if constexpr (kk == 3) {                 // the next stage has landed, this one's fragments are held
                ++s;
                abuf = abuf + 1 == ABUF ? 0 : abuf + 1;
                rg::wait_vm<vm_of(0)>();
                rg::barrier_lds();
            }
            __builtin_amdgcn_sched_barrier(0);
            frags((kk + 1) % 4, abuf, af[nxt]);
            if constexpr (kk == 0) {
#pragma unroll
                for (int i = 0; i < MT; i++) sx[i] = lds_ld<float>(sx_row + abuf * (C::SXROWS * 4) + i * 128);
            }
#pragma unroll
            for (int i = 0; i < MT; i++) {
                if constexpr (kk == 0) {
#pragma unroll
                    for (int q = 0; q < 16; q++) I[i][q] = 0;
                }
                I[i] = __builtin_amdgcn_mfma_i32_32x32x32_i8(af[cur][i], bf[cur], I[i], 0, 0, 0);
            }
            const float dg = d;
            if constexpr (kk == 3) d = dec.begin();
            bf[nxt] = dec.template chunk<(kk + 1) % 4>();
            if constexpr (kk == 3) {
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int i = 0; i < MT; i++) fold_tile(acc[i], I[i], dg, sx[i], std::make_integer_sequence<int, 16>());
            }
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (kk == 0) {
                if (b & 1) issue_w(g + DW, 1, 2);
                else issue_w(g + DW, 0, 1);
            }
            if constexpr (kk == 1) issue_a(s + DA);
        });
    }
    rg::wait_vm<0>();

    const int gc = wave * 32 + l32;                  // tile column
    if (job >= J.n_full) {
        float* T = ws + (size_t)(job - J.n_full) * (C::BM * C::BN);
#pragma unroll
        for (int i = 0; i < MT; i++)
#pragma unroll
            for (int q = 0; q < 16; q++) {
                const int r = i * 32 + 8 * (q >> 2) + 4 * lh + (q & 3);
                if (m0 + r < M) T[r * C::BN + gc] = acc[i][q];
            }
        return;
    }
    void* Cp = P.C[mi];
    const int ldc = P.ldc[mi], gn = n0 + gc;
#pragma unroll
    for (int i = 0; i < MT; i++)
#pragma unroll
        for (int q = 0; q < 16; q++) {
            const int gm = m0 + i * 32 + 8 * (q >> 2) + 4 * lh + (q & 3);
            if (gm < M && gn < N) {
                if (C_F16) ((_Float16*)Cp)[(size_t)gm * ldc + gn] = (_Float16)acc[i][q];
                else ((float*)Cp)[(size_t)gm * ldc + gn] = acc[i][q];
            }
        }
}

// us of a round and a 128-group (see rg::Shape and plan below)
constexpr rg::Shape kShapes[3] = {{32, 256, 3.0f, 1.02f, 1.02f, 1.0f}, {64, 256, 3.0f, 1.3f, 1.3f, 1.0f}, {128, 256, 3.0f, 1.9f, 1.9f, 1.0f}};

template <class C>
hipError_t launch_cfg(const int8_t* A8, const float* SX, int ldS, const rg::Mats& P, float* ws, int c_dtype, bool v4, int M,
                      int K, const GemmJobs& J, hipStream_t s) {
    static_assert(C::kLds <= 160 * 1024, "LDS");
    static const hipError_t attr = [] {
        hipError_t e = hipFuncSetAttribute((const void*)k_gemm_i8_short<C, true>, hipFuncAttributeMaxDynamicSharedMemorySize, C::kLds);
        if (e == hipSuccess)
            e = hipFuncSetAttribute((const void*)k_gemm_i8_short<C, false>, hipFuncAttributeMaxDynamicSharedMemorySize, C::kLds);
        return e;
    }();
    if (attr != hipSuccess) return attr;
    if (c_dtype == 1)
        hipLaunchKernelGGL((k_gemm_i8_short<C, true>), dim3(J.n_jobs), dim3(512), C::kLds, s, A8, SX, ldS, P, ws, M, K, J);
    else
        hipLaunchKernelGGL((k_gemm_i8_short<C, false>), dim3(J.n_jobs), dim3(512), C::kLds, s, A8, SX, ldS, P, ws, M, K, J);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    return rg::launch_pieces_sum<C::BM, C::BN>(ws, P, c_dtype, v4, M, J, s);
}

}  // namespace short_i8

// The kernel of a call (k: of short_i8::kShapes, or kTall) and its schedule, with K pieces or
// (pieces false) whole tiles only: the short tiles, whose row offsets are 32-bit, where the cost model has
// them cheaper than the tall kernel.  That: whole rounds of 256 x 128 tiles at 4 + 1.33 us per group,
// then K pieces, whose sum costs 7 us and their bytes (whole tiles out, real rows back) at 6.2 TB/s.
// Fitted together with kShapes to every schedule of 1086 sizes (K 1024..17408, N 300..34816, 9..3000
// rows): what is chosen takes on average 0.4 %, and at one size in a hundred 9 % or more, longer than
// the best, and is slower than the tall kernel by more than 3 % at 7 sizes, 9 % at most.  (Fitted
// to a few shapes, with pieces at 4 us and 4 TB/s: 0.7 %, 13 %; 15 sizes, 18 %: 200 rows of 10240 ->
// 2500 30.2 us against 25.2, of 5120 -> 5120 31.9 / 27.4; 1000 of 1024 -> 17408 61.9 / 52.7.)
constexpr int kTall = 3;
rg::Plan plan(int M, int K, int N, int n_cu, bool pieces) {
    const int nbk = K / kGroup;
    GemmJobs J = plan_gemm_jobs(M, N, K, BM, BN, n_cu);   // one workgroup per CU
    if (!pieces) {
        const int T = J.n_full + (J.n_jobs - J.n_full) / J.S;
        J = {J.G, T, 1, T};
    }
    const int rem = J.n_jobs - J.n_full;
    const double rows = (double)M / ((M + BM - 1) / BM);                    // real rows per tile
    double us = (J.n_full + n_cu - 1) / n_cu * (4.0 + nbk * 1.33);
    if (rem) us += 4.0 + (nbk + J.S - 1) / J.S * 1.33 + 7.0 + rem * BN * (BM + rows) * 4.0 / 6.2e6;
    if (K <= (1 << 23)) {
        const rg::Plan t = rg::choose(short_i8::kShapes, M, (N + 255) / 256, nbk, n_cu, pieces);
        if (t.us < us) return t;
    }
    return {J, (float)us, kTall};
}

}  // namespace

hipError_t launch_quant_rows(const uint16_t* X, int8_t* Q, float* SX, int M, int K, int ldS, hipStream_t s) {
    const long groups = (long)M * (K / kGroup);
    hipLaunchKernelGGL(k_quant_rows, dim3((unsigned)((groups + 15) / 16)), dim3(256), 0, s, (const _Float16*)X, Q, SX,
                       M, K, ldS);
    return hipGetLastError();
}

PrefillPlan plan_gemm_i8(int M, int K, int N, int n_cu, bool pieces) {
    const rg::Plan p = plan(M, K, N, n_cu, pieces);
    return p.k == kTall ? rg::prefill_plan(p.J, BM, BN)
                        : rg::prefill_plan(p.J, short_i8::kShapes[p.k].bm, short_i8::kShapes[p.k].bn);
}

hipError_t launch_gemm_i8(const int8_t* A8, const float* SX, int ldS, const uint8_t* W, void* C, int c_dtype,
                          int ldc, int M, int K, int N, hipStream_t s) {
    // the dynamic-LDS limit of both instantiations, raised once per process (a function-local
    // static: thread-safe initialisation)
    static const hipError_t attr = [] {
        hipError_t e = hipFuncSetAttribute((const void*)k_gemm_ptq1_i8<true>, hipFuncAttributeMaxDynamicSharedMemorySize, kLdsBytes);
        if (e == hipSuccess)
            e = hipFuncSetAttribute((const void*)k_gemm_ptq1_i8<false>, hipFuncAttributeMaxDynamicSharedMemorySize, kLdsBytes);
        return e;
    }();
    if (attr != hipSuccess) return attr;
    int n_cu = 0;
    float* ws = nullptr;
    hipError_t e = gemm_device(false, s, &n_cu, &ws);
    if (e != hipSuccess) return e;
    rg::Plan p = plan(M, K, N, n_cu, true);
    if (p.J.n_jobs > p.J.n_full && gemm_device(true, s, &n_cu, &ws) != hipSuccess) {
        // no workspace (the stream's first call is captured, or memory is short): whole tiles
        (void)hipGetLastError();
        p = plan(M, K, N, n_cu, false);
    }
    rg::Mats P{};
    P.W[0] = W;
    P.C[0] = C;
    P.N[0] = N;
    P.ldc[0] = ldc;
    for (int i = 1; i <= rg::kMaxMats; i++) P.g0[i] = 0x7fffffff;
    const bool v4 = N % 4 == 0 && ldc % 4 == 0 && ((uintptr_t)C & 15) == 0;
    switch (p.k) {
        case 0: return short_i8::launch_cfg<short_i8::Cfg<1>>(A8, SX, ldS, P, ws, c_dtype, v4, M, K, p.J, s);
        case 1: return short_i8::launch_cfg<short_i8::Cfg<2>>(A8, SX, ldS, P, ws, c_dtype, v4, M, K, p.J, s);
        case 2: return short_i8::launch_cfg<short_i8::Cfg<4>>(A8, SX, ldS, P, ws, c_dtype, v4, M, K, p.J, s);
    }
    if (c_dtype == 1)
        hipLaunchKernelGGL(k_gemm_ptq1_i8<true>, dim3(p.J.n_jobs), dim3(64 * (kCW + 4)), kLdsBytes, s, A8, SX, ldS, W, C, ldc, ws,
                           M, K, N, p.J);
    else
        hipLaunchKernelGGL(k_gemm_ptq1_i8<false>, dim3(p.J.n_jobs), dim3(64 * (kCW + 4)), kLdsBytes, s, A8, SX, ldS, W, C, ldc,
                           ws, M, K, N, p.J);
    e = hipGetLastError();
    if (e != hipSuccess) return e;
    return rg::launch_pieces_sum<BM, BN>(ws, P, c_dtype, v4, M, p.J, s);
}

}  // namespace kata
