// Prefill GEMM skeleton with the weights decoded straight into MFMA operand registers
// (gemm_f16.hip: PTQ1_0, gemm_q8.hip: Q8_0): C[M][N] = A[M][K] * W[N][K]^T, fp16 x fp16 -> fp32.  The
// int8 GEMM's tiles of up to 128 rows (gemm_i8.hip) have their own loop over the copies, waits and
// layouts here, and all of them share the cost model and the sum of K pieces.
//
// A workgroup of NWR x NWC waves computes a BM x BN tile of C; wave (wr, wc) owns 32 MT rows
// and 32 NT columns as MT x NT tiles of v_mfma_f32_32x32x16_f16.  Lane l of the B operand
// holds 8 consecutive k of column l % 32, so a lane decodes the weights of its own column and
// no decoded weight goes through LDS: LDS traffic is the A fragments, 16 MT bytes per lane for
// MT x NT MFMAs, and the packed weight bytes.
//  * A advances in stages of KS k, copied into LDS by DMA DA stages ahead (DA + 1 buffers);
//    a row of a stage is KS / 8 chunks of 16 B, chunk c stored at c ^ swizzle(row).
//  * The packed weight bytes of a group of blocks of the tile's BN weight rows are copied
//    into LDS by DMA DW groups ahead; a lane reads the words of its columns one block ahead.
//  * All vector-memory instructions of the loop are LDS copies, which the compiler cannot
//    count; the waits below do, so every wave issues the same number per stage (copies past
//    the end repeat the last stage or group).
#pragma once
#include <algorithm>
#include <array>
#include <utility>

#include "common.h"
#include "gemm_sched.h"
#include "launch.h"
#include "lds_dma.h"

namespace kata {
namespace rg {

typedef float v16f __attribute__((ext_vector_type(16)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));

// The 1..4 matrices of one launch (same A): matrix i is W[i] (N[i] rows), its output C[i] with
// row stride ldc[i]; column groups [g0[i], g0[i + 1]) of BN columns are its.
constexpr int kMaxMats = 4;
struct Mats {
    const uint8_t* W[kMaxMats];
    void* C[kMaxMats];
    int N[kMaxMats];
    int ldc[kMaxMats];
    int g0[kMaxMats + 1];
};
// the matrix of column group cg (entries past the last matrix start past every group)
__device__ inline int mat_of(const Mats& P, int cg) { return (cg >= P.g0[1]) + (cg >= P.g0[2]) + (cg >= P.g0[3]); }

template <int MT_, int NT_, int NWR_, int NWC_, int KS_, int DA_, int DW_, int WPE_>
struct Cfg {
    static constexpr int MT = MT_, NT = NT_, NWR = NWR_, NWC = NWC_, KS = KS_, DA = DA_, DW = DW_, WPE = WPE_;
    static constexpr int WAVES = NWR * NWC, THREADS = 64 * WAVES;
    static constexpr int BM = 32 * MT * NWR, BN = 32 * NT * NWC;
    static constexpr int SPB = 128 / KS;                 // stages per 128-k block
    static constexpr int ROWB = KS * 2, CPR = KS / 8;    // bytes and 16-byte chunks of a stage row
    static constexpr int ABUF = DA + 1, ASTAGE = BM * ROWB;
    static constexpr int NA = BM * CPR / THREADS;        // A copies per thread and stage
    static_assert(BM * CPR % THREADS == 0, "whole A copies per thread");
};

// f(integral_constant<int, i>) for i = 0 .. NN-1, unrolled at compile time
template <int I, int NN, typename F>
__device__ inline void unroll_impl(F&& f) {
    if constexpr (I < NN) {
        f(std::integral_constant<int, I>{});
        unroll_impl<I + 1, NN>(f);
    }
}
template <int NN, typename F>
__device__ inline void unroll(F&& f) {
    unroll_impl<0, NN>(f);
}

template <int VM>
__device__ inline void wait_vm() {
    static_assert(VM >= 0 && VM < 64, "vmcnt");
    __builtin_amdgcn_s_waitcnt((VM & 15) | ((VM >> 4) << 14) | (7 << 4) | (15 << 8));
}
// LDS by byte address (the kernels have no static LDS: their dynamic LDS starts at 0)
template <class T>
__device__ inline T lds_ld(uint32_t a) {
    return *(const __attribute__((address_space(3))) T*)(size_t)a;
}
// every LDS read of this wave has returned, then the workgroup barrier
__device__ inline void barrier_lds() {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt((63 & 15) | ((63 >> 4) << 14) | (7 << 4) | (0 << 8));
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

// One job.  D: the weight format (Ptq1F16 in gemm_f16.hip, Q8F16 in gemm_q8.hip): its copies, and
// chunk<kk, general>(t), the B operand of 16-k step kk and column tile t, steps in order.  A format
// reads its words from LDS one block ahead (read, unpacked by begin) or two steps ahead (look).
// TWO_FORMS: begin's result selects the general form of the chunks.
template <class C, class D, bool C_F16>
__device__ inline void run(const _Float16* __restrict__ A, int lda, const Mats& P, float* __restrict__ ws, int M,
                           int K, const GemmJobs& J) {
    constexpr int MT = C::MT, NT = C::NT, KS = C::KS, SPB = C::SPB, ROWB = C::ROWB, CPR = C::CPR;
    constexpr int DA = C::DA, DW = C::DW, NA = C::NA, ABUF = C::ABUF;
    constexpr int SPG = D::GROUP * SPB;                       // stages per weight group
    constexpr int NW = D::template copies<C>();               // weight copies per thread and group
    static_assert(DW * SPG >= DA + 1, "a group has landed when its first words are read, in the stage before its own");
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wr = wave / C::NWC, wc = wave % C::NWC;
    const int l32 = lane & 31, lh = lane >> 5;
    const int nbk = K >> 7;
    int job, tile, kb0, nb;
    gemm_job(J, nbk, job, tile, kb0, nb);
    const int m0 = (tile / J.G) * C::BM, mi = mat_of(P, tile % J.G), n0 = (tile % J.G - P.g0[mi]) * C::BN;
    const uint8_t* W = P.W[mi];
    const int N = P.N[mi];
    const int nst = nb * SPB;
    const int ng = (nb + D::GROUP - 1) / D::GROUP;
    constexpr uint32_t Ws = ABUF * C::ASTAGE;                 // LDS: A stages, weight groups

    // ---- A copies: instruction i of this thread copies LDS piece p = THREADS i + tid of the
    // stage: row p / CPR, slot p % CPR, which holds global chunk slot ^ swizzle(row).  The offset
    // is limited to the last chunk of row M - 1: rows past M hold anything in bounds.
    auto swizzle = [](int r) { return KS == 32 ? (r >> 2) & 3 : KS == 64 ? (r >> 1) & 7 : r & 15; };
    constexpr int RPI = C::THREADS / CPR;                     // rows per instruction
    static_assert(RPI % 16 == 0, "the swizzle does not depend on the instruction");
    const uint32_t avo = (uint32_t)(tid / CPR) * (uint32_t)lda * 2u + (uint32_t)(((tid % CPR) ^ swizzle(tid / CPR)) << 4);
    const uint32_t a_lds = 1024u * wave;
    auto issue_a = [&](int st, int buf, int i0, int i1) {     // copies i0 .. i1-1 of stage st
        const _Float16* ko = A + (size_t)kb0 * 128 + (size_t)min(st, nst - 1) * KS;
#pragma unroll
        for (int i = i0; i < i1; i++) {
            const int r0 = min(m0 + i * RPI, M - 1);
            const uint32_t lim = (uint32_t)(M - 1 - r0) < (uint32_t)RPI ? (uint32_t)(M - 1 - r0) * (uint32_t)lda * 2u + (ROWB - 16) : 0xffffffffu;
            dma16(ko + (size_t)r0 * lda, min(avo, lim), a_lds + buf * C::ASTAGE + i * (C::THREADS * 16));
        }
    };
    D dec;
    dec.template init<C>(W, nbk, kb0, nb, n0, N, tid, wave, wc, l32, lh, Ws);
    auto issue_w = [&](int g, int i0, int i1) { dec.template issue<C>(min(g, ng - 1), g % (DW + 1), i0, i1); };
    // A group's weight copies are issued in its DW-th last group's first stage, or, where they
    // still land in time, over all of that group's stages
    constexpr bool SPREAD = (DW - 1) * SPG >= DA;
    auto w0 = [](int sp) constexpr { return SPREAD ? sp * NW / SPG : sp == 0 ? 0 : NW; };

    v16f acc[MT][NT];
#pragma unroll
    for (int i = 0; i < MT; i++)
#pragma unroll
        for (int t = 0; t < NT; t++)
#pragma unroll
            for (int q = 0; q < 16; q++) acc[i][t][q] = 0.0f;

    // prologue: the issues of the virtual stages before 0, in the loop's order
    constexpr int PRE = DA > DW * SPG ? DA : DW * SPG;
    unroll<PRE>([&](auto ic) {
        constexpr int j = decltype(ic)::value - PRE;
        constexpr int sp = ((j % SPG) + SPG) % SPG;
        if constexpr (j >= -DW * SPG) issue_w((j - sp) / SPG + DW, w0(sp), w0(sp + 1));
        if constexpr (j >= -DA) issue_a(j + DA, (j + DA) % ABUF, 0, NA);
    });
    // copies that may still fly when stage sp (of its group) starts: those issued after A(s),
    // which is issued over stage s - DA, after that stage's weight copies
    auto vm_of = [w0](int sp) constexpr {
        int n = (DA - 1) * NA;
        for (int j = sp - DA + 1; j < sp; j++) n += w0((j + SPG) % SPG + 1) - w0((j + SPG) % SPG);
        return n;
    };
    // A fragment addresses: row l32 of each 32-row tile, chunk 2 kk + lh
    const uint32_t a_row = (uint32_t)(wr * 32 * MT + l32) * ROWB + (uint32_t)((lh ^ swizzle(l32)) << 4);
    constexpr int NKK = KS / 16;
    int s = 0, abuf = 0, nbuf = DA % ABUF;                    // stage, its buffer, buffer of stage s + DA
    v8h af[2][MT], bf[2][NT];
    auto frags = [&](auto kc, v8h (&f)[MT]) {
        constexpr int kk = decltype(kc)::value;
        const uint32_t at = abuf * C::ASTAGE + (a_row ^ (uint32_t)(kk << 5));
#pragma unroll
        for (int i = 0; i < MT; i++) f[i] = lds_ld<v8h>(at + i * 32 * ROWB);
    };
    // The stage after stage s starts: its copies have landed and every wave has read the last
    // stage's fragments
    auto next_stage = [&](auto spc) {
        wait_vm<vm_of(decltype(spc)::value)>();
        barrier_lds();
    };
    // first fragments and chunk
    next_stage(std::integral_constant<int, 0>{});
    dec.template read<C, 0>(0, 0, nb);
    dec.template look<C, 6>(-1);
    frags(std::integral_constant<int, 0>{}, af[0]);
    bool big = dec.template begin<C>();
#pragma unroll
    for (int t = 0; t < NT; t++) bf[0][t] = dec.template chunk<0, true>(t);
    dec.template look<C, 7>(-1);
    // Step kk of a block: the fragments and the decode of step kk + 1 run beside the MFMAs of
    // step kk.  A block's chunk 0 is decoded before its scales choose the form of the others.
    auto do_block = [&](auto jc, int g, auto bigc) {
        constexpr int JB = decltype(jc)::value;
        constexpr bool BIG = decltype(bigc)::value;
        unroll<8>([&](auto kc) {
            constexpr int kb = decltype(kc)::value, h = kb / NKK, kk = kb % NKK, sp = JB * SPB + h;
            constexpr int cur = kb & 1, nxt = cur ^ 1;
            if constexpr (kk + 1 == NKK) {
                ++s;
                abuf = abuf + 1 == ABUF ? 0 : abuf + 1;
                nbuf = nbuf + 1 == ABUF ? 0 : nbuf + 1;
                next_stage(std::integral_constant<int, (sp + 1) % SPG>{});
            }
            if constexpr (kb == 7) big = dec.template begin<C>();
            unroll<NT>([&](auto tc) {
                constexpr int t = decltype(tc)::value;
                __builtin_amdgcn_sched_barrier(0);
                if constexpr (t == 0) {
                    frags(std::integral_constant<int, (kk + 1) % NKK>{}, af[nxt]);
                    if constexpr (kk == 0 && h == SPB - 1) {  // the next block's words
                        if constexpr (JB + 1 < D::GROUP)
                            dec.template read<C, JB + 1>(g, g % (DW + 1), nb);
                        else
                            dec.template read<C, 0>(g + 1, (g + 1) % (DW + 1), nb);
                    }
                    dec.template look<C, kb>(g);
                }
                if constexpr (kb < 7) bf[nxt][t] = dec.template chunk<(kb + 1) % 8, BIG>(t);
                else bf[nxt][t] = dec.template chunk<0, true>(t);
#pragma unroll
                for (int i = 0; i < MT; i++)
                    acc[i][t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(af[cur][i], bf[cur][t], acc[i][t], 0, 0, 0);
                if constexpr (t == 0) __builtin_amdgcn_sched_group_barrier(0x100, MT, 0);
#pragma unroll
                for (int i = 0; i < MT; i++) {
                    __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
                    __builtin_amdgcn_sched_group_barrier(0x2, 5, 0);
                }
                __builtin_amdgcn_sched_barrier(0);
                if constexpr (kk == 0 && t == 0) issue_w(g + DW, w0(sp), w0(sp + 1));
                // the copies of stage s + DA, spread over the steps before the stage's last (whose
                // barrier comes first)
                if constexpr (kk + 1 < NKK) {
                    constexpr int slots = (NKK - 1) * NT, i0 = kk * NT + t;
                    issue_a(s + DA, nbuf, i0 * NA / slots, (i0 + 1) * NA / slots);
                }
            });
        });
    };
    // the fast form until a block's scales need the general one, then that to the end
    int b0 = 0;
    auto blocks = [&](auto bigc) {
        for (int g = b0 / D::GROUP; g < ng; g++) {
            bool stop = false;
            unroll<D::GROUP>([&](auto jc) {
                const int b = g * D::GROUP + decltype(jc)::value;
                if (!stop && b >= b0 && b < nb) {
                    stop = !decltype(bigc)::value && big;
                    if (stop) b0 = b;
                    else do_block(jc, g, bigc);
                }
            });
            if (stop) return;
        }
        b0 = nb;
    };
    blocks(std::false_type{});
    if constexpr (D::TWO_FORMS)
        if (__builtin_expect(b0 < nb, 0)) blocks(std::true_type{});
    wait_vm<0>();                                             // the repeated copies, before the LDS is given back

    // store: lane holds D[8(q/4) + 4 lh + q%4][l32] of each 32 x 32 tile
    if (job >= J.n_full) {
        // piece: the fp32 tile, [BM][BN], rows past M left out
        float* T = ws + (size_t)(job - J.n_full) * (C::BM * C::BN);
#pragma unroll
        for (int i = 0; i < MT; i++)
#pragma unroll
            for (int t = 0; t < NT; t++)
#pragma unroll
                for (int q = 0; q < 16; q++) {
                    const int r = (wr * MT + i) * 32 + 8 * (q >> 2) + 4 * lh + (q & 3);
                    if (m0 + r < M) T[r * C::BN + (wc * NT + t) * 32 + l32] = acc[i][t][q];
                }
        return;
    }
    void* Cp = P.C[mi];
    const int ldc = P.ldc[mi];
#pragma unroll
    for (int i = 0; i < MT; i++)
#pragma unroll
        for (int t = 0; t < NT; t++) {
            const int gn = n0 + (wc * NT + t) * 32 + l32;
#pragma unroll
            for (int q = 0; q < 16; q++) {
                const int gm = m0 + (wr * MT + i) * 32 + 8 * (q >> 2) + 4 * lh + (q & 3);
                if (gm < M && gn < N) {
                    if (C_F16) ((_Float16*)Cp)[(size_t)gm * ldc + gn] = (_Float16)acc[i][t][q];
                    else ((float*)Cp)[(size_t)gm * ldc + gn] = acc[i][t][q];
                }
            }
        }
}

// C for the split tiles: the sum of a tile's pieces ([BM][BN] fp32 each, slot order) in piece
// order.  One thread per 4 consecutive columns of a tile row; the pieces' loads are all in
// flight before the sum.  V4: every row of every C starts 16-byte aligned (4 N apart).
template <int BM, int BN, bool C_F16, bool V4>
__global__ __launch_bounds__(256) void k_pieces_sum(const float* __restrict__ ws, Mats P, int M, GemmJobs J) {
    const int t = J.n_full + blockIdx.y;                    // split tile
    const int e = blockIdx.x * 256 + threadIdx.x;           // quad of the tile
    const int r = e / (BN / 4), c4 = (e % (BN / 4)) * 4;
    const int mi = mat_of(P, t % J.G), N = P.N[mi], ldc = P.ldc[mi];
    const int gm = (t / J.G) * BM + r, gn0 = (t % J.G - P.g0[mi]) * BN + c4;
    if (gm >= M || gn0 >= N) return;
    const float* T = ws + (size_t)blockIdx.y * J.S * (BM * BN) + r * BN + c4;
    v4f v[kMaxPieces];
#pragma unroll
    for (int p = 0; p < kMaxPieces; p++)
        if (p < J.S) v[p] = *(const v4f*)(T + (size_t)p * (BM * BN));
    v4f o = v[0];
#pragma unroll
    for (int p = 1; p < kMaxPieces; p++)
        if (p < J.S) o += v[p];
    if (V4) {
        if (C_F16) {
            typedef _Float16 h4 __attribute__((ext_vector_type(4)));
            *(h4*)((_Float16*)P.C[mi] + (size_t)gm * ldc + gn0) = h4{(_Float16)o[0], (_Float16)o[1], (_Float16)o[2], (_Float16)o[3]};
        } else {
            *(v4f*)((float*)P.C[mi] + (size_t)gm * ldc + gn0) = o;
        }
        return;
    }
#pragma unroll
    for (int i = 0; i < 4; i++) {
        if (gn0 + i < N) {
            if (C_F16) ((_Float16*)P.C[mi])[(size_t)gm * ldc + gn0 + i] = (_Float16)o[i];
            else ((float*)P.C[mi])[(size_t)gm * ldc + gn0 + i] = o[i];
        }
    }
}

template <int BM, int BN>
inline hipError_t launch_pieces_sum(const float* ws, const Mats& P, int c_dtype, bool v4, int M, const GemmJobs& J,
                                    hipStream_t s) {
    const int rem = J.n_jobs - J.n_full;
    if (!rem) return hipSuccess;
    const int rows = std::min(BM, (M + 7) & ~7);            // row tiles above the last are whole
    const dim3 grid(rows * BN / 4 / 256, (unsigned)(rem / J.S));
    if (c_dtype == 1) {
        if (v4) hipLaunchKernelGGL((k_pieces_sum<BM, BN, true, true>), grid, dim3(256), 0, s, ws, P, M, J);
        else hipLaunchKernelGGL((k_pieces_sum<BM, BN, true, false>), grid, dim3(256), 0, s, ws, P, M, J);
    } else {
        if (v4) hipLaunchKernelGGL((k_pieces_sum<BM, BN, false, true>), grid, dim3(256), 0, s, ws, P, M, J);
        else hipLaunchKernelGGL((k_pieces_sum<BM, BN, false, false>), grid, dim3(256), 0, s, ws, P, M, J);
    }
    return hipGetLastError();
}

// Schedules.  A configuration runs one workgroup per CU (8 waves, or 4 with the whole register
// file) and is described by the microseconds in which a round of its tiles starts and stores and
// those that a 128-k block of a tile takes on a mostly idle chip (t_alone) and with every CU busy
// (t_full; in between, in proportion to the busy CUs).
struct Shape {
    int bm, bn;
    float start, t_alone, t_full;
    float short_gain;    // all of a table alike, see choose
};
struct Plan {
    GemmJobs J;
    float us;
    int k;               // configuration
};
constexpr int kPieceFloats = 2 * 256 * 128;               // workspace floats per CU
// The cheapest schedule of T = row tiles x column groups tiles on n_cu workgroups: whole tiles
// for the full rounds and the rest split S ways, or every tile split; a split costs the
// pieces' way through memory and back (4 TB/s) and a launch (4 us).
// Where every tile is split, pieces have at least min_blocks blocks.
inline Plan plan(const Shape& c, int M, int G, int nbk, int n_cu, bool pieces, int min_blocks) {
    const long T = (long)((M + c.bm - 1) / c.bm) * G;
    const double rows = (double)M / ((M + c.bm - 1) / c.bm);                // real rows per tile
    auto part = [&](long jobs, int blocks) {                                // a set of equal jobs
        const long rounds = (jobs + n_cu - 1) / n_cu;
        const double busy = (double)jobs / (double)(rounds * n_cu);
        return rounds * (c.start + blocks * std::max((double)c.t_alone, c.t_full * busy));
    };
    Plan best{{G, (int)T, 1, (int)T}, (float)part(T, nbk), 0};
    if (!pieces) return best;
    for (long rem : {T % n_cu, T}) {
        for (int S = 2; rem && S <= kMaxPieces && S * (rem == T ? min_blocks : 1) <= nbk; S++) {
            if ((double)rem * S * c.bm * c.bn > (double)n_cu * kPieceFloats) break;
            const double us = (T > rem ? part(T - rem, nbk) : 0.0) + part(rem * S, (nbk + S - 1) / S) + 4.0 +
                              rem * S * rows * c.bn * 8.0 / 4e6;
            if (us < best.us) best = {{G, (int)(T - rem), S, (int)(T - rem + rem * S)}, (float)us, 0};
        }
    }
    return best;
}

// The cheapest of `shapes`, the first of equal ones.  The model flatters pieces of a few blocks (each
// starts and ends its own way through memory), so a schedule with pieces of 2 to 7 blocks is
// taken only where the model has it below short_gain of the best without.
template <size_t kShapes>
inline Plan choose(const Shape (&shapes)[kShapes], int M, int G, int nbk, int n_cu, bool pieces) {
    auto cheapest = [&](int min_blocks) {
        Plan best{};
        for (int i = 0; i < (int)kShapes; i++) {
            Plan p = plan(shapes[i], M, G, nbk, n_cu, pieces, min_blocks);
            p.k = i;
            if (i == 0 || p.us < best.us) best = p;
        }
        return best;
    };
    const Plan any = cheapest(2), sure = cheapest(8);
    return any.us <= shapes[0].short_gain * sure.us ? any : sure;
}
inline PrefillPlan prefill_plan(const GemmJobs& J, int bm, int bn) {
    return {bm, bn, J.n_full, (J.n_jobs - J.n_full) / J.S, J.S};
}
// launch's plan of matrices N[0 .. count-1]
template <size_t kShapes>
inline PrefillPlan prefill_plan(const Shape (&shapes)[kShapes], int M, int K, int count, const int* N, int n_cu, bool pieces) {
    int G = 0;
    for (int i = 0; i < count; i++) G += (N[i] + shapes[0].bn - 1) / shapes[0].bn;
    const Plan p = choose(shapes, M, G, K / 128, n_cu, pieces);
    return prefill_plan(p.J, shapes[p.k].bm, shapes[p.k].bn);
}

template <class D, class C, bool C_F16>
__global__ __launch_bounds__(C::THREADS, C::WPE) void k_gemm(const _Float16* __restrict__ A, int lda, Mats P,
                                                             float* __restrict__ ws, int M, int K, GemmJobs J) {
    run<C, D, C_F16>(A, lda, P, ws, M, K, J);
}

template <class D, class C>
hipError_t launch_cfg(const _Float16* A, int lda, const Mats& P, float* ws, int c_dtype, bool v4, int M, int K,
                      const GemmJobs& J, hipStream_t s) {
    static constexpr int kLds = C::ABUF * C::ASTAGE + (C::DW + 1) * D::template slot_bytes<C>();
    static_assert(kLds <= 160 * 1024, "LDS");
    // the dynamic-LDS limit of both instantiations, raised once per process (a function-local
    // static: thread-safe initialisation)
    static const hipError_t attr = [] {
        hipError_t e = hipFuncSetAttribute((const void*)k_gemm<D, C, true>, hipFuncAttributeMaxDynamicSharedMemorySize, kLds);
        if (e == hipSuccess)
            e = hipFuncSetAttribute((const void*)k_gemm<D, C, false>, hipFuncAttributeMaxDynamicSharedMemorySize, kLds);
        return e;
    }();
    if (attr != hipSuccess) return attr;
    if (c_dtype == 1)
        hipLaunchKernelGGL((k_gemm<D, C, true>), dim3(J.n_jobs), dim3(C::THREADS), kLds, s, A, lda, P, ws, M, K, J);
    else
        hipLaunchKernelGGL((k_gemm<D, C, false>), dim3(J.n_jobs), dim3(C::THREADS), kLds, s, A, lda, P, ws, M, K, J);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    return launch_pieces_sum<C::BM, C::BN>(ws, P, c_dtype, v4, M, J, s);
}

// C[i] = A W[i]^T for 1..4 matrices of weight format D, on the cheapest of the configurations
// (all with the same column width) that `shapes` describes in the same order.
template <class D, class... Cs>
hipError_t launch(const Shape (&shapes)[sizeof...(Cs)], const _Float16* A, int lda, int count, const uint8_t* const* W, void* const* C,
                  int c_dtype, const int* ldc, int M, int K, const int* N, hipStream_t s) {
    constexpr int kShapes = sizeof...(Cs), BN = std::get<0>(std::array<int, kShapes>{Cs::BN...});
    static_assert(((Cs::BN == BN) && ...), "one column width");
    if (count < 1 || count > kMaxMats) return hipErrorInvalidValue;
    // the copies' row offsets are 32-bit: rows further apart go one by one
    if (lda > (1 << 24) && M > 1) {
        for (int m = 0; m < M; m++) {
            void* Cm[kMaxMats];
            for (int i = 0; i < count; i++) Cm[i] = (uint8_t*)C[i] + (size_t)m * ldc[i] * (c_dtype == 1 ? 2 : 4);
            hipError_t e = launch<D, Cs...>(shapes, A + (size_t)m * lda, K, count, W, Cm, c_dtype, ldc, 1, K, N, s);
            if (e != hipSuccess) return e;
        }
        return hipSuccess;
    }
    // and so are those of the weight rows of a tile: longer rows go a few at a time
    const size_t row_bytes = (size_t)(K / 128) * D::kBlockB;
    if (row_bytes > 0xffffffffu / BN) {
        const int n = (int)std::max<size_t>(1, 0xffffffffu / row_bytes);
        for (int i = 0; i < count; i++)
            for (int n0 = 0; count > 1 || N[i] > n ? n0 < N[i] : false; n0 += n) {
                const uint8_t* Wn = W[i] + (size_t)n0 * row_bytes;
                void* Cn = (uint8_t*)C[i] + (size_t)n0 * (c_dtype == 1 ? 2 : 4);
                const int Nn = std::min(n, N[i] - n0);
                hipError_t e = launch<D, Cs...>(shapes, A, lda, 1, &Wn, &Cn, c_dtype, ldc + i, M, K, &Nn, s);
                if (e != hipSuccess) return e;
            }
        if (count > 1 || N[0] > n) return hipSuccess;
    }
    int n_cu = 0;
    float* ws = nullptr;
    hipError_t e = gemm_device(false, s, &n_cu, &ws);
    if (e != hipSuccess) return e;
    Mats P{};
    bool v4 = true;
    int G = 0;
    for (int i = 0; i < kMaxMats; i++) {
        P.g0[i] = i < count ? G : 0x7fffffff;
        if (i >= count) continue;
        P.W[i] = W[i];
        P.C[i] = C[i];
        P.N[i] = N[i];
        P.ldc[i] = ldc[i];
        G += (N[i] + BN - 1) / BN;
        v4 &= N[i] % 4 == 0 && ldc[i] % 4 == 0 && ((uintptr_t)C[i] & 15) == 0;
    }
    P.g0[kMaxMats] = 0x7fffffff;
    Plan p = choose(shapes, M, G, K / 128, n_cu, true);
    if (p.J.n_jobs > p.J.n_full && gemm_device(true, s, &n_cu, &ws) != hipSuccess) {
        // no workspace (the stream's first call is captured, or memory is short): whole tiles
        (void)hipGetLastError();
        p = choose(shapes, M, G, K / 128, n_cu, false);
    }
    int i = 0;
    ((i++ == p.k ? (void)(e = launch_cfg<D, Cs>(A, lda, P, ws, c_dtype, v4, M, K, p.J, s)) : (void)0), ...);
    return e;
}

}  // namespace rg
}  // namespace kata
