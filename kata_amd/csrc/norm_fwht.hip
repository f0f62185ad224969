// Input transform of every ternary matmul: (residual add +) RMSNorm / SwiGLU / GDN head
// permutation, times the sign vector, then the normalised 1024-point Walsh-Hadamard
// transform of each 1024-block (the model's rotated basis).
//
// Semantics (shaders/common.h:20-42, shaders/ops.metal:30-54,86-106,
// shaders/prefill.metal:59-97,266-285), per token row m and element i < W:
//   mode 0: v = x + y (y optional), xnew = v, inv = 1/sqrt(mean(v^2) + 1e-6),
//           u = v * inv * gs, hout = v * inv * gamma (optional)
//   mode 1: u = silu(src) * src2 * gs          mode 2: u = src[perm(i)] * gs (GDN heads)
//   mode 3: u = src * gs
//   out[block b][j] = (1/32) sum_k (-1)^popcount(j & k) u[1024 b + k]
// fp32 arithmetic; out fp32 or fp16, rows [M][W] or (M = 2) the two tokens interleaved
// per element, [W][2] (the half2 operand of the T = 2 verify GEMV), or (M <= 2 decode, M <= 8
// wide) the GEMV's operand form of the fp32 values (gemv_operand.h), staged per 1024-block in
// LDS and written as whole 16-byte A rows.
//
// Design: a 256-thread workgroup per (1024-block, token) (with the norm each reads the row for its
// sum of squares, L2-resident after the first), or per token row where that is the faster
// (the row read once, held in registers).  Element k = 4 tid + r of a
// block: bits 0-1 are a thread's registers, bits 2-7 its lane (butterflies by cross-lane
// exchange), bits 8-9 its wave (one LDS transpose).  The sum of squares is reduced in a
// fixed order: a butterfly across the wave's lanes, then the 4 waves through LDS.
#include "common.h"
#include "gemv_operand.h"
#include "launch.h"

#include <type_traits>

namespace kata {

namespace {

constexpr float kRmsEps = 1e-6f;   // config/kata_m6.h:21
__constant__ DenseImgOff kOperandOff = make_dense_img_off();

// The value of lane l ^ m for m = 1, 2 (DPP quad permutations), 4 (DPP row shifts: the partner is
// in the lane's row of 16, l + m when bit m is clear, l - m when set; bound_ctrl reads 0 for
// sources outside the row, so the unselected shift is harmless) and 8 (DPP row rotation).  Both
// shifts are computed in every lane before the select: a conditional expression with the DPP
// moves as operands evaluates one per lane, which becomes a branch in which the moves read
// disabled source lanes (zeros).
template <int m>
__device__ inline float partner(float v, int lane) {
    const int iv = __builtin_bit_cast(int, v);
    int pv;
    if constexpr (m == 1) {
        pv = __builtin_amdgcn_mov_dpp(iv, 0xB1, 0xf, 0xf, true);           // quad_perm [1, 0, 3, 2]
    } else if constexpr (m == 2) {
        pv = __builtin_amdgcn_mov_dpp(iv, 0x4E, 0xf, 0xf, true);           // quad_perm [2, 3, 0, 1]
    } else if constexpr (m == 4) {
        const int up = __builtin_amdgcn_mov_dpp(iv, 0x104, 0xf, 0xf, true);   // row_shl:4
        const int dn = __builtin_amdgcn_mov_dpp(iv, 0x114, 0xf, 0xf, true);   // row_shr:4
        pv = lane & 4 ? dn : up;
    } else {
        static_assert(m == 8, "partner in the row");
        pv = __builtin_amdgcn_mov_dpp(iv, 0x128, 0xf, 0xf, true);          // row_ror:8
    }
    return __builtin_bit_cast(float, pv);
}
// For m = 16, 32: lo = the value of the lane with bit m clear, hi = of the one with it set (both
// in both lanes; a vector instruction, where a cross-lane permute goes through LDS)
template <int m>
__device__ inline void halves(float v, float& lo, float& hi) {
    const uint32_t u = __builtin_bit_cast(uint32_t, v);
    if constexpr (m == 16) {
        const auto r = __builtin_amdgcn_permlane16_swap(u, u, false, false);
        lo = __builtin_bit_cast(float, (uint32_t)r[0]);
        hi = __builtin_bit_cast(float, (uint32_t)r[1]);
    } else {
        const auto r = __builtin_amdgcn_permlane32_swap(u, u, false, false);
        lo = __builtin_bit_cast(float, (uint32_t)r[0]);
        hi = __builtin_bit_cast(float, (uint32_t)r[1]);
    }
}

__device__ inline float wave_sum(float a, int lane) {
    // fixed-order butterfly over the 64 lanes
    float lo, hi;
    halves<32>(a, lo, hi);
    a = lo + hi;
    halves<16>(a, lo, hi);
    a = lo + hi;
    a += partner<8>(a, lane);
    a += partner<4>(a, lane);
    a += partner<2>(a, lane);
    a += partner<1>(a, lane);
    return a;
}

// natural-order butterflies over NB blocks of 1024: for bit h the pair (k, k | h) becomes
// (a + b, a - b).  The blocks go through each level together: two barriers for all of them, and
// the cross-lane moves of one block fill the waits of another's.
template <int NB>
__device__ inline void fwht1024(float (&v)[NB][4], int tid, float* xs) {
#pragma clang fp contract(off)                   // the sums of rounded products, in every caller
    const int lane = tid & 63;
#pragma unroll
    for (int n = 0; n < NB; n++) {
        const float a = v[n][0] + v[n][1], b = v[n][0] - v[n][1], c = v[n][2] + v[n][3], d = v[n][2] - v[n][3];
        v[n][0] = a + c;
        v[n][1] = b + d;
        v[n][2] = a - c;
        v[n][3] = b - d;
    }
    // the pair (l, l ^ m): the lane with bit m clear takes the sum, the other the difference
    auto level = [&](auto mc) {
        constexpr int m = decltype(mc)::value;
        const bool hi = lane & m;
#pragma unroll
        for (int n = 0; n < NB; n++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                float& x = v[n][r];
                if constexpr (m <= 8) {
                    const float p = partner<m>(x, lane);
                    x = hi ? p - x : x + p;
                } else {
                    float l, h;
                    halves<m>(x, l, h);
                    x = l + (hi ? -h : h);
                }
            }
    };
    level(std::integral_constant<int, 1>{});
    level(std::integral_constant<int, 2>{});
    level(std::integral_constant<int, 4>{});
    level(std::integral_constant<int, 8>{});
    level(std::integral_constant<int, 16>{});
    level(std::integral_constant<int, 32>{});
    // bits 8-9: element k = 4 tid + r; thread t then owns elements t + 256 j (j = 0..3)
#pragma unroll
    for (int n = 0; n < NB; n++)
#pragma unroll
        for (int r = 0; r < 4; r++) xs[1024 * n + 4 * tid + r] = v[n][r];
    __syncthreads();
#pragma unroll
    for (int n = 0; n < NB; n++) {
        float e[4];
#pragma unroll
        for (int j = 0; j < 4; j++) e[j] = xs[1024 * n + tid + 256 * j];
        const float a2 = e[0] + e[1], b2 = e[0] - e[1], c2 = e[2] + e[3], d2 = e[2] - e[3];
        e[0] = a2 + c2;
        e[1] = b2 + d2;
        e[2] = a2 - c2;
        e[3] = b2 - d2;
#pragma unroll
        for (int j = 0; j < 4; j++) xs[1024 * n + tid + 256 * j] = e[j];
    }
    __syncthreads();
#pragma unroll
    for (int n = 0; n < NB; n++)
#pragma unroll
        for (int r = 0; r < 4; r++) v[n][r] = xs[1024 * n + 4 * tid + r] * 0.03125f;
}

__device__ inline float silu(float x) { return x / (1.0f + expf(-x)); }

// GDN output order: element i of the grouped head layout reads tiled position
// h + 128 (k + 16 rr) for i = 128 t + h, t = 3 k + rr (shaders/ops.metal:47)
__device__ inline int gdn_perm(int i) {
    const int h = i & 127, t = i >> 7, rr = t % 3, k = t / 3;
    return h + 128 * (k + 16 * rr);
}

// This workgroup's 8 blocks of token m (elements 4 tid + r of the 1024-block blk) in the
// decode GEMV's operand form: the 32 lanes of a block reduce its amax, the limbs go to an
// LDS copy of the 8 block images, then 128 threads store the token's 16-byte A rows.
__device__ inline void store_operand(const float (&v)[4], uint2 offw, int tid, int blk, int m, int M, int W,
                                     uint8_t* xs, uint8_t* __restrict__ xq) {
#pragma clang fp contract(off)
    const int BLK = gemv_xq_blk_bytes(M), qbytes = gemv_xq_qbytes(W, M);
    float a = 0.0f;
#pragma unroll
    for (int r = 0; r < 4; r++) a = fmaxf(a, gemv_amax_term(v[r]));
    a = half32_max(a);
    float inv, sc;
    gemv_block_scale(a, inv, sc);
    const int bl = tid >> 5, b = 8 * blk + bl;
    __syncthreads();                              // the transform's last reads of xs
    uint8_t* img = xs + bl * BLK + 32 * m;
#pragma unroll
    for (int r = 0; r < 4; r++) {
        const int off = (int)(((r < 2 ? offw.x : offw.y) >> (16 * (r & 1))) & 0xffffu);
        gemv_limbs(v[r], inv, img[off], img[off + 16]);
    }
    if ((tid & 31) == 0) ((int2*)(xq + 4 * qbytes))[b * M + m] = make_int2(__builtin_bit_cast(int, sc), 0);
    __syncthreads();
    if (tid < 128) {
        // row (mm, g, limb) of block bl: A image bytes mm (8 M 16) + g (2 M 16) + (2 m + limb) 16
        const int pb = tid >> 4, mm = (tid >> 3) & 1, g = (tid >> 1) & 3, limb = tid & 1;
        const int off = mm * (4 * 2 * M * 16) + g * (2 * M * 16) + (2 * m + limb) * 16;
        const int bb = 8 * blk + pb;
        *(uint4*)(xq + (bb & 3) * qbytes + (bb >> 2) * BLK + off) = *(const uint4*)(xs + pb * BLK + off);
    }
}

// The same for M = 3..8 tokens in the wide GEMV's operand form: block b's image at 2048 b,
// A row 2 m + limb of lane group g of MFMA mm at 1024 mm + 256 g + 16 (2 m + limb), the
// scales of token pair p at 2048 nb + 32 b + 8 p.  The workgroups of token 0 also clear
// the rows and scales of tokens M..7 of their blocks.
__device__ inline void store_operand_wide(const float (&v)[4], uint2 offw, int tid, int blk, int m, int M, int W,
                                          uint8_t* xs, uint8_t* __restrict__ xq) {
#pragma clang fp contract(off)
    constexpr int BLK = kWideImgBlk;
    const int nb = W >> 7;
    float a = 0.0f;
#pragma unroll
    for (int r = 0; r < 4; r++) a = fmaxf(a, gemv_amax_term(v[r]));
    a = half32_max(a);
    float inv, sc;
    gemv_block_scale(a, inv, sc);
    const int bl = tid >> 5, b = 8 * blk + bl;
    __syncthreads();                              // the transform's last reads of xs
    // staging: per block the token's 16 A rows [mm 2][g 4][limb 2][16 B] (256 B)
    uint8_t* img = xs + bl * 256;
#pragma unroll
    for (int r = 0; r < 4; r++) {
        const int o = (int)(((r < 2 ? offw.x : offw.y) >> (16 * (r & 1))) & 0xffffu);   // [mm][g][row 16][16 B]
        const int so = (o >> 10) * 128 + ((o >> 8) & 3) * 32 + (o & 15);
        gemv_limbs(v[r], inv, img[so], img[so + 16]);
    }
    float* scl = (float*)(xq + (size_t)nb * BLK);
    if ((tid & 31) == 0) scl[b * 8 + m] = sc;
    __syncthreads();
    if (tid < 128) {
        const int pb = tid >> 4, mm = (tid >> 3) & 1, g = (tid >> 1) & 3, limb = tid & 1;
        const int bb = 8 * blk + pb;
        *(uint4*)(xq + (size_t)bb * BLK + mm * 1024 + g * 256 + (2 * m + limb) * 16) =
            *(const uint4*)(xs + pb * 256 + mm * 128 + g * 32 + limb * 16);
    }
    if (m == 0) {
        // rows 2 M .. 15 of the 8 blocks' 8 (mm, g) groups, and the scales of tokens M..7
        const int nr = 16 - 2 * M;
        for (int i = tid; i < 8 * 8 * nr; i += 256) {
            const int pb = i / (8 * nr), rem = i % (8 * nr), grp = rem / nr, row = 2 * M + rem % nr;
            *(uint4*)(xq + (size_t)(8 * blk + pb) * BLK + grp * 256 + row * 16) = make_uint4(0, 0, 0, 0);
        }
        if (tid < 8 * (8 - M)) scl[(8 * blk + tid / (8 - M)) * 8 + M + tid % (8 - M)] = 0.0f;
    }
}

// flags: 2 = write xnew, 4 = write hout, 8 = hout fp16.  NORM: mode 0, ADD: of x + y.
// ROW: grid M, a workgroup holds a row (NB = W/1024), read once.  Otherwise a workgroup holds one
// block (NB = 1) and, with NORM, reads the rest of its row for the sum of squares.  Workgroups go
// round robin to 8 XCDs; from 8 rows on, grid (8 W/1024, M/8) puts the blocks of row 8 y + i on XCD i
// one after the other: the row comes once from HBM and then from that XCD's L2.  x + y, norm to fp16, us with
// the rows or the blocks of one row consecutive / so: 333 rows of 6144 18 / 19 / 8.9, 7300 rows
// 468 / 362 / 188, 7300 rows of 17408 3555 / 1254 / 880; SwiGLU, 7300 rows of 17408, 250 / 224 / 220.
// NR: 1024-blocks of the row whose loads are in flight together (for a shorter row its first block
// again: free at widths 3072 and 4096, at 2048 four of six: 512 rows of x + y 5.2 us, 4.4 with NR 2,
// 4.7 with the loads one by one).
template <int NB, bool NORM, bool ROW, bool ADD, int NR = 1>
__global__ __launch_bounds__(256) void k_norm_fwht(const float* __restrict__ src, const float* __restrict__ src2,
                                                   const float* __restrict__ gs, void* __restrict__ out, int out_dtype,
                                                   int out_layout, float* __restrict__ xnew,
                                                   const float* __restrict__ gamma, void* __restrict__ hout,
                                                   int flags, int W, int M, int mode) {
    __shared__ float xs[NB * 1024];
    __shared__ float part[4];
    const int tid = threadIdx.x;
    const int m = ROW ? blockIdx.x : M < 8 ? blockIdx.y : 8 * blockIdx.y + (blockIdx.x & 7);
    const int blk0 = ROW ? 0 : M < 8 ? blockIdx.x : blockIdx.x >> 3;
    if (!ROW && m >= M) return;
    const size_t ro = (size_t)m * W;
    // the operand form's image offsets of this thread's 4 elements, loaded first (their
    // latency then overlaps the row loads)
    [[maybe_unused]] uint2 offw = make_uint2(0, 0);
    if constexpr (NB == 1) {
        if (out_dtype == 2) offw = *(const uint2*)&kOperandOff.v[M <= 2 ? M - 1 : 2][(4 * tid) & 127];
    }
    // Few rows are bound by latency: every load of the blocks and of the row's sum of squares is
    // issued before the first is used, from addresses that are always valid instead of under
    // branches, whose joins wait.  x + y, norm and operand at W = 5120 in a graph: 4.14 -> 3.40 us
    // at 1 row, 4.39 -> 3.68 at 6 (2.1 us of it are the launch).
    float4 g[NB], gm[NORM ? NB : 1];
#pragma unroll
    for (int b = 0; b < NB; b++) {
        const int base = (blk0 + b) * 1024 + 4 * tid;
        g[b] = *(const float4*)(gs + base);
        if constexpr (NORM) gm[b] = *(const float4*)((flags & 4 ? gamma : gs) + base);
    }
    // v = x (+ y) of this thread's elements 1024 (blk0 + b) + 4 tid + r, b < NB
    [[maybe_unused]] float s[NORM ? NB : 1][4];
    float inv = 1.0f;
    if constexpr (NORM) {
        const float* const yrow = ADD ? src2 + ro : nullptr;
        const float4 zero = make_float4(0.f, 0.f, 0.f, 0.f);
        float4 ra[ROW ? 1 : NR], rc[ROW ? 1 : NR];
        if constexpr (!ROW) {
#pragma unroll
            for (int j = 0; j < NR; j++) {
                const int i = 4 * tid + (1024 * j < W ? 1024 * j : 0);
                ra[j] = *(const float4*)(src + ro + i);
                rc[j] = ADD ? *(const float4*)(yrow + i) : zero;
            }
        }
#pragma unroll
        for (int b = 0; b < NB; b++) {
            const int base = (blk0 + b) * 1024 + 4 * tid;
            const float4 a = *(const float4*)(src + ro + base);
            const float4 c = ADD ? *(const float4*)(yrow + base) : zero;
            s[b][0] = a.x + c.x;
            s[b][1] = a.y + c.y;
            s[b][2] = a.z + c.z;
            s[b][3] = a.w + c.w;
        }
        float ss = 0.0f;
        auto add = [&](const float4& a, const float4& c) {
            const float v0 = a.x + c.x, v1 = a.y + c.y, v2 = a.z + c.z, v3 = a.w + c.w;
            ss += (v0 * v0 + v1 * v1) + (v2 * v2 + v3 * v3);
        };
        if constexpr (!ROW) {
#pragma unroll
            for (int j = 0; j < NR; j++)
                if (1024 * j < W) add(ra[j], rc[j]);
            for (int i = 4 * tid + 1024 * NR; i < W; i += 1024) {
                add(*(const float4*)(src + ro + i), ADD ? *(const float4*)(yrow + i) : zero);
            }
        } else {
#pragma unroll
            for (int b = 0; b < NB; b++) ss += (s[b][0] * s[b][0] + s[b][1] * s[b][1]) + (s[b][2] * s[b][2] + s[b][3] * s[b][3]);
        }
        ss = wave_sum(ss, tid & 63);
        if ((tid & 63) == 0) part[tid >> 6] = ss;
        __syncthreads();
        inv = 1.0f / sqrtf((part[0] + part[1] + part[2] + part[3]) / (float)W + kRmsEps);
    }
    float v[NB][4];
#pragma unroll
    for (int b = 0; b < NB; b++) {
        const int base = (blk0 + b) * 1024 + 4 * tid;
        const float gv[4] = {g[b].x, g[b].y, g[b].z, g[b].w};
        if constexpr (NORM) {
            if (flags & 2) *(float4*)(xnew + ro + base) = make_float4(s[b][0], s[b][1], s[b][2], s[b][3]);
            if (flags & 4) {
                const float h[4] = {s[b][0] * inv * gm[b].x, s[b][1] * inv * gm[b].y, s[b][2] * inv * gm[b].z, s[b][3] * inv * gm[b].w};
                if (flags & 8) {
                    typedef _Float16 h4 __attribute__((ext_vector_type(4)));
                    *(h4*)((_Float16*)hout + ro + base) = h4{(_Float16)h[0], (_Float16)h[1], (_Float16)h[2], (_Float16)h[3]};
                } else {
                    *(float4*)((float*)hout + ro + base) = make_float4(h[0], h[1], h[2], h[3]);
                }
            }
#pragma unroll
            for (int r = 0; r < 4; r++) v[b][r] = s[b][r] * inv * gv[r];
        } else if (mode == 1) {
            const float4 a = *(const float4*)(src + ro + base);
            const float4 c = *(const float4*)(src2 + ro + base);
            const float av[4] = {a.x, a.y, a.z, a.w}, cv[4] = {c.x, c.y, c.z, c.w};
#pragma unroll
            for (int r = 0; r < 4; r++) v[b][r] = silu(av[r]) * cv[r] * gv[r];
        } else if (mode == 2) {
            const float4 a = *(const float4*)(src + ro + gdn_perm(base));    // base..base + 3 in one head
            const float av[4] = {a.x, a.y, a.z, a.w};
#pragma unroll
            for (int r = 0; r < 4; r++) v[b][r] = av[r] * gv[r];
        } else {
            const float4 a = *(const float4*)(src + ro + base);
            const float av[4] = {a.x, a.y, a.z, a.w};
#pragma unroll
            for (int r = 0; r < 4; r++) v[b][r] = av[r] * gv[r];
        }
    }
    fwht1024(v, tid, xs);
#pragma unroll
    for (int b = 0; b < NB; b++) {
        const int base = (blk0 + b) * 1024 + 4 * tid;
        if constexpr (NB == 1) {                 // staged in xs: one block per workgroup
            if (out_dtype == 2) {
                if (M <= 2)
                    store_operand(v[b], offw, tid, blk0, m, M, W, (uint8_t*)xs, (uint8_t*)out);
                else
                    store_operand_wide(v[b], offw, tid, blk0, m, M, W, (uint8_t*)xs, (uint8_t*)out);
                return;
            }
        }
        if (out_dtype == 0) {
            *(float4*)((float*)out + ro + base) = make_float4(v[b][0], v[b][1], v[b][2], v[b][3]);
        } else if (out_layout == 0) {
            typedef _Float16 h4 __attribute__((ext_vector_type(4)));
            *(h4*)((_Float16*)out + ro + base) = h4{(_Float16)v[b][0], (_Float16)v[b][1], (_Float16)v[b][2], (_Float16)v[b][3]};
        } else {
            _Float16* o = (_Float16*)out;        // [W][2]: token m at 2 i + m
#pragma unroll
            for (int r = 0; r < 4; r++) o[2 * (base + r) + m] = (_Float16)v[b][r];
        }
    }
}

}  // namespace

hipError_t launch_norm_fwht(const float* src, const float* src2, const float* gs, void* out, int out_dtype,
                            int out_layout, float* xnew, const float* gamma, void* hout, int flags, int W, int M,
                            int mode, hipStream_t s) {
    auto go = [&](auto kern, dim3 grid) {
        hipLaunchKernelGGL(kern, grid, dim3(256), 0, s, src, src2, gs, out, out_dtype, out_layout, xnew, gamma, hout,
                           flags, W, M, mode);
        return hipGetLastError();
    };
    const dim3 blocks = M < 8 ? dim3(W / 1024, M) : dim3(8 * (W / 1024), (M + 7) / 8);
    // Without the norm nothing is shared by a row's blocks: blocks at every size (width 5120 to fp16, us
    // by rows / by blocks: 64 rows of SwiGLU 6.9 / 3.1, 7300 75.5 / 67.4; plain 5.8 / 2.8, 39.9 / 36.6).
    if (mode != 0) return go(k_norm_fwht<1, false, false, false>, blocks);
    // With it, whole rows per workgroup read a row once, blocks per workgroup W/1024 times but with
    // as many times the waves.  Width 5120, x + y to fp16, us by blocks / by rows: 64 rows 4.2 / 5.0,
    // 129 4.9 / 5.5, 200 5.7 / 5.8, 256 6.5 / 6.1, 512 10.2 / 8.6, 7300 161 / 94.  At width 1024 the
    // block is the row.
    auto norm = [&](auto add) {
        constexpr bool ADD = decltype(add)::value;
        if (W == 1024) return go(k_norm_fwht<1, true, true, ADD>, dim3(M));
        if (W == 5120 && M > 200) return go(k_norm_fwht<5, true, true, ADD>, dim3(M));
        if (W == 2048) return go(k_norm_fwht<1, true, false, ADD, 2>, blocks);
        return go(k_norm_fwht<1, true, false, ADD, 6>, blocks);
    };
    return flags & 1 ? norm(std::true_type{}) : norm(std::false_type{});
}

}  // namespace kata
