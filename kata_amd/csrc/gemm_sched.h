// Tile schedule of the prefill GEMMs: the piece bookkeeping (gemm_job, the workspace) of all of
// them, and the plan of the tall int8 kernel (gemm_i8.hip; the others plan in gemm_reg.h).
//
// C is cut into tiles, tile t = (row tile t / G, column group t % G).  Tiles 0 .. n_full - 1 are
// taken whole by one workgroup each; the others are split along K into S pieces, one workgroup
// each, so that few tiles, or the last round of many, fill the chip too.  A piece writes its fp32
// partial tile to the stream's workspace and rg::k_pieces_sum adds the pieces of each split
// tile in piece order (deterministic).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>

namespace kata {

constexpr int kMaxPieces = 16;   // K pieces of one split tile

struct GemmJobs {
    int G;        // column groups
    int n_full;   // whole tiles (jobs 0 .. n_full-1)
    int S;        // pieces per split tile
    int n_jobs;   // workgroups: piece slot j = job - n_full is piece j % S of tile n_full + j / S
};

// The plan of the tall int8 kernel: with `slots` workgroups resident at once, whole rounds of `slots`
// tiles, and the r tiles left over in S = min(slots / r, kMaxPieces, K blocks) pieces.
inline GemmJobs plan_gemm_jobs(int M, int N, int K, int TBM, int TBN, int slots) {
    GemmJobs J;
    J.G = (N + TBN - 1) / TBN;
    const long T = (long)((M + TBM - 1) / TBM) * J.G;
    const int nbk = K / 128;
    long rem = T % slots;
    int S = rem ? std::min(std::min(slots / (int)rem, kMaxPieces), nbk) : 1;
    if (S < 2) {
        S = 1;
        rem = 0;
    }
    J.n_full = (int)(T - rem);
    J.S = S;
    J.n_jobs = (int)(J.n_full + rem * S);
    return J;
}

// The job of this workgroup: tile, first K block and K blocks.  Workgroups are dispatched
// round robin over 8 XCDs: within the whole tiles and within the pieces, consecutive jobs
// (tiles sharing A rows) are placed on one XCD, whose L2 then serves them.
__device__ inline void gemm_job(const GemmJobs& J, int nbk, int& job, int& tile, int& kb0, int& nb) {
    job = blockIdx.x;
    const int lo = job < J.n_full ? 0 : J.n_full;
    const int n = job < J.n_full ? J.n_full : J.n_jobs - J.n_full;
    const int i = job - lo;
    // (a bijection for any n: XCD x takes n / 8 jobs, one more for x < n % 8)
    job = lo + (i % 8) * (n / 8) + min(i % 8, n % 8) + i / 8;
    if (job < J.n_full) {
        tile = job;
        kb0 = 0;
        nb = nbk;
    } else {
        const int j = job - J.n_full, piece = j % J.S;
        tile = J.n_full + j / J.S;
        kb0 = (int)(((long)piece * nbk) / J.S);
        nb = (int)(((long)(piece + 1) * nbk) / J.S) - kb0;
    }
}

// The calling thread's device: its CU count and (need_ws) the K-piece workspace of stream s
// (room for two 256 x 128 fp32 tiles per CU: 64 MB on MI355X), allocated on the first call on
// that (device, stream) that asks for it and kept; calls on other streams use their own.
hipError_t gemm_device(bool need_ws, hipStream_t s, int* n_cu, float** ws);

}  // namespace kata
