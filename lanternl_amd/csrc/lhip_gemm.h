// lhip_gemm.h -- what the GEMM translation units share: the kernel arguments,
// the tile raster and the launchers that cross them.
#ifndef LHIP_GEMM_H
#define LHIP_GEMM_H

#include "lhip_internal.h"

namespace lhip {

// Map the linear workgroup id to a (tile_m, tile_n) pair: XCD-contiguous
// chunks, then GROUP_M-row-band grouped raster inside the chunk order.
__device__ __forceinline__ void tile_coords(int pid, int nwg, int tiles_m, int tiles_n, int& tm, int& tn)
{
    constexpr int kXcds = 8;
    constexpr int kGroupM = 8;
    if ((nwg % kXcds) == 0) pid = (pid % kXcds) * (nwg / kXcds) + pid / kXcds;
    const int per_group = kGroupM * tiles_n;
    const int group = pid / per_group;
    const int first_m = group * kGroupM;
    const int gsz = min(tiles_m - first_m, kGroupM);
    const int in_group = pid - group * per_group;
    tm = first_m + in_group % gsz;
    tn = in_group / gsz;
}

// Kernel arguments (one struct: the launch passes it by value).
struct GemmArgs {
    int M, N, K;
    float alpha, beta;
    const float* A; int lda; long long sA, sA2;
    const float* B; int ldb; long long sB, sB2;
    float* C; int ldc; long long sC, sC2;
    const float* R; int ldr;          // the beta term reads R (R == C unless a residual is given)
    int tiles_m, tiles_n, vecA, vecB, inner;
    int splits, kchunk;               // split-K: blockIdx.z = slice, K range [z*kchunk, (z+1)*kchunk)
    float* ws;                        // split-K partials [split][batch][M][N]
    int Kb;                           // batch-reduce: K = kblocks * Kb, block j reads A + j*sAk, B + j*sBk
    long long sAk, sBk;
    int tail;                         // x3: only the last `tail` tiles are split (partials in ws as [slice][tile][tile elements])
    int skip_reduce;                  // split-K slices stay in ws for the caller to sum
    size_t ws_floats_avail;           // floats available at ws (skinny path's split plan)
};

// The three-term bf16 GEMM (lhip_gemm_x3.hip): its tile and split-K plan for a
// product, and the launch.
constexpr int kX3K = 16;   // k per stage; batch-reduce blocks must be whole stages
constexpr size_t kX3WsFloats = static_cast<size_t>(1) << 24;   // most split-K partials a plan may use
struct X3Plan {
    int tile;             // index into the kernel's tile table
    int splits, kchunk;   // split-K slices and their length
    int tail;             // > 0: only the last `tail` tiles are split (the rest run whole)
    size_t ws_floats;     // the slices' partials
};
// kb: the block length of a batch-reduce (0: one block, which may be split);
// tail_ok: the last tiles alone may be split (the launch then reduces them itself).
// False when no tile takes the operands (leading dimensions past 32-bit
// offsets, partial stages in a batch-reduce).
bool x3_plan(int ta, int tb, int m, int n, int k, int kb, int lda, int ldb, int ldc, int batch, size_t ws_floats,
             bool tail_ok, X3Plan* out);
// Grouped A^T.B products on it (offsets within the limits of x3_plan's operands).
int launch_x3_grouped_tn(const GroupedTN* g, int ngroups, int K, hipStream_t stream);
int launch_x3(int tile, bool br, int ta, int tb, const GemmArgs& g, int batch, hipStream_t stream);

// K slices of the skinny path (lhip_gemm.hip).
int skinny_plan(int m, int n, int k, size_t ws_floats, int* kchunk_out);
// The split-K slices and partials (floats) of the documented limits (lhip_gemm_limits.hip).
int splitk_plan(int m, int n, int k, int batch, size_t ws_floats, int* kchunk);
size_t documented_partials(int transa, int transb, int m, int n, int k, int batch);

// The ordered sum of split-K slices into C (lhip_gemm.hip).
int launch_reduce(const GemmArgs& g, int batch, hipStream_t stream);

}  // namespace lhip

#endif  // LHIP_GEMM_H
