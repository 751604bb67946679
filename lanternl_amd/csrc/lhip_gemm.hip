// lhip_gemm.hip -- fp32 GEMM family on CDNA4 matrix cores (v_mfma_f32_32x32x2f32).
//
// C = alpha * op(A) * op(B) + beta * C, row-major, op = identity or transpose.
// Serves the three products of the reference's strided luaTL_gemm_ex
// (cuda/luaTL_train.cu:1075-1094 -> luaTL_gemm_ex_launch 391-476): A.B for the
// forward, A.B^T (matmul_dx) and A^T.B (matmul_dw) for the backward
// (ai/gpu/luaTL_train.lua:154-182), and the host-table products of
// ai/core/matrix.lua (multiply :541, matmul_nt :597, matmul_tn :627).
//
// This file holds the dispatch (sgemm_run), the fp32-core kernels of the small
// and skinny products, the grouped weight gradients and the ordered split-K
// reduce; everything larger runs on the three-term bf16 kernel of
// lhip_gemm_x3.hip.  By rule (each with its measurements at the rule):
//   * up to 16 rows of C (32 on a large aligned B), B stored K x N: one
//     streaming pass over B (skinny_best);
//   * fewer 32x32 tiles than CUs: 16x16 tiles, K split over the waves of a
//     workgroup (tiny_best);
//   * at most one 64x64 tile per CU over a short aligned K: 64x64 tiles on two
//     wave sets (ks_best);
//   * otherwise lhip_gemm_x3.hip's tile and split (x3_plan).
// The workgroup ids of a product are remapped so that consecutive tiles of a row
// band land on the same XCD (blocks are dispatched round-robin over the 8 XCDs,
// each with its own L2), then grouped kGroupM bands at a time for L2 reuse.
#include <algorithm>
#include <type_traits>

#include "lhip_gemm.h"
#include "lhip_reduce.h"

namespace lhip {
namespace {

typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef float floatx4 __attribute__((ext_vector_type(4)));

constexpr int kThreads = 256;  // 4 wave64s
constexpr int kSmallU = 8;     // K steps whose loads the small kernel issues together

// Loads a ROWS x COLS tile of a row-major matrix into registers, float4 per
// thread per pass, consecutive threads walking the contiguous dimension.
template <int ROWS, int COLS>
struct TileRegs {
    static constexpr int CQ = COLS / 4;            // float4s per tile row
    static constexpr int RPP = kThreads / CQ;      // tile rows per pass
    static constexpr int PASSES = ROWS / RPP;
    static_assert(COLS % 4 == 0 && kThreads % CQ == 0 && ROWS % RPP == 0, "tile/thread mismatch");
    float4 v[PASSES];

    // Every element in bounds and the stored rows 16-byte aligned: one
    // unconditional float4 load per pass (no branch for a wait to be
    // conservative about).
    // Rows past rmax and columns past cmax (cmax % 4 == 0) are clamped into
    // the operand: they only reach outputs that are not stored.
    __device__ __forceinline__ void load_full(const float* __restrict__ g, int ld, int r0, int c0, int rmax, int cmax,
                                              int tid)
    {
        const int cq = tid % CQ;
        const int rr = tid / CQ;
        const int c = min(c0 + 4 * cq, cmax - 4);
#pragma unroll
        for (int p = 0; p < PASSES; ++p) {
            const int r = min(r0 + rr + p * RPP, rmax - 1);
            const float4 t = *reinterpret_cast<const float4*>(g + static_cast<long long>(r) * ld + c);
            v[p].x = t.x; v[p].y = t.y; v[p].z = t.z; v[p].w = t.w;   // per component: stays in VGPRs
        }
    }

    // Store as lds[row][col] (tile orientation kept; LD % 4 == 0).
    template <int LD>
    __device__ __forceinline__ void store_direct(float* lds, int tid) const
    {
        const int cq = tid % CQ;
        const int rr = tid / CQ;
#pragma unroll
        for (int p = 0; p < PASSES; ++p)
            *reinterpret_cast<float4*>(lds + (rr + p * RPP) * LD + 4 * cq) = v[p];
    }

    // Store transposed as lds[col][row].
    template <int LD>
    __device__ __forceinline__ void store_transposed(float* lds, int tid) const
    {
        const int cq = tid % CQ;
        const int rr = tid / CQ;
#pragma unroll
        for (int p = 0; p < PASSES; ++p) {
            const int r = rr + p * RPP;
            lds[(4 * cq + 0) * LD + r] = v[p].x;
            lds[(4 * cq + 1) * LD + r] = v[p].y;
            lds[(4 * cq + 2) * LD + r] = v[p].z;
            lds[(4 * cq + 3) * LD + r] = v[p].w;
        }
    }
};

// C = alpha * sum_s ws[s] + beta * R, the slices summed in order (deterministic).
__global__ void __launch_bounds__(256)
splitk_reduce(const GemmArgs g, int batch)
{
    const long long mn = static_cast<long long>(g.M) * g.N;
    const long long total = mn * batch;
    const long long pstride = mn * batch;
    const long long stride = static_cast<long long>(gridDim.x) * blockDim.x;
    for (long long idx = blockIdx.x * static_cast<long long>(blockDim.x) + threadIdx.x; idx < total; idx += stride) {
        const long long z = idx / mn, rc = idx - z * mn;
        const int row = static_cast<int>(rc / g.N), col = static_cast<int>(rc - static_cast<long long>(row) * g.N);
        float sum = 0.f;
        const float* src = g.ws + idx;
        for (int p = 0; p < g.splits; ++p) sum += src[p * pstride];
        const long long coff = (z / g.inner) * g.sC2 + (z % g.inner) * g.sC;
        float* dst = g.C + coff + static_cast<long long>(row) * g.ldc + col;
        const float v = g.alpha * sum;
        if (g.beta != 0.f) {
            const float* r = g.R ? g.R + coff + static_cast<long long>(row) * g.ldr + col : dst;
            *dst = v + g.beta * (*r);
        } else {
            *dst = v;
        }
    }
}

// Float4 form of splitk_reduce for batch 1 (N % 4 == 0, ldc % 4 == 0 and
// 16-byte aligned C, R): four columns per thread, the slices' loads issued
// eight at a time, summed in slice order.
__global__ void __launch_bounds__(256)
splitk_reduce4(const GemmArgs g)
{
    const long long mn4 = static_cast<long long>(g.M) * g.N / 4;
    const long long stride = static_cast<long long>(gridDim.x) * blockDim.x;
    const int n4 = g.N / 4;
    for (long long idx = blockIdx.x * static_cast<long long>(blockDim.x) + threadIdx.x; idx < mn4; idx += stride) {
        const int row = static_cast<int>(idx / n4), col = 4 * static_cast<int>(idx - static_cast<long long>(row) * n4);
        const float4* src = reinterpret_cast<const float4*>(g.ws) + idx;
        float4 sum = make_float4(0.f, 0.f, 0.f, 0.f);
        int p = 0;
        for (; p + 8 <= g.splits; p += 8) {
            float4 t[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) t[u] = src[(p + u) * mn4];
#pragma unroll
            for (int u = 0; u < 8; ++u) { sum.x += t[u].x; sum.y += t[u].y; sum.z += t[u].z; sum.w += t[u].w; }
        }
        for (; p < g.splits; ++p) {
            const float4 t = src[p * mn4];
            sum.x += t.x; sum.y += t.y; sum.z += t.z; sum.w += t.w;
        }
        float4* dst = reinterpret_cast<float4*>(g.C + static_cast<long long>(row) * g.ldc + col);
        float4 v = make_float4(g.alpha * sum.x, g.alpha * sum.y, g.alpha * sum.z, g.alpha * sum.w);
        if (g.beta != 0.f) {
            const float4 r = g.R ? *reinterpret_cast<const float4*>(g.R + static_cast<long long>(row) * g.ldr + col) : *dst;
            v.x += g.beta * r.x; v.y += g.beta * r.y; v.z += g.beta * r.z; v.w += g.beta * r.w;
        }
        *dst = v;
    }
}

// 64x64 tiles on two wave sets per workgroup (512 threads): set s takes the
// 32-deep K chunks s, s + 2, ... with its own double-buffered LDS, so each SIMD
// holds two waves and each set's chain of dependent chunk loads is half as
// long; the sets' partial tiles meet in LDS (fixed order).  Two register sets
// per wave set: chunk kt + 4 is in flight while chunk kt runs and chunk kt + 2
// goes to LDS.  Every load is unconditional (past its last chunk a set reloads
// that chunk and never stores it), so the wait before an LDS store counts only
// the loads of the chunk being stored.
constexpr int kKsTile = 64, kKsK = 32;

template <bool TA, bool TB>
__global__ void __launch_bounds__(2 * kThreads)
sgemm_mfma_ks_kernel(const GemmArgs g)
{
    constexpr int BM = kKsTile, BN = kKsTile, BK = kKsK, KS = 2;
    constexpr int WM = BM / 2, WN = BN / 2;
    constexpr int LDA = TA ? BM + 4 : BM + 1;
    constexpr int LDB = TB ? BN + 1 : BN + 4;
    __shared__ float As[KS][2][BK * LDA];
    __shared__ float Bs[KS][2][BK * LDB];
    const int M = g.M, N = g.N;
    const int tid = threadIdx.x;
    const int grp = __builtin_amdgcn_readfirstlane(tid >> 8), gt = tid & 255;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane((tid >> 6) & 3);
    const int lr = lane & 31, lk = lane >> 5;
    int tm, tn;
    tile_coords(blockIdx.x, gridDim.x, g.tiles_m, g.tiles_n, tm, tn);
    const int m0 = tm * BM, n0 = tn * BN;
    const long long zo = blockIdx.y / g.inner, zi = blockIdx.y % g.inner;
    const float* __restrict__ A = g.A + zo * g.sA2 + zi * g.sA;
    const float* __restrict__ B = g.B + zo * g.sB2 + zi * g.sB;
    const long long coff = zo * g.sC2 + zi * g.sC;
    const int wm = (wave >> 1) * WM, wn = (wave & 1) * WN;
    TileRegs<TA ? BK : BM, TA ? BM : BK> ra, ra2;
    TileRegs<TB ? BN : BK, TB ? BK : BN> rb, rb2;
    auto gload_to = [&](auto& xa, auto& xb, int k0) {
        // K is whole chunks; M and N are clamped (M % 4 == 0 when A is stored
        // K-major, N % 4 == 0 when B is)
        if (TA) xa.load_full(A, g.lda, k0, m0, g.K, M, gt);
        else    xa.load_full(A, g.lda, m0, k0, M, g.K, gt);
        if (TB) xb.load_full(B, g.ldb, n0, k0, N, g.K, gt);
        else    xb.load_full(B, g.ldb, k0, n0, g.K, N, gt);
    };
    auto lstore_from = [&](const auto& xa, const auto& xb, int buf) {
        if (TA) xa.template store_direct<LDA>(As[grp][buf], gt);
        else    xa.template store_transposed<LDA>(As[grp][buf], gt);
        if (TB) xb.template store_transposed<LDB>(Bs[grp][buf], gt);
        else    xb.template store_direct<LDB>(Bs[grp][buf], gt);
    };
    floatx16 acc;
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[r] = 0.f;
    const int nk = g.K / BK;
    const int iters = (nk + KS - 1) / KS;
    auto mma = [&](int cur) {
        const float* as = As[grp][cur];
        const float* bs = Bs[grp][cur];
#pragma unroll
        for (int kk = 0; kk < BK; kk += 2) {
            const float a = as[(kk + lk) * LDA + wm + lr], b = bs[(kk + lk) * LDB + wn + lr];
            acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, acc, 0, 0, 0);
        }
    };
    gload_to(ra, rb, min(grp, nk - 1) * BK);
    gload_to(ra2, rb2, min(grp + KS, nk - 1) * BK);
    lstore_from(ra, rb, 0);
    __syncthreads();
    // the register sets are picked at compile time (a run-time choice between
    // them would put both in scratch memory)
    auto body = [&](int it, auto setc) {
        constexpr int L = decltype(setc)::value;   // the set loaded; the other is stored
        auto& la = L == 0 ? ra : ra2;
        auto& lb = L == 0 ? rb : rb2;
        const auto& sa = L == 0 ? ra2 : ra;
        const auto& sb = L == 0 ? rb2 : rb;
        const int cur = it & 1;
        const int kt = it * KS + grp;
        gload_to(la, lb, min(kt + 2 * KS, nk - 1) * BK);
        if (kt < nk) mma(cur);
        if (kt + KS < nk) lstore_from(sa, sb, cur ^ 1);
        __syncthreads();
    };
    // No branch around the second body (past the last iteration it only
    // reloads the last chunk; its MFMAs and LDS store are skipped), so every
    // path through the loop has the same loads in flight and each LDS store
    // waits for its own chunk alone (tied head 7.04 -> 6.88 us).
    for (int it = 0; it < iters; it += 2) {
        body(it, std::integral_constant<int, 0>{});
        body(it + 1, std::integral_constant<int, 1>{});
    }
    float* red = &As[0][0][0];   // set 1 leaves its partial tile here
    static_assert(4096 <= KS * 2 * BK * LDA, "reduction area");
    if (grp > 0) {
#pragma unroll
        for (int r = 0; r < 16; ++r) red[wave * 1024 + r * 64 + lane] = acc[r];
    }
    __syncthreads();
    if (grp > 0) return;
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[r] += red[wave * 1024 + r * 64 + lane];
    // Accumulator layout of a 32x32 block: element r of lane l sits at
    // row 8*(r/4) + 4*(l/32) + r%4, column l%32.
    float* __restrict__ C = g.C + coff;
    const float* R = g.R ? g.R + coff : C;
    const int ldr = g.R ? g.ldr : g.ldc;
    const int col = n0 + wn + lr;
    if (col >= N) return;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
        const int row = m0 + wm + 8 * (r >> 2) + 4 * lk + (r & 3);
        if (row < M) {   // streamed out, not left dirty in L2 for the kernel's end
            const float v = g.alpha * acc[r];
            __builtin_nontemporal_store((g.beta != 0.f) ? v + g.beta * R[static_cast<long long>(row) * ldr + col] : v,
                                        &C[static_cast<long long>(row) * g.ldc + col]);
        }
    }
}

// ---------------------------------------------------------------------------
// Skinny products (M <= 32 rows of C, B stored K x N): the work is one
// streaming pass over B, HBM-bound.  With one or two rows of C this VALU form
// streams B (2 to 4 FMAs per float4 of B); three to 32 rows take the MFMA
// form below, since at 16 rows the 64 FMAs per float4 outrun the VALU (packed
// fp32 is not used).  Each wave covers 256 columns with one float4 per lane.  The workgroup walks its K slice in chunks of kSkinnyKC
// rows: the chunk of A is staged in LDS as [k][m] (zero past M and past the
// slice), then wave w streams rows [w*KC/4, (w+1)*KC/4) of the chunk, U rows of
// B in flight, reading the M values of A of a row as broadcast LDS reads.
// Waves 1..3 hand their sums to wave 0 through LDS, added in wave order.  A K
// split over blockIdx.y writes [split][M][N] partials that splitk_reduce adds
// in split order.
constexpr int kSkinnyMax = 32;
constexpr int kSkinnyCols = 256;    // columns per workgroup (64 lanes x float4)
constexpr int kSkinnyKC = 256;      // K rows of A staged per chunk

template <int MS, bool TA, bool VEC>
__global__ void __launch_bounds__(256)
sgemm_skinny_kernel(const GemmArgs g)
{
    constexpr int U = MS >= 8 ? 4 : 8;
    constexpr int KC = kSkinnyKC;
    static_assert(KC % (4 * U) == 0, "a chunk must split into whole U-row steps per wave");
    constexpr int kRed = 3 * MS * 64;                    // float4s: waves 1..3 x MS rows x 64 lanes
    constexpr int kTab = KC * MS / 4;                    // float4s: A chunk [KC][MS]
    __shared__ float4 smem[kRed > kTab ? kRed : kTab];
    float* atab = reinterpret_cast<float*>(smem);
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int M = g.M, N = g.N;
    const int n0 = blockIdx.x * kSkinnyCols + 4 * lane;
    const int k0 = blockIdx.y * g.kchunk;
    const int k1 = min(g.K, k0 + g.kchunk);
    const bool colfull = VEC && n0 + 3 < N;
    float4 acc[MS];
#pragma unroll
    for (int m = 0; m < MS; ++m) acc[m] = make_float4(0.f, 0.f, 0.f, 0.f);
    for (int kc0 = k0; kc0 < k1; kc0 += KC) {
        const int nk = min(KC, k1 - kc0);
        for (int i = tid; i < KC * MS; i += 256) {
            const int c = TA ? i / MS : i % KC;
            const int m = TA ? i % MS : i / KC;
            float v = 0.f;
            if (c < nk && m < M)
                v = TA ? g.A[static_cast<long long>(kc0 + c) * g.lda + m]
                       : g.A[static_cast<long long>(m) * g.lda + kc0 + c];
            atab[c * MS + m] = v;
        }
        __syncthreads();
        const int rpw = (nk + 4 * U - 1) / (4 * U) * U;   // rows per wave in this chunk
        const int rb = wv * rpw;
        const int re = min(rb + rpw, nk);
        for (int r = rb; r < re; r += U) {
            float4 b[U];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                b[u] = make_float4(0.f, 0.f, 0.f, 0.f);
                if (r + u < re) {
                    const float* src = g.B + static_cast<long long>(kc0 + r + u) * g.ldb + n0;
                    if (colfull) {
                        const floatx4 v = __builtin_nontemporal_load(reinterpret_cast<const floatx4*>(src));
                        b[u] = make_float4(v.x, v.y, v.z, v.w);
                    } else {
                        b[u].x = n0 + 0 < N ? src[0] : 0.f;
                        b[u].y = n0 + 1 < N ? src[1] : 0.f;
                        b[u].z = n0 + 2 < N ? src[2] : 0.f;
                        b[u].w = n0 + 3 < N ? src[3] : 0.f;
                    }
                }
            }
            // rows past the slice hold zeros in both atab and b
#pragma unroll
            for (int u = 0; u < U; ++u) {
                float a[MS];
                const float* arow = atab + (r + u) * MS;
                if constexpr (MS >= 4) {
#pragma unroll
                    for (int q = 0; q < MS / 4; ++q) {
                        const float4 t = reinterpret_cast<const float4*>(arow)[q];
                        a[4 * q] = t.x; a[4 * q + 1] = t.y; a[4 * q + 2] = t.z; a[4 * q + 3] = t.w;
                    }
                } else {
#pragma unroll
                    for (int m = 0; m < MS; ++m) a[m] = arow[m];
                }
#pragma unroll
                for (int m = 0; m < MS; ++m) {
                    acc[m].x += a[m] * b[u].x;
                    acc[m].y += a[m] * b[u].y;
                    acc[m].z += a[m] * b[u].z;
                    acc[m].w += a[m] * b[u].w;
                }
            }
        }
        __syncthreads();   // atab is rewritten by the next chunk (and reused below)
    }
    if (wv > 0) {
#pragma unroll
        for (int m = 0; m < MS; ++m) smem[((wv - 1) * MS + m) * 64 + lane] = acc[m];
    }
    __syncthreads();
    if (wv != 0) return;
#pragma unroll
    for (int m = 0; m < MS; ++m) {
#pragma unroll
        for (int w = 0; w < 3; ++w) {
            const float4 t = smem[(w * MS + m) * 64 + lane];
            acc[m].x += t.x; acc[m].y += t.y; acc[m].z += t.z; acc[m].w += t.w;
        }
    }
    const bool split = g.splits > 1;
    float* base = split ? g.ws + static_cast<long long>(blockIdx.y) * M * N : g.C;
    const int ld = split ? N : g.ldc;
    const bool vst = colfull && (split ? (N % 4 == 0) : (g.ldc % 4 == 0 && (reinterpret_cast<uintptr_t>(g.C) & 15u) == 0));
#pragma unroll
    for (int m = 0; m < MS; ++m) {
        if (m < M) {
            float v[4] = {acc[m].x, acc[m].y, acc[m].z, acc[m].w};
            float* dst = base + static_cast<long long>(m) * ld + n0;
            if (!split) {
                const float* rr = g.R ? g.R + static_cast<long long>(m) * g.ldr + n0 : dst;
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (n0 + e < N) v[e] = g.alpha * v[e] + (g.beta != 0.f ? g.beta * rr[e] : 0.f);
            }
            if (vst) {
                *reinterpret_cast<float4*>(dst) = make_float4(v[0], v[1], v[2], v[3]);
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (n0 + e < N) dst[e] = v[e];
            }
        }
    }
}

// Skinny products with 3..32 rows of C on the matrix cores.  The VALU form
// above would spend up to 32 FMAs per float4 of B, more than the VALU issues at
// HBM rate; v_mfma_f32_16x16x4f32 covers 16 rows at once, and MG groups of 16
// rows (MG = ceil(M / 16)) reuse each float4 of B for 4 * MG MFMAs.  Each wave
// covers 64 columns: lane (q = l/16, p = l%16) loads the float4
// B[k][c0+4p .. c0+4p+3] of row k = k0 + 4s + q of step s (four 256-byte row
// segments per step), and MFMA e (e = 0..3) multiplies element e of it, so MFMA
// e computes the columns c0 + 4p + e with A[16g + p][k] as its A operand (zero
// past M).  Accumulator register r of MFMA e then holds C[16g + 4q + r][c0 + 4p
// + e]: each lane owns 4x4 blocks, stored as float4 rows.  Splits as in the
// VALU form.
constexpr int kSkinnyMfmaCols = 64;

// A is staged in LDS per chunk of KC K rows (loading it per step, MG scalar
// loads a lane per 4-row step each touching 16 rows, measured 6% slower at 16
// rows).  Eight
// waves (two per SIMD) take the 4-row steps w, w + 8, ... of a chunk.  A chunk
// is loaded as float4 along k (thread (m, k4): A[m][kc + 4k4 .. +3]) and written
// k-major As[k][m] with row stride 80 (16k + m spreads a wave's writes and the
// operand reads As[(4s + q) * 80 + 16g + p] over all 64 banks).  The next
// chunk's A and B are loaded into a second register set before the current
// chunk's MFMAs.  The waves' sums meet in two fixed rounds (waves 4..7 into
// 0..3, then 1..3 into 0).
constexpr int kSkinnyKCA = 128;
constexpr int kSkinnyLdsA = 80;
constexpr int kSkinnyLdsWaves = 8;

template <bool TA, bool VEC, int MG>
__global__ void __launch_bounds__(64 * kSkinnyLdsWaves)
sgemm_skinny_mfma_lds_kernel(const GemmArgs g)
{
    constexpr int NW = kSkinnyLdsWaves;
    constexpr int NT = 64 * NW;
    constexpr int KC = kSkinnyKCA;
    constexpr int U = KC / (4 * NW);                    // 4-row steps per wave per chunk
    constexpr int UA = 16 * MG * (KC / 4) / NT;         // A float4 units per thread per chunk
    static_assert(UA >= 1 && 16 * MG * (KC / 4) % NT == 0, "A chunk units must split evenly");
    // one LDS region for the A chunks and, after the last chunk, the waves' sums
    constexpr int kAs = KC * kSkinnyLdsA;               // floats
    constexpr int kRed = 4 * 4 * MG * 64 * 4;           // floats: 4 waves' partial tiles
    __shared__ floatx4 lds[(kAs > kRed ? kAs : kRed) / 4];
    float* As = reinterpret_cast<float*>(lds);
    floatx4 (*red)[4 * MG][64] = reinterpret_cast<floatx4 (*)[4 * MG][64]>(lds);
    const int lane = threadIdx.x & 63;
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int p = lane & 15, q = lane >> 4;
    const int M = g.M, N = g.N;
    const int col = blockIdx.x * kSkinnyMfmaCols + 4 * p;
    const int k0 = blockIdx.y * g.kchunk;
    const int k1 = min(g.K, k0 + g.kchunk);
    const bool colfull = VEC && col + 3 < N;
    floatx4 acc[MG][4];
#pragma unroll
    for (int gi = 0; gi < MG; ++gi)
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[gi][e] = floatx4{0.f, 0.f, 0.f, 0.f};

    struct Chunk { float4 b[U]; float a[UA][4]; };
    auto load = [&](Chunk& c, int kc) {
        const int kn = min(KC, k1 - kc);
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int kl = 4 * (wv + NW * u) + q;
            c.b[u] = make_float4(0.f, 0.f, 0.f, 0.f);
            if (kl < kn) {
                const float* src = g.B + static_cast<long long>(kc + kl) * g.ldb + col;
                if (colfull) {
                    const floatx4 v = __builtin_nontemporal_load(reinterpret_cast<const floatx4*>(src));
                    c.b[u] = make_float4(v.x, v.y, v.z, v.w);
                } else {
                    c.b[u].x = col + 0 < N ? src[0] : 0.f;
                    c.b[u].y = col + 1 < N ? src[1] : 0.f;
                    c.b[u].z = col + 2 < N ? src[2] : 0.f;
                    c.b[u].w = col + 3 < N ? src[3] : 0.f;
                }
            }
        }
#pragma unroll
        for (int j = 0; j < UA; ++j) {
            const int idx = threadIdx.x + NT * j;
            const int m = idx % (16 * MG), k4 = idx / (16 * MG);
            if (!TA && g.vecA && m < M && 4 * k4 + 3 < kn) {   // kc is a multiple of 4
                const float4 v = *reinterpret_cast<const float4*>(g.A + static_cast<long long>(m) * g.lda + kc + 4 * k4);
                c.a[j][0] = v.x; c.a[j][1] = v.y; c.a[j][2] = v.z; c.a[j][3] = v.w;
                continue;
            }
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int kl = 4 * k4 + e;
                c.a[j][e] = (m < M && kl < kn)
                                ? (TA ? g.A[static_cast<long long>(kc + kl) * g.lda + m]
                                      : g.A[static_cast<long long>(m) * g.lda + kc + kl])
                                : 0.f;
            }
        }
    };
    auto consume = [&](const Chunk& c, int kc) {
        const int kn = min(KC, k1 - kc);
        __syncthreads();   // the previous chunk's operand reads are done
#pragma unroll
        for (int j = 0; j < UA; ++j) {
            const int idx = threadIdx.x + NT * j;
            const int m = idx % (16 * MG), k4 = idx / (16 * MG);
#pragma unroll
            for (int e = 0; e < 4; ++e) As[(4 * k4 + e) * kSkinnyLdsA + m] = c.a[j][e];
        }
        __syncthreads();
        return kn;
    };
    auto mma = [&](const Chunk& c, int kn) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int st = wv + NW * u;
            if (4 * st >= kn) break;                     // uniform
            const float* ar = As + (4 * st + q) * kSkinnyLdsA + p;
#pragma unroll
            for (int gi = 0; gi < MG; ++gi) {
                const float a = ar[16 * gi];
                acc[gi][0] = __builtin_amdgcn_mfma_f32_16x16x4f32(a, c.b[u].x, acc[gi][0], 0, 0, 0);
                acc[gi][1] = __builtin_amdgcn_mfma_f32_16x16x4f32(a, c.b[u].y, acc[gi][1], 0, 0, 0);
                acc[gi][2] = __builtin_amdgcn_mfma_f32_16x16x4f32(a, c.b[u].z, acc[gi][2], 0, 0, 0);
                acc[gi][3] = __builtin_amdgcn_mfma_f32_16x16x4f32(a, c.b[u].w, acc[gi][3], 0, 0, 0);
            }
        }
    };
    // two register sets: chunk c + 1 is loaded while chunk c runs its MFMAs
    if (k0 < k1) {
        Chunk c0, c1;
        load(c0, k0);
        for (int kc = k0; kc < k1; kc += 2 * KC) {
            int kn = consume(c0, kc);
            if (kc + KC < k1) load(c1, kc + KC);
            mma(c0, kn);
            if (kc + KC >= k1) break;
            kn = consume(c1, kc + KC);
            if (kc + 2 * KC < k1) load(c0, kc + 2 * KC);
            mma(c1, kn);
        }
    }
    __syncthreads();   // the last chunk's operand reads are done: the region becomes the hand-off
    if (wv >= 4) {
#pragma unroll
        for (int gi = 0; gi < MG; ++gi)
#pragma unroll
            for (int e = 0; e < 4; ++e) red[wv - 4][4 * gi + e][lane] = acc[gi][e];
    }
    __syncthreads();
    if (wv < 4) {
#pragma unroll
        for (int gi = 0; gi < MG; ++gi)
#pragma unroll
            for (int e = 0; e < 4; ++e) acc[gi][e] += red[wv][4 * gi + e][lane];
    }
    __syncthreads();
    if (wv >= 1 && wv < 4) {
#pragma unroll
        for (int gi = 0; gi < MG; ++gi)
#pragma unroll
            for (int e = 0; e < 4; ++e) red[wv - 1][4 * gi + e][lane] = acc[gi][e];
    }
    __syncthreads();
    if (wv != 0) return;
#pragma unroll
    for (int gi = 0; gi < MG; ++gi)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
#pragma unroll
            for (int w = 0; w < 3; ++w) acc[gi][e] += red[w][4 * gi + e][lane];
        }
    const bool split = g.splits > 1;
    float* base = split ? g.ws + static_cast<long long>(blockIdx.y) * M * N : g.C;
    const int ld = split ? N : g.ldc;
    const bool vst = colfull && (split ? (N % 4 == 0) : (g.ldc % 4 == 0 && (reinterpret_cast<uintptr_t>(g.C) & 15u) == 0));
#pragma unroll
    for (int gr = 0; gr < 4 * MG; ++gr) {
        const int gi = gr >> 2, r = gr & 3;
        const int row = 16 * gi + 4 * q + r;
        if (row >= M) continue;
        float v[4] = {acc[gi][0][r], acc[gi][1][r], acc[gi][2][r], acc[gi][3][r]};
        float* dst = base + static_cast<long long>(row) * ld + col;
        if (!split) {
            const float* rr = g.R ? g.R + static_cast<long long>(row) * g.ldr + col : dst;
#pragma unroll
            for (int e = 0; e < 4; ++e)
                if (col + e < N) v[e] = g.alpha * v[e] + (g.beta != 0.f ? g.beta * rr[e] : 0.f);
        }
        if (vst) {
            *reinterpret_cast<float4*>(dst) = make_float4(v[0], v[1], v[2], v[3]);
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e)
                if (col + e < N) dst[e] = v[e];
        }
    }
}

// ---------------------------------------------------------------------------
// Tiny problems (fewer 32x32 output tiles than CUs, e.g. the 512x128 outputs
// of the C2 step): one workgroup per 16x16 output tile, four times as many
// workgroups as the 32x32 kernel, so the fp32 MFMA work (64 cycles per
// 32x32x2 or 32 per 16x16x4 instruction and SIMD) spreads over more CUs.
// Same scheme as the small kernel with v_mfma_f32_16x16x4f32: for a 16-deep
// K step at k0, lane l (row or column l%16, group q = l/16) holds
// op(A)[row][k0+4q .. k0+4q+3] and op(B)[k0+4q .. k0+4q+3][col]; MFMA i of the
// step multiplies element i of both, so its four k slots (one per lane group)
// are k0+4q+i and the four MFMAs cover k0 .. k0+15 exactly once.  The NW
// waves (4, or 8 for one-pass slices deeper than 256) take the 16-deep steps
// w, w+NW, ...; their tiles are summed in LDS in wave order.  Steps wholly
// past the end of K issue no MFMA.  BR as above.
template <bool TA, bool TB, bool BR, bool PIPE, int NW = 4>
__global__ void __launch_bounds__(64 * NW)
sgemm_tiny_kernel(const GemmArgs g)
{
    __shared__ float red[NW][4][64];
    const int M = g.M, N = g.N;
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    // wave-uniform (readfirstlane): the K-step bounds below become scalar
    // branches, so a pass's loads issue back to back with no exec-mask joins
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lr = lane & 15;
    const int q = lane >> 4;
    int tm, tn;
    xcd_tile(blockIdx.x, gridDim.x, g.tiles_n, tm, tn);
    const int m0 = tm * 16, n0 = tn * 16;
    const long long zo = blockIdx.y / g.inner, zi = blockIdx.y % g.inner;
    const float* __restrict__ A = g.A + zo * g.sA2 + zi * g.sA;
    const float* __restrict__ B = g.B + zo * g.sB2 + zi * g.sB;
    const long long coff = zo * g.sC2 + zi * g.sC;
    const int kbeg = blockIdx.z * g.kchunk;
    const int kend = min(g.K, kbeg + g.kchunk);
    const int row = m0 + lr;
    const int col = n0 + lr;
    const bool rok = row < M, cok = col < N;
    // rows / columns past the edge load from row / column 0 (a valid address)
    const int rowc = rok ? row : 0, colc = cok ? col : 0;

    floatx4 acc;
#pragma unroll
    for (int r = 0; r < 4; ++r) acc[r] = 0.f;

    // A pass covers the wave's next U 16-deep steps; with more than one pass
    // the next pass's loads are issued before this pass's MFMAs (two register
    // sets), so the passes' load latencies overlap.
    constexpr int U = kSmallU;
    auto load_pass = [&](int kp, float (&a)[U][4], float (&b)[U][4]) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int ks = kp + 16 * NW * u;                 // wave-uniform step start
            const bool live = ks < kend;                // uniform
            // Without a second pass to overlap, steps past the end are skipped
            // by a scalar branch.  A pipelined pass keeps a fixed load count
            // (the wait before the previous pass's MFMAs counts them): its dead
            // steps load from kbeg and are zeroed.
            if (!PIPE && !live) break;
            const int kl = live ? ks + 4 * q : kbeg;
            const bool sfull = live && ks + 16 <= kend; // uniform: every lane's four k are in range
            const int kend_l = live ? kend - kl : 0;
            int kb = kl;
            const float* __restrict__ Ab = A;
            const float* __restrict__ Bb = B;
            if (BR) {
                // block of this k: with Kb % 16 == 0 a 16-deep step lies in one
                // block, so the index is the wave-uniform step start's
                const int j = (g.Kb % 16 == 0 && live) ? ks / g.Kb : kl / g.Kb;
                kb = kl - j * g.Kb;
                Ab = A + j * g.sAk;
                Bb = B + j * g.sBk;
            }
            // Rows of A past M and columns of B past N only reach outputs that
            // are not stored, so they load from row / column 0 unmasked; only
            // k past the end (the last step) must contribute zeros.
            if (!TA) {
                const float* src = Ab + static_cast<long long>(rowc) * g.lda + kb;
                if (sfull && g.vecA) {
                    const float4 v = *reinterpret_cast<const float4*>(src);
                    a[u][0] = v.x; a[u][1] = v.y; a[u][2] = v.z; a[u][3] = v.w;
                } else if (sfull) {
#pragma unroll
                    for (int i = 0; i < 4; ++i) a[u][i] = src[i];
                } else {
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        const float v = src[i < kend_l ? i : 0];
                        a[u][i] = i < kend_l ? v : 0.f;
                    }
                }
            } else {
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const bool ok = sfull || i < kend_l;
                    const float v = Ab[static_cast<long long>(ok ? kb + i : kbeg) * g.lda + rowc];
                    a[u][i] = (sfull || ok) ? v : 0.f;
                }
            }
            if (!TB) {
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const bool ok = sfull || i < kend_l;
                    const float v = Bb[static_cast<long long>(ok ? kb + i : kbeg) * g.ldb + colc];
                    b[u][i] = (sfull || ok) ? v : 0.f;
                }
            } else {
                const float* src = Bb + static_cast<long long>(colc) * g.ldb + kb;
                if (sfull && g.vecB) {
                    const float4 v = *reinterpret_cast<const float4*>(src);
                    b[u][0] = v.x; b[u][1] = v.y; b[u][2] = v.z; b[u][3] = v.w;
                } else if (sfull) {
#pragma unroll
                    for (int i = 0; i < 4; ++i) b[u][i] = src[i];
                } else {
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        const float v = src[i < kend_l ? i : 0];
                        b[u][i] = i < kend_l ? v : 0.f;
                    }
                }
            }
        }
    };
    // Pipelined passes (K > 512) keep the per-element guarded loads: with
    // them the compiler overlaps the next pass's loads with this pass's MFMAs
    // (measured: 15 us for the C2 dxf product against 23 us with the
    // unmasked loads above).
    auto load_pass_guarded = [&](int kp, float (&a)[U][4], float (&b)[U][4]) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int kl = kp + 16 * NW * u + 4 * q;
            const bool kfull = kl + 3 < kend;
            const int kend_l = kend - kl;
            int kb = kl;
            const float* __restrict__ Ab = A;
            const float* __restrict__ Bb = B;
            if (BR) {
                // block of this k: with Kb % 16 == 0 a 16-deep step lies in one
                // block, so the index is the wave-uniform step start's
                int j;
                if (g.Kb % 16 == 0) {
                    const int ks = __builtin_amdgcn_readfirstlane(kp + 16 * NW * u);
                    j = ks / g.Kb;
                } else {
                    j = kl / g.Kb;
                }
                kb = kl - j * g.Kb;
                Ab = A + j * g.sAk;
                Bb = B + j * g.sBk;
            }
            if (!TA) {
                const float* src = Ab + static_cast<long long>(row) * g.lda + kb;
                if (g.vecA && rok && kfull) {
                    const float4 v = *reinterpret_cast<const float4*>(src);
                    a[u][0] = v.x; a[u][1] = v.y; a[u][2] = v.z; a[u][3] = v.w;
                } else {
#pragma unroll
                    for (int i = 0; i < 4; ++i) a[u][i] = (rok && i < kend_l) ? src[i] : 0.f;
                }
            } else {
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    a[u][i] = (rok && i < kend_l) ? Ab[static_cast<long long>(kb + i) * g.lda + row] : 0.f;
            }
            if (!TB) {
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    b[u][i] = (cok && i < kend_l) ? Bb[static_cast<long long>(kb + i) * g.ldb + col] : 0.f;
            } else {
                const float* src = Bb + static_cast<long long>(col) * g.ldb + kb;
                if (g.vecB && cok && kfull) {
                    const float4 v = *reinterpret_cast<const float4*>(src);
                    b[u][0] = v.x; b[u][1] = v.y; b[u][2] = v.z; b[u][3] = v.w;
                } else {
#pragma unroll
                    for (int i = 0; i < 4; ++i) b[u][i] = (cok && i < kend_l) ? src[i] : 0.f;
                }
            }
        }
    };
    // When every live step of the pass is a full 16-deep step (the slice
    // length kend - kbeg a multiple of 16: steps start at kbeg + 16j, so a
    // step that starts before kend also ends by it), the operands' contiguous
    // loads are float4-aligned and, for
    // batch-reduce, a step never straddles a block, the pass loads with no
    // selects: each load's register is final, dead steps are skipped by
    // wave-uniform branches, and all the pass's loads issue before the first
    // wait.
    const bool fast_ops = (TA || g.vecA) && (!TB || g.vecB) && (!BR || g.Kb % 16 == 0);
    auto load_pass_full = [&](int kp, float (&a)[U][4], float (&b)[U][4]) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int ks = kp + 16 * NW * u;
            if (ks >= kend) break;
            const int kl = ks + 4 * q;
            int kb = kl;
            const float* __restrict__ Ab = A;
            const float* __restrict__ Bb = B;
            if (BR) {
                const int j = ks / g.Kb;
                kb = kl - j * g.Kb;
                Ab = A + j * g.sAk;
                Bb = B + j * g.sBk;
            }
            if (!TA) {
                const float4 v = *reinterpret_cast<const float4*>(Ab + static_cast<long long>(rowc) * g.lda + kb);
                a[u][0] = v.x; a[u][1] = v.y; a[u][2] = v.z; a[u][3] = v.w;
            } else {
#pragma unroll
                for (int i = 0; i < 4; ++i) a[u][i] = Ab[static_cast<long long>(kb + i) * g.lda + rowc];
            }
            if (!TB) {
#pragma unroll
                for (int i = 0; i < 4; ++i) b[u][i] = Bb[static_cast<long long>(kb + i) * g.ldb + colc];
            } else {
                const float4 v = *reinterpret_cast<const float4*>(Bb + static_cast<long long>(colc) * g.ldb + kb);
                b[u][0] = v.x; b[u][1] = v.y; b[u][2] = v.z; b[u][3] = v.w;
            }
        }
    };
    auto mma_pass = [&](int kp, const float (&a)[U][4], const float (&b)[U][4]) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (kp + 16 * NW * u >= kend) break;   // wave-uniform: nothing left in this pass
#pragma unroll
            for (int i = 0; i < 4; ++i) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a[u][i], b[u][i], acc, 0, 0, 0);
        }
    };
    int kp = kbeg + 16 * wave;
    if (!PIPE) {   // K fits one pass: one register set
        if (fast_ops && (kend - kbeg) % 16 == 0 && kp < kend) {
            float a0[U][4], b0[U][4];
            load_pass_full(kp, a0, b0);
            __builtin_amdgcn_sched_barrier(0);   // keep every load ahead of the first MFMA
#pragma unroll
            for (int u = 0; u < U; ++u) {
                if (kp + 16 * NW * u >= kend) break;
#pragma unroll
                for (int i = 0; i < 4; ++i) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a0[u][i], b0[u][i], acc, 0, 0, 0);
            }
        } else if (kp < kend) {
            float a0[U][4], b0[U][4];
            load_pass(kp, a0, b0);
            mma_pass(kp, a0, b0);
        }
    } else if (kp < kend) {
        float a0[U][4], b0[U][4], a1[U][4], b1[U][4];
        load_pass_guarded(kp, a0, b0);
        while (true) {
            const int k1 = kp + 16 * NW * U;
            if (k1 < kend) load_pass_guarded(k1, a1, b1);
            mma_pass(kp, a0, b0);
            if (k1 >= kend) break;
            const int k2 = k1 + 16 * NW * U;
            if (k2 < kend) load_pass_guarded(k2, a0, b0);
            mma_pass(k1, a1, b1);
            if (k2 >= kend) break;
            kp = k2;
        }
    }

    // thread (wave w < 4, lane l) finishes accumulator register w of lane l,
    // summing the NW waves' partial tiles in wave order
#pragma unroll
    for (int r = 0; r < 4; ++r) red[wave][r][lane] = acc[r];
    __syncthreads();
    if (wave >= 4) return;
    float v = red[0][wave][lane];
#pragma unroll
    for (int w = 1; w < NW; ++w) v += red[w][wave][lane];
    const int orow = m0 + 4 * q + wave;
    const int ocol = n0 + lr;
    if (orow >= M || ocol >= N) return;
    if (g.splits > 1) {
        float* wz = g.ws + (static_cast<long long>(blockIdx.z) * gridDim.y + blockIdx.y) * (static_cast<long long>(M) * N);
        wz[static_cast<long long>(orow) * N + ocol] = v;
        return;
    }
    float* __restrict__ C = g.C + coff;
    const float* R = g.R ? g.R + coff : C;
    const int ldr = g.R ? g.ldr : g.ldc;
    const float o = g.alpha * v;
    C[static_cast<long long>(orow) * g.ldc + ocol] =
        (g.beta != 0.f) ? o + g.beta * R[static_cast<long long>(orow) * ldr + ocol] : o;
}

// Eight waves share K once it is long enough for each to get a full pass.
// PIPE: K needs more than one pass of the four waves (64 * kSmallU deep)
template <bool PIPE, int NW>
void launch_tiny_t(int ta, int tb, const GemmArgs& g, dim3 grid, hipStream_t stream)
{
    const dim3 block(64 * NW);
    if (g.Kb != g.K) {
        if (!tb) klaunch(sgemm_tiny_kernel<false, false, true, PIPE, NW>, grid, block, 0, stream, g);
        else klaunch(sgemm_tiny_kernel<false, true, true, PIPE, NW>, grid, block, 0, stream, g);
    } else if (!ta && !tb) klaunch(sgemm_tiny_kernel<false, false, false, PIPE, NW>, grid, block, 0, stream, g);
    else if (ta && !tb) klaunch(sgemm_tiny_kernel<true, false, false, PIPE, NW>, grid, block, 0, stream, g);
    else if (!ta && tb) klaunch(sgemm_tiny_kernel<false, true, false, PIPE, NW>, grid, block, 0, stream, g);
    else klaunch(sgemm_tiny_kernel<true, true, false, PIPE, NW>, grid, block, 0, stream, g);
}

int launch_tiny(int ta, int tb, GemmArgs g, int batch, hipStream_t stream)
{
    g.tiles_m = ceil_div(g.M, 16);
    g.tiles_n = ceil_div(g.N, 16);
    const long long nwg = static_cast<long long>(g.tiles_m) * g.tiles_n;
    if (nwg > 0x7fffffffLL) return fail(LHIP_E_CAPACITY, "sgemm: %lld workgroups exceed the grid limit", nwg);
    if (g.splits <= 1) { g.splits = 1; g.kchunk = g.K; g.ws = nullptr; }
    dim3 grid(static_cast<unsigned>(nwg), batch, g.splits);
    // one pass of four waves covers 64 * kSmallU of K; a one-pass slice deeper
    // than 256 runs on eight waves (half the loads and MFMAs per wave)
    if (g.kchunk > 64 * kSmallU) launch_tiny_t<true, 4>(ta, tb, g, grid, stream);
    else if (g.kchunk > 256) launch_tiny_t<false, 8>(ta, tb, g, grid, stream);
    else launch_tiny_t<false, 4>(ta, tb, g, grid, stream);
    int rc = check_launch("sgemm (tiny): kernel launch");
    if (rc != LHIP_OK || g.splits <= 1 || g.skip_reduce) return rc;
    return launch_reduce(g, batch, stream);
}

// Skinny path: M <= 32, B not transposed, one product (no batch, no
// batch-reduce), at least one full wave of columns.
bool skinny_ok(int ta, int tb, int m, int n, int batch, int kblocks)
{
    (void)ta;
    return !tb && m >= 1 && m <= kSkinnyMax && n >= kSkinnyCols && batch == 1 && kblocks == 1;
}

// Rows of C up to which the VALU form is used; 3..32 rows take the MFMA form.
constexpr int kSkinnyValuMax = 2;

}  // namespace

// K slices of the skinny path: about two workgroups per CU, at least 64 K rows
// per workgroup, and partials (written, then read back by the reduce) at most
// a quarter of B's bytes: 2 * s * m * n <= k * n / 4.
int skinny_plan(int m, int n, int k, size_t ws_floats, int* kchunk_out)
{
    const int cus = st().cu_count > 0 ? st().cu_count : 256;
    const long long cb = ceil_div(n, m <= kSkinnyValuMax ? kSkinnyCols : kSkinnyMfmaCols);
    // about two workgroups per CU for the VALU form and the one-group (M <= 16)
    // MFMA form; one for the eight-wave MFMA form on two groups (M = 4, 8, 16
    // at K = N = 4096: 24.1, 24.5, 21.1 us on one per CU, 19.6, 19.6, 19.3 on
    // two; M = 32: 29.2 on one, 30.7 on two)
    const long long per_cu = m <= 16 ? 2 : 1;
    long long s = (per_cu * cus + cb - 1) / cb;
    s = std::min<long long>(s, k / 64);
    s = std::min<long long>(s, std::max<long long>(1, k / (8LL * m)));
    const long long mn = static_cast<long long>(m) * n;
    if (mn > 0) s = std::min<long long>(s, static_cast<long long>(ws_floats / mn));
    if (s < 2) {
        *kchunk_out = k;
        return 1;
    }
    const int kchunk = ceil_div(ceil_div(k, s), 4) * 4;
    *kchunk_out = kchunk;
    return ceil_div(k, kchunk);
}

namespace {

template <bool TA, bool VEC>
void launch_skinny_t(const GemmArgs& g, dim3 grid, hipStream_t stream)
{
    if (g.M == 1) klaunch(sgemm_skinny_kernel<1, TA, VEC>, grid, 256, 0, stream, g);
    else klaunch(sgemm_skinny_kernel<2, TA, VEC>, grid, 256, 0, stream, g);
}

int launch_skinny(int ta, GemmArgs g, hipStream_t stream)
{
    g.kchunk = g.K;
    g.splits = g.ws ? skinny_plan(g.M, g.N, g.K, g.ws_floats_avail, &g.kchunk) : 1;
    if (g.splits <= 1) { g.splits = 1; g.kchunk = g.K; }
    const bool vec = g.vecB;
    if (g.M <= kSkinnyValuMax) {
        const dim3 grid(ceil_div(g.N, kSkinnyCols), g.splits);
        if (ta) { if (vec) launch_skinny_t<true, true>(g, grid, stream); else launch_skinny_t<true, false>(g, grid, stream); }
        else { if (vec) launch_skinny_t<false, true>(g, grid, stream); else launch_skinny_t<false, false>(g, grid, stream); }
    } else {
        const dim3 grid(ceil_div(g.N, kSkinnyMfmaCols), g.splits);
        auto go = [&](auto mgc) {
            constexpr int MG = decltype(mgc)::value;
            constexpr int T = 64 * kSkinnyLdsWaves;
            if (ta) {
                if (vec) klaunch(sgemm_skinny_mfma_lds_kernel<true, true, MG>, grid, T, 0, stream, g);
                else klaunch(sgemm_skinny_mfma_lds_kernel<true, false, MG>, grid, T, 0, stream, g);
            } else {
                if (vec) klaunch(sgemm_skinny_mfma_lds_kernel<false, true, MG>, grid, T, 0, stream, g);
                else klaunch(sgemm_skinny_mfma_lds_kernel<false, false, MG>, grid, T, 0, stream, g);
            }
        };
        if (g.M <= 16) go(std::integral_constant<int, 1>{});
        else go(std::integral_constant<int, 2>{});
    }
    int rc = check_launch("sgemm (skinny): kernel launch");
    if (rc != LHIP_OK || g.splits <= 1) return rc;
    return launch_reduce(g, 1, stream);
}

// One 64x64 tile per CU at most, whole 32-deep chunks of a short K and
// operands whose rows take float4 loads: the fp32 cores and one load round trip
// beat the conversion and the deeper pipeline of the three-term kernel (the C2
// step's tied head, 512x2000x128: 6.1 us against 7.9; 64 batches of
// 256x64x256: 11.3-12.4 us against 12.3-12.9; past K = 256 the three-term
// kernel is faster: 2048x512x512 13.6 against 14.8).  M and N need not be whole tiles: rows and columns past them
// are clamped into the operands.
bool ks_best(int ta, int tb, int m, int n, int k, int batch, int vecA, int vecB)
{
    const int cus = st().cu_count > 0 ? st().cu_count : 256;
    const long long tiles64 = static_cast<long long>(ceil_div(m, kKsTile)) * ceil_div(n, kKsTile) * batch;
    return tiles64 <= cus && k <= 256 && k % kKsK == 0 && vecA && vecB && (!ta || m % 4 == 0) && (tb || n % 4 == 0);
}

int launch_ks(int ta, int tb, GemmArgs g, int batch, hipStream_t stream)
{
    g.tiles_m = ceil_div(g.M, kKsTile);
    g.tiles_n = ceil_div(g.N, kKsTile);
    const dim3 grid(static_cast<unsigned>(g.tiles_m) * g.tiles_n, batch, 1), block(2 * kThreads, 1, 1);
    if (!ta && !tb) klaunch(sgemm_mfma_ks_kernel<false, false>, grid, block, 0, stream, g);
    else if (ta && !tb) klaunch(sgemm_mfma_ks_kernel<true, false>, grid, block, 0, stream, g);
    else if (!ta && tb) klaunch(sgemm_mfma_ks_kernel<false, true>, grid, block, 0, stream, g);
    else klaunch(sgemm_mfma_ks_kernel<true, true>, grid, block, 0, stream, g);
    return check_launch("sgemm: kernel launch");
}

}  // namespace

int launch_reduce(const GemmArgs& g, int batch, hipStream_t stream)
{
    const bool vec4 = batch == 1 && g.N % 4 == 0 && g.ldc % 4 == 0 && aligned16(g.C) && aligned16(g.ws) &&
                      (!g.R || (g.ldr % 4 == 0 && aligned16(g.R)));
    if (vec4) {
        const long long total4 = static_cast<long long>(g.M) * g.N / 4;
        long long rg = (total4 + 255) / 256;
        const long long cap = static_cast<long long>(st().cu_count > 0 ? st().cu_count : 256) * 4;
        if (rg > cap) rg = cap;
        klaunch(splitk_reduce4, static_cast<int>(rg), 256, 0, stream, g);
        return check_launch("sgemm: split-K reduce");
    }
    const long long total = static_cast<long long>(g.M) * g.N * batch;
    long long rg = (total + 255) / 256;
    const long long cap = static_cast<long long>(st().cu_count > 0 ? st().cu_count : 256) * 4;
    if (rg > cap) rg = cap;
    klaunch(splitk_reduce, static_cast<int>(rg), 256, 0, stream, g, batch);
    return check_launch("sgemm: split-K reduce");
}

namespace {

// Grouped transposed-A products (the weight gradients of the LMTrain step:
// dW = X^T . dY with X, dY row-major over the same B*T rows, every layer's and
// the tied embedding's in one launch).  Workgroup id -> (group, tile) through
// the groups' first-tile table; each 32x32 tile is computed like
// sgemm_small_kernel<TA, !TB>: NW waves split K into 8-deep steps, lane l
// (row or column l%32, half h = l/32) holding A^T[row][k0+4h..+3] (four loads
// down a column of the stored A, coalesced over the 32 rows) and
// B[k0+4h..+3][col], v_mfma_f32_32x32x2f32, partial tiles summed in LDS in
// wave order.  (Fallback for operands that cannot take float4 loads.)
constexpr int kGroupedTile = 32;

struct GroupedTNArgs {
    GroupedTN e[kGroupedMax];
    int tile0[kGroupedMax + 1];
    int tiles_n[kGroupedMax];
    int ngroups, K;
    ColsumSet cs;     // column sums run by the workgroups after the last tile
    int cs_cb;        // 32-column blocks per column-sum job
    int cs_blocks;    // cs.njobs * cs_cb
    int tp, cp;       // 64x64 kernel: tiles, column-sum workgroups per XCD
    int cs_per_wg;    // 64x64 kernel: column-sum blocks per workgroup
    int do_sc;        // 64x64 kernel: run the groups' scatters
    double* ss_out;   // 64x64 kernel: per-workgroup sums of squares of the stored values (or NULL)
};

template <int NW>
__global__ void __launch_bounds__(64 * NW) sgemm_grouped_tn_kernel(const GroupedTNArgs ga)
{
    __shared__ float red[NW][16][64];
    // XCD-contiguous tiles: workgroups are dispatched round-robin over the 8
    // XCDs, so id p runs on XCD p % 8; XCD x takes the tiles
    // [x*G/8, (x+1)*G/8) (G padded to a multiple of 8), i.e. whole groups and
    // row bands, whose operands then stay in that XCD's L2.
    const int per_xcd = gridDim.x / 8;
    const int id = (blockIdx.x % 8) * per_xcd + blockIdx.x / 8;
    if (id >= ga.tile0[ga.ngroups]) return;   // padding
    int gi = 0;
    for (int i = 1; i < ga.ngroups; ++i)
        if (id >= ga.tile0[i]) gi = i;
    const GroupedTN& e = ga.e[gi];
    const int local = id - ga.tile0[gi];
    const int tm = local / ga.tiles_n[gi], tn = local - tm * ga.tiles_n[gi];
    const int K = ga.K;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, lr = lane & 31, h = lane >> 5;
    const int m0 = tm * kGroupedTile, n0 = tn * kGroupedTile;
    const int row = m0 + lr, col = n0 + lr;
    const bool rok = row < e.M, cok = col < e.N;
    floatx16 acc;
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[r] = 0.f;
    constexpr int U = kSmallU;
    for (int kp = 8 * wave; kp < K; kp += 8 * NW * U) {
        float a[U][4], b[U][4];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int kl = kp + 8 * NW * u + 4 * h;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const bool kin = kl + i < K;
                a[u][i] = (rok && kin) ? e.A[static_cast<long long>(kl + i) * e.lda + row] : 0.f;
                b[u][i] = (cok && kin) ? e.B[static_cast<long long>(kl + i) * e.ldb + col] : 0.f;
            }
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (kp + 8 * NW * u >= K) break;   // wave-uniform
#pragma unroll
            for (int i = 0; i < 4; ++i) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a[u][i], b[u][i], acc, 0, 0, 0);
        }
    }
#pragma unroll
    for (int r = 0; r < 16; ++r) red[wave][r][lane] = acc[r];
    __syncthreads();
    // thread (wave w, lane l) finishes accumulator registers (16/NW)w .. of lane l
    constexpr int RPW = 16 / NW;
    const int ocol = n0 + (lane & 31);
    const int lk = lane >> 5;
#pragma unroll
    for (int q = 0; q < RPW; ++q) {
        const int r = RPW * wave + q;
        float v = red[0][r][lane];
#pragma unroll
        for (int w = 1; w < NW; ++w) v += red[w][r][lane];
        const int orow = m0 + 8 * (r >> 2) + 4 * lk + (r & 3);
        if (orow < e.M && ocol < e.N) e.C[static_cast<long long>(orow) * e.ldc + ocol] = v;
    }
}

// LDS-staged form of the grouped kernel, for groups whose operands allow
// float4 loads (leading dimensions % 4 == 0, 16-byte aligned bases).  Both
// operands are stored K-major (A is K x M, B is K x N), so a 64-deep chunk of
// each is copied into LDS unchanged with float4 loads (four per thread per
// chunk), double-buffered; wave w then runs the 8 MFMA steps of chunk rows
// 16w .. 16w+15 on the whole 32x32 tile, reading each operand fragment as one
// conflict-free ds_read_b32 (lanes 0-31 row k, 32-63 row k+1).  The waves'
// tiles are summed in LDS in wave order.  Workgroups past the last tile run the
// column-sum jobs of ga.cs, one 32-column block each (colsum4_block).
constexpr int kGroupedBK = 64;

__global__ void __launch_bounds__(256) sgemm_grouped_tn_lds_kernel(const GroupedTNArgs ga)
{
    constexpr int T = kGroupedTile, BK = kGroupedBK;
    __shared__ float As[2][BK][T];
    __shared__ float Bs[2][BK][T];
    __shared__ float red[4][16][64];
    const int per_xcd = gridDim.x / 8;
    const int id = (blockIdx.x % 8) * per_xcd + blockIdx.x / 8;
    if (id >= ga.tile0[ga.ngroups]) {
        const int cid = id - ga.tile0[ga.ngroups];
        if (cid >= ga.cs_blocks) return;   // padding
        const int job = cid / ga.cs_cb, cb = cid - job * ga.cs_cb;
        colsum4_block(ga.cs.partial[job], ga.cs.nparts[job], ga.cs.out[job], ga.cs.cols, 32 * cb, ga.cs.acc,
                      reinterpret_cast<float4 (*)[8]>(&red[0][0][0]));
        return;
    }
    int gi = 0;
    for (int i = 1; i < ga.ngroups; ++i)
        if (id >= ga.tile0[i]) gi = i;
    const GroupedTN& e = ga.e[gi];
    const int local = id - ga.tile0[gi];
    const int tm = local / ga.tiles_n[gi], tn = local - tm * ga.tiles_n[gi];
    const int K = ga.K;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, lr = lane & 31, lk = lane >> 5;
    const int m0 = tm * T, n0 = tn * T;
    // chunk loader: thread t covers chunk rows t/8 and t/8 + 32, float4 column (t%8)*4
    const int lrow = tid >> 3, lc4 = (tid & 7) * 4;
    const bool am_ok = m0 + lc4 < e.M, bn_ok = n0 + lc4 < e.N;   // M, N % 4 == 0 (host check)
    float4 ra[2], rb[2];
    auto gload = [&](int k0) {
#pragma unroll
        for (int p = 0; p < 2; ++p) {
            const int k = k0 + lrow + 32 * p;
            const bool kin = k < K;
            ra[p] = (kin && am_ok) ? *reinterpret_cast<const float4*>(e.A + static_cast<long long>(k) * e.lda + m0 + lc4)
                                   : make_float4(0.f, 0.f, 0.f, 0.f);
            rb[p] = (kin && bn_ok) ? *reinterpret_cast<const float4*>(e.B + static_cast<long long>(k) * e.ldb + n0 + lc4)
                                   : make_float4(0.f, 0.f, 0.f, 0.f);
        }
    };
    auto lstore = [&](int buf) {
#pragma unroll
        for (int p = 0; p < 2; ++p) {
            *reinterpret_cast<float4*>(&As[buf][lrow + 32 * p][lc4]) = ra[p];
            *reinterpret_cast<float4*>(&Bs[buf][lrow + 32 * p][lc4]) = rb[p];
        }
    };
    floatx16 acc;
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[r] = 0.f;
    const int nk = (K + BK - 1) / BK;
    gload(0);
    lstore(0);
    __syncthreads();
    for (int kt = 0; kt < nk; ++kt) {
        const int cur = kt & 1;
        const bool more = kt + 1 < nk;
        if (more) gload((kt + 1) * BK);
#pragma unroll
        for (int st = 0; st < 8; ++st) {
            const int kr = 16 * wave + 2 * st + lk;
            acc = __builtin_amdgcn_mfma_f32_32x32x2f32(As[cur][kr][lr], Bs[cur][kr][lr], acc, 0, 0, 0);
        }
        if (more) lstore(cur ^ 1);
        __syncthreads();
    }
#pragma unroll
    for (int r = 0; r < 16; ++r) red[wave][r][lane] = acc[r];
    __syncthreads();
    // thread (wave w, lane l) finishes accumulator registers 4w .. 4w+3 of lane l
    const int ocol = n0 + lr;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const int r = 4 * wave + q;
        const float v = ((red[0][r][lane] + red[1][r][lane]) + red[2][r][lane]) + red[3][r][lane];
        const int orow = m0 + 8 * (r >> 2) + 4 * lk + (r & 3);
        if (orow < e.M && ocol < e.N) e.C[static_cast<long long>(orow) * e.ldc + ocol] = v;
    }
}

// Sum over the workgroup of each thread's double (wave order, then wave 0's
// thread 0 adds the waves in order) into ss_out[blockIdx.x].
template <int NW>
__device__ __forceinline__ void block_sumsq_out(double v, double* ss_out, double* red)
{
    v = wave_sum(v);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    if (threadIdx.x == 0) {
        double t = 0.0;
#pragma unroll
        for (int w = 0; w < NW; ++w) t += red[w];
        ss_out[blockIdx.x] = t;
    }
}

// 64x64 tiles for the same float4-loadable groups.  The tile's 32x32
// quadrants belong to four waves, and KS sets of four waves take the BK-deep
// K chunks in turn (set s: chunks s, s+KS, ..., each set with its own
// double-buffered LDS), so each chain of dependent chunk loads is 1/KS as
// long; the partial quadrants are added in LDS in set order.  KS = 2 with
// 64-deep chunks for short K; KS = 4 with 32-deep chunks from K = 512 on
// (four waves per SIMD: the C2 step's launch, K = 512, 19.3 -> 18.1 us).  At
// the LM step's shapes (K = batch*seq rows) this is about one workgroup per
// CU, and nothing is re-read by a neighbouring tile as often as with 32x32
// tiles.
// Placement: XCD x (blocks b with b % 8 == x) takes tiles [x*tp, (x+1)*tp)
// first and then cp workgroups of column-sum jobs, each running up to
// cs_per_wg 32-column blocks in turn, so no XCD holds more tiles than CUs.
// BUF: the chunk loads are buffer loads whose records end at each operand's
// last element, so rows past K read as zeros from the hardware's range check
// with no branch, and every chunk load is issued on every path (past the last
// chunk a load fetches zeros); the compiler's memory-count waits then hold
// each LDS store for its own chunk only.  (Behind the per-lane bounds branches
// it waited for every load in flight, the chunk two ahead included, before
// each store and again before each iteration's loads.)  Columns past M or N
// read whatever lies there instead of zeros: they only reach output rows and
// columns that are never stored or counted.  The host takes this form when
// every operand's byte offsets stay below 2^31.
template <int KS, int BK, bool BUF = false>
__global__ void __launch_bounds__(256 * KS) sgemm_grouped_tn_lds64_kernel(const GroupedTNArgs ga)
{
    constexpr int T = 64, P = BK / 16;
    static_assert(BK % 16 == 0 && (KS - 1) * 4096 <= KS * 2 * BK * T, "reduction area");
    __shared__ __align__(16) float As[KS][2][BK][T];
    __shared__ __align__(16) float Bs[KS][2][BK][T];
    __shared__ double ssred[4 * KS];
    __shared__ int sclst[4][1024];   // per wave of set 0: a scatter round's (token, row) list
    const int xcd = blockIdx.x % 8, j = blockIdx.x / 8;
    const int ntiles = ga.tile0[ga.ngroups];
    if (j >= ga.tp) {
        const int w = xcd * ga.cp + (j - ga.tp);
        double sq = 0.0;
        for (int q = 0; q < ga.cs_per_wg; ++q) {
            const int cid = w * ga.cs_per_wg + q;
            if (cid >= ga.cs_blocks) break;   // uniform
            const int job = cid / ga.cs_cb, cb = cid - job * ga.cs_cb;
            const float4 t = colsum4_block<256 * KS>(ga.cs.partial[job], ga.cs.nparts[job], ga.cs.out[job],
                                                     ga.cs.cols, 32 * cb, ga.cs.acc,
                                                     reinterpret_cast<float4 (*)[8]>(&As[0][0][0][0]));
            sq += static_cast<double>(t.x) * t.x + static_cast<double>(t.y) * t.y +
                  static_cast<double>(t.z) * t.z + static_cast<double>(t.w) * t.w;
            __syncthreads();   // red is reused by the next block
        }
        if (ga.ss_out) block_sumsq_out<4 * KS>(sq, ga.ss_out, ssred);
        return;
    }
    const int id = xcd * ga.tp + j;
    if (id >= ntiles) {   // padding
        if (ga.ss_out && threadIdx.x == 0) ga.ss_out[blockIdx.x] = 0.0;
        return;
    }
    int gi = 0;
    for (int i = 1; i < ga.ngroups; ++i)
        if (id >= ga.tile0[i]) gi = i;
    const GroupedTN& e = ga.e[gi];
    const int local = id - ga.tile0[gi];
    const int tm = local / ga.tiles_n[gi], tn = local - tm * ga.tiles_n[gi];
    const int K = ga.K;
    const int tid = threadIdx.x, lane = tid & 63, lr = lane & 31, lk = lane >> 5;
    const int grp = __builtin_amdgcn_readfirstlane(tid >> 8), gt = tid & 255;
    const int wave = __builtin_amdgcn_readfirstlane((tid >> 6) & 3);
    const int wm = 32 * (wave & 1), wn = 32 * (wave >> 1);
    const int m0 = tm * T, n0 = tn * T;
    // chunk loader of a set: thread t covers chunk rows t/16 + 16p (p < 4), float4 column (t%16)*4
    const int lrow = gt >> 4, lc4 = (gt & 15) * 4;
    const bool am_ok = m0 + lc4 < e.M, bn_ok = n0 + lc4 < e.N;   // M, N % 4 == 0 (host check)
    // two register sets: a set's next-but-one chunk is in flight while the
    // current chunk's MFMAs run and the next chunk goes to LDS
    float4 ra0[P], rb0[P], ra1[P], rb1[P];
    typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
    // buffer records: (K - 1) full rows plus the last row's M (N) columns
    const __amdgpu_buffer_rsrc_t rsa = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<float*>(e.A), 0, BUF ? ((K - 1) * e.lda + e.M) * 4 : 0, 0x00020000);
    const __amdgpu_buffer_rsrc_t rsb = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<float*>(e.B), 0, BUF ? ((K - 1) * e.ldb + e.N) * 4 : 0, 0x00020000);
    auto gload = [&](int k0, float4 (&ra)[P], float4 (&rb)[P]) {
        if constexpr (BUF) {
#pragma unroll
            for (int p = 0; p < P; ++p) {
                const int k = k0 + lrow + 16 * p;
                ra[p] = __builtin_bit_cast(float4, __builtin_amdgcn_raw_buffer_load_b128(
                                                       rsa, (k * e.lda + m0 + lc4) * 4, 0, 0));
                rb[p] = __builtin_bit_cast(float4, __builtin_amdgcn_raw_buffer_load_b128(
                                                       rsb, (k * e.ldb + n0 + lc4) * 4, 0, 0));
            }
            return;
        }
#pragma unroll
        for (int p = 0; p < P; ++p) {
            const int k = k0 + lrow + 16 * p;
            const bool kin = k < K;
            ra[p] = (kin && am_ok) ? *reinterpret_cast<const float4*>(e.A + static_cast<long long>(k) * e.lda + m0 + lc4)
                                   : make_float4(0.f, 0.f, 0.f, 0.f);
            rb[p] = (kin && bn_ok) ? *reinterpret_cast<const float4*>(e.B + static_cast<long long>(k) * e.ldb + n0 + lc4)
                                   : make_float4(0.f, 0.f, 0.f, 0.f);
        }
    };
    auto lstore = [&](int buf, const float4 (&ra)[P], const float4 (&rb)[P]) {
#pragma unroll
        for (int p = 0; p < P; ++p) {
            *reinterpret_cast<float4*>(&As[grp][buf][lrow + 16 * p][lc4]) = ra[p];
            *reinterpret_cast<float4*>(&Bs[grp][buf][lrow + 16 * p][lc4]) = rb[p];
        }
    };
    floatx16 acc;
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[r] = 0.f;
    // Scatter C[id_i] += scale * rows[i] over the tokens i whose id falls in
    // this wave's 32 rows, in token order.  A round lists the matches among 512
    // tokens in LDS (slot = rank in token order).  The first SC matches of the
    // first round are fetched before the products start, so their loads
    // overlap the chunk loads, and added after the products; any others are
    // fetched after the products, eight at a time.
    constexpr int SC = 24;
    const bool scat = ga.do_sc && e.sc_n > 0 && grp == 0;
    const int ocol = n0 + wn + lr;
    const int rlo = m0 + wm;
    int* lst = &sclst[wave][0];
    int idpre[8];
    if (scat) {
        // unconditional loads (clamped index) keep the memory-count waits of
        // the chunk loads exact
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            const int i = 64 * u + lane;
            const int v = e.sc_ids[min(i, e.sc_n - 1)];
            idpre[u] = i < e.sc_n ? v : -1;
        }
    }
    auto build_list = [&](int base) -> int {   // wave-uniform match count
        int total = 0;
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            const int i = base + 64 * u + lane;
            const int idv = base == 0 ? idpre[u] : (i < e.sc_n ? e.sc_ids[i] : -1);
            const int rel = idv - rlo;
            const bool hit = i < e.sc_n && rel >= 0 && rel < 32 && idv < e.M;
            const unsigned long long mask = __ballot(hit);
            if (hit) {
                const int slot = total + __popcll(mask & ((1ull << lane) - 1ull));
                lst[2 * slot] = i;
                lst[2 * slot + 1] = rel;
            }
            total += __popcll(mask);
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        return total;
    };
    const float scl = e.sc_scale;
    const int nk = (K + BK - 1) / BK;
    const int iters = (nk + KS - 1) / KS;   // every set passes the same barriers
    gload(grp * BK, ra0, rb0);
    if (BUF || iters > 1) gload((grp + KS) * BK, ra1, rb1);
    float sv[SC];             // rows of the first SC matches, fetched during the products
    unsigned srel[SC / 4];    // their rows within the wave's 32, 8 bits each (0xff: none)
    int first_total = 0;
    if (scat) {
        first_total = build_list(0);
        const int ccol = min(ocol, e.N - 1);
        int2 ent[SC];   // (token, row) pairs, read unconditionally so the reads batch
#pragma unroll
        for (int c = 0; c < SC; ++c) ent[c] = reinterpret_cast<const int2*>(lst)[c];
#pragma unroll
        for (int c = 0; c < SC; ++c) {
            const int tok = c < first_total ? ent[c].x : 0;   // row 0 stands in (its value is not used)
            sv[c] = e.sc_rows[static_cast<long long>(tok) * e.sc_ld + ccol];
        }
#pragma unroll
        for (int q = 0; q < SC / 4; ++q) {
            unsigned w = 0;
#pragma unroll
            for (int b = 0; b < 4; ++b) {
                const int c = 4 * q + b;
                w |= static_cast<unsigned>(c < first_total ? ent[c].y : 0xff) << (8 * b);
            }
            srel[q] = w;
        }
        __builtin_amdgcn_wave_barrier();   // the list is rewritten after the products
    }
    lstore(0, ra0, rb0);
    __syncthreads();
    auto chunk_mfma = [&](int buf, int kt) {
        if (kt < nk) {
#pragma unroll
            for (int st = 0; st < BK / 2; ++st) {
                const int kr = 2 * st + lk;   // lanes 0-31 read row k, 32-63 row k+1
                acc = __builtin_amdgcn_mfma_f32_32x32x2f32(As[grp][buf][kr][wm + lr], Bs[grp][buf][kr][wn + lr], acc,
                                                           0, 0, 0);
            }
        }
    };
    // iteration it computes the set's chunk it*KS + grp from LDS buffer it%2,
    // stores chunk it+1 (loaded an iteration earlier) into the other buffer
    // and issues the loads of chunk it+2
    for (int it = 0; it < iters; it += 2) {
        if (BUF || it + 2 < iters) gload(((it + 2) * KS + grp) * BK, ra0, rb0);
        chunk_mfma(0, it * KS + grp);
        if (it + 1 < iters) lstore(1, ra1, rb1);
        __syncthreads();
        if (!BUF && it + 1 >= iters) break;   // BUF: the second half's MFMAs skip themselves
        if (BUF || it + 3 < iters) gload(((it + 3) * KS + grp) * BK, ra1, rb1);
        chunk_mfma(1, (it + 1) * KS + grp);
        if (it + 2 < iters) lstore(0, ra0, rb0);
        __syncthreads();
    }
    if (KS > 1) {   // sets 1..KS-1's partial quadrants added to set 0's, in set order
        float* red = &As[0][0][0][0];
        if (grp > 0) {
#pragma unroll
            for (int r = 0; r < 16; ++r) red[((grp - 1) * 64 + wave * 16 + r) * 64 + lane] = acc[r];
        }
        __syncthreads();
        if (grp == 0) {
#pragma unroll
            for (int t = 0; t < KS - 1; ++t)
#pragma unroll
                for (int r = 0; r < 16; ++r) acc[r] += red[(t * 64 + wave * 16 + r) * 64 + lane];
        }
    }
    if (scat) {
        // register r of lane l holds C(8(r/4) + 4(l/32) + r%4, l%32) of the
        // wave's quadrant: listed row rel (wave-uniform) lands in register
        // 4(rel/8) + rel%4 of the lanes with l/32 == (rel/4)%2
        auto add_row = [&](int rel, float v) {
            const int rr = ((rel >> 3) << 2) | (rel & 3);
            const float a = v * scl;
            acc[rr] += lk == ((rel >> 2) & 1) ? a : 0.f;   // uniform index: one relative move
        };
#pragma unroll
        for (int q = 0; q < SC / 4; ++q) {
            const unsigned w = __builtin_amdgcn_readfirstlane(srel[q]);
#pragma unroll
            for (int b = 0; b < 4; ++b)
                if (4 * q + b < first_total) add_row((w >> (8 * b)) & 0xff, sv[4 * q + b]);
        }
        if (e.sc_n > 512 || first_total > SC) {
            for (int base = 0; base < e.sc_n; base += 512) {
                const int total = build_list(base);
                for (int c0 = base == 0 ? SC : 0; c0 < total; c0 += 8) {
                    float v[8];
#pragma unroll
                    for (int c = 0; c < 8; ++c) {
                        const int tok = lst[2 * (c0 + c)];
                        v[c] = c0 + c < total && ocol < e.N ? e.sc_rows[static_cast<long long>(tok) * e.sc_ld + ocol]
                                                           : 0.f;
                    }
#pragma unroll
                    for (int c = 0; c < 8; ++c)
                        if (c0 + c < total) add_row(__builtin_amdgcn_readfirstlane(lst[2 * (c0 + c) + 1]), v[c]);
                }
                __builtin_amdgcn_wave_barrier();   // the list is rewritten by the next round
            }
        }
    }
    double sq = 0.0;
    if (grp == 0 && ocol < e.N) {
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const int orow = m0 + wm + 8 * (r >> 2) + 4 * lk + (r & 3);
            if (orow < e.M) {
                __builtin_nontemporal_store(acc[r], &e.C[static_cast<long long>(orow) * e.ldc + ocol]);
                sq += static_cast<double>(acc[r]) * acc[r];
            }
        }
    }
    if (ga.ss_out) block_sumsq_out<4 * KS>(sq, ga.ss_out, ssred);
}

}  // namespace

int sgemm_grouped_tn(const GroupedTN* g, int ngroups, int K, hipStream_t stream, const ColsumSet* cs,
                     GroupedExtras* ex)
{
    if (ex) {
        ex->fused = 0;
        ex->ss_parts = 0;
    }
    if (ngroups <= 0) {
        if (cs && cs->njobs > 0)
            return rmsnorm_bwd_colsum_multi(cs->partial, cs->nparts, cs->out, cs->njobs, cs->cols, cs->acc, stream);
        return LHIP_OK;
    }
    if (ngroups > kGroupedMax) return fail(LHIP_E_ARG, "sgemm_grouped_tn: %d groups (at most %d)", ngroups, kGroupedMax);
    if (K <= 0) return fail(LHIP_E_SHAPE, "sgemm_grouped_tn: K=%d", K);
    GroupedTNArgs ga{};
    bool vec = true;
    long long tiles64 = 0;
    for (int i = 0; i < ngroups; ++i) {
        const GroupedTN& e = g[i];
        if (e.M <= 0 || e.N <= 0) return fail(LHIP_E_SHAPE, "sgemm_grouped_tn: group %d is %dx%d", i, e.M, e.N);
        if (!e.A || !e.B || !e.C) return fail(LHIP_E_NULL, "sgemm_grouped_tn: group %d has a NULL operand", i);
        if (e.lda < e.M || e.ldb < e.N || e.ldc < e.N)
            return fail(LHIP_E_SHAPE, "sgemm_grouped_tn: group %d leading dimensions", i);
        vec = vec && e.lda % 4 == 0 && e.ldb % 4 == 0 && e.M % 4 == 0 && e.N % 4 == 0 && aligned16(e.A) &&
              aligned16(e.B);
        tiles64 += static_cast<long long>(ceil_div(e.M, 64)) * ceil_div(e.N, 64);
    }
    // 64x64 tiles once they give a quarter of the CUs work and fit one
    // workgroup per CU, or where K is so short that running the scatter and the
    // squared norm in the same launch is worth more than the finer tiles
    // (256x64x2 step, 128 rows: 106 -> 100 us; but 500x64x2, 2048 rows: 178 on
    // 32x32, 211 on these); 32x32 otherwise
    const int cus = st().cu_count > 0 ? st().cu_count : 256;
    const bool wide = vec && tiles64 <= cus && (4 * tiles64 >= cus || K <= 256);
    // More than one 64x64 tile per CU, or operands that take no float4 loads:
    // the three-term kernel (29 products of a 4000x512x4 model over 2048
    // tokens: 674 us on the 32x32 tiles, 316 us on this)
    bool x3 = tiles64 > cus || (!vec && 4 * tiles64 >= cus);
    for (int i = 0; i < ngroups; ++i)
        x3 = x3 && std::max({g[i].lda, g[i].ldb, 8 * g[i].ldc}) < 1 << 25;
    if (x3) {
        if (int rc = launch_x3_grouped_tn(g, ngroups, K, stream)) return rc;
        if (!cs || cs->njobs <= 0) return LHIP_OK;
        return rmsnorm_bwd_colsum_multi(cs->partial, cs->nparts, cs->out, cs->njobs, cs->cols, cs->acc, stream);
    }
    const int tile = wide ? 64 : kGroupedTile;
    long long tiles = 0;
    for (int i = 0; i < ngroups; ++i) {
        const GroupedTN& e = g[i];
        ga.e[i] = e;
        ga.tile0[i] = static_cast<int>(tiles);
        ga.tiles_n[i] = ceil_div(e.N, tile);
        tiles += static_cast<long long>(ceil_div(e.M, tile)) * ga.tiles_n[i];
        if (tiles > 0x7fffffffLL) return fail(LHIP_E_CAPACITY, "sgemm_grouped_tn: too many tiles");
    }
    ga.tile0[ngroups] = static_cast<int>(tiles);
    ga.ngroups = ngroups;
    ga.K = K;
    // column sums in the same launch when they take the float4 form too
    bool cs_fused = false;
    if (vec && cs && cs->njobs > 0) {
        if (cs->njobs > kColsumJobs) return fail(LHIP_E_ARG, "sgemm_grouped_tn: %d column-sum jobs", cs->njobs);
        cs_fused = cs->cols > 0 && cs->cols % 4 == 0;
        for (int i = 0; i < cs->njobs && cs_fused; ++i)
            cs_fused = cs->nparts[i] > 0 && cs->partial[i] && cs->out[i] && aligned16(cs->partial[i]) &&
                       aligned16(cs->out[i]);
        if (cs_fused) {
            ga.cs = *cs;
            ga.cs_cb = ceil_div(cs->cols, 32);
            ga.cs_blocks = cs->njobs * ga.cs_cb;
        }
    }
    unsigned grid = static_cast<unsigned>((tiles + ga.cs_blocks + 7) / 8 * 8);   // whole XCD rounds
    if (wide) {
        // per XCD: its tiles, then column-sum workgroups on the CUs left over
        ga.tp = static_cast<int>((tiles + 7) / 8);
        ga.cp = 0;
        ga.cs_per_wg = 1;
        if (ga.cs_blocks > 0) {
            ga.cp = std::max(1, cus / 8 - ga.tp);
            ga.cp = std::min(ga.cp, (ga.cs_blocks + 7) / 8);
            ga.cs_per_wg = (ga.cs_blocks + 8 * ga.cp - 1) / (8 * ga.cp);
        }
        grid = static_cast<unsigned>(8 * (ga.tp + ga.cp));
        // the scatters and the per-workgroup sums of squares, when the column
        // sums run here too (every stored value then passes through this launch)
        if (ex && ex->ss_out && static_cast<int>(grid) <= ex->ss_cap && (!cs || cs->njobs == 0 || cs_fused)) {
            for (int i = 0; i < ngroups; ++i)
                if (g[i].sc_n > 0 && (!g[i].sc_ids || !g[i].sc_rows || g[i].sc_ld < g[i].N))
                    return fail(LHIP_E_ARG, "sgemm_grouped_tn: group %d scatter arguments", i);
            ga.do_sc = 1;
            ga.ss_out = ex->ss_out;
            ex->fused = 1;
            ex->ss_parts = static_cast<int>(grid);
        }
        // buffer loads when every byte offset a chunk load can form (rows up
        // to K plus the loads past the last chunk) stays below 2^31
        bool buf = true;
        for (int i = 0; i < ngroups; ++i) {
            const long long rows = static_cast<long long>(K) + 512;
            buf = buf && (rows * g[i].lda + 64) * 4 < (1LL << 31) && (rows * g[i].ldb + 64) * 4 < (1LL << 31);
        }
        if (K >= 512) {
            if (buf) klaunch(sgemm_grouped_tn_lds64_kernel<4, 32, true>, grid, 1024, 0, stream, ga);
            else klaunch(sgemm_grouped_tn_lds64_kernel<4, 32>, grid, 1024, 0, stream, ga);
        } else if (buf) {
            klaunch(sgemm_grouped_tn_lds64_kernel<2, kGroupedBK, true>, grid, 512, 0, stream, ga);
        } else {
            klaunch(sgemm_grouped_tn_lds64_kernel<2, kGroupedBK>, grid, 512, 0, stream, ga);
        }
    }
    else if (vec) klaunch(sgemm_grouped_tn_lds_kernel, grid, 256, 0, stream, ga);
    else if (K >= 256) klaunch(sgemm_grouped_tn_kernel<8>, grid, 512, 0, stream, ga);
    else klaunch(sgemm_grouped_tn_kernel<4>, grid, 256, 0, stream, ga);
    int rc = check_launch("sgemm_grouped_tn");
    if (rc != LHIP_OK || cs_fused || !cs || cs->njobs <= 0) return rc;
    return rmsnorm_bwd_colsum_multi(cs->partial, cs->nparts, cs->out, cs->njobs, cs->cols, cs->acc, stream);
}

// 16x16 tiles whose consumer sums the slices itself (no reduce launch): one
// software pass per slice, slices a multiple of 64 deep.
int tiny_unreduced_plan(int m, int n, int k, size_t ws_floats, int* kchunk_out)
{
    constexpr int pass = 64 * kSmallU;
    if (k <= pass) return 1;
    long long s = std::min<long long>(ceil_div(k, pass), 64);
    s = std::min<long long>(s, static_cast<long long>(ws_floats / (static_cast<size_t>(m) * n)));
    if (s < 2) return 1;
    const int kchunk = ceil_div(ceil_div(k, static_cast<int>(s)), 64) * 64;
    *kchunk_out = kchunk;
    return ceil_div(k, kchunk);
}

// Products with few 32x32 tiles that stay on 16x16 tiles: four times the
// workgroups, and up to K = 512 one round trip of loads.  Up to two tiles per CU
// with K up to 256, or 512 for the first quarter past one (512x640x256 NN 6.0 us
// against 8.5, 512x512x512 8.5 against 12.1, 521x665x186 TN 6.8 against 9.3, but
// unaligned NT 8.9 against 7.2; 800x800x130, 2.4 tiles per CU, 8.9 against 7.5).
// With fewer tiles than CUs K up to 1024; up to 2048 when both operands take
// float4 loads (256x256x1536 NT 11.1 us against 12.1 on the three-term kernel, 512x128x2000 10.2 against 11.6;
// unaligned 238x474x1199 28.4 against 12.4); up to 4096 where B is read along
// its rows and the product is one column tile wide, or A is K-major
// (4096x16x4096 NN 21.2 against 25.0, TN 23.2 against 31.0; 128x128x4096 TN
// 10.8 against 12.8; but 16x4096x4096 NT 38.4 against 23.8).
bool tiny_best(int ta, int tb, int m, int n, int k, int batch, int vecA, int vecB)
{
    const int cus = st().cu_count > 0 ? st().cu_count : 256;
    const long long tiles32 = static_cast<long long>(ceil_div(m, 32)) * ceil_div(n, 32) * batch;
    if (tiles32 >= cus)
        return tiles32 < 2 * cus && ((k <= 256 && (!tb || (vecA && vecB))) || (!tb && k <= 512 && 4 * tiles32 <= 5 * cus));
    if (k <= 1024 || (k <= 2048 && vecA && vecB)) return true;
    return k <= 4096 && !tb && ((ta && vecA && vecB) || (n <= 16 && vecA));
}

// Up to 16 rows of C the product is one streaming pass over B; from 17 to 32
// rows that form is level with the three-term kernel on a large aligned B
// (32x4096x1024 13.0 us against 13.8, 32x4096x4096 27.8 against 26.8) and
// behind it elsewhere (32x2000x512 12.2 against 10.5, 32x777x1500 15.1 against
// 11.8), and further behind with more rows (40x4096x4096 32.0 against 27.3).
bool skinny_best(int m, int n, int k, int vecB)
{
    return m <= 16 || (m <= kSkinnyMax && vecB && static_cast<long long>(n) * k >= 1LL << 22);
}

int sgemm_run(int ta, int tb, int m, int n, int k, float alpha,
              const float* A, int lda, long long sA, const float* B, int ldb, long long sB, float beta,
              float* C, int ldc, long long sC, int batch, const GemmOpts& o, hipStream_t stream)
{
    if (m < 0 || n < 0 || k < 0 || batch < 0)
        return fail(LHIP_E_SHAPE, "sgemm: negative size (m=%d n=%d k=%d batch=%d)", m, n, k, batch);
    if (m == 0 || n == 0 || batch == 0) return LHIP_OK;
    if (!C) return fail(LHIP_E_NULL, "sgemm: C is NULL");
    if (k > 0 && (!A || !B)) return fail(LHIP_E_NULL, "sgemm: A or B is NULL");
    const int a_cols = ta ? m : k;   // stored column count of A
    const int b_cols = tb ? k : n;
    if (k > 0 && lda < (a_cols > 0 ? a_cols : 1))
        return fail(LHIP_E_SHAPE, "sgemm: lda=%d < %d", lda, a_cols);
    if (k > 0 && ldb < (b_cols > 0 ? b_cols : 1))
        return fail(LHIP_E_SHAPE, "sgemm: ldb=%d < %d", ldb, b_cols);
    if (ldc < n) return fail(LHIP_E_SHAPE, "sgemm: ldc=%d < n=%d", ldc, n);
    if (o.R && o.ldr < n) return fail(LHIP_E_SHAPE, "sgemm: ldr=%d < n=%d", o.ldr, n);
    if (batch > 65535) return fail(LHIP_E_CAPACITY, "sgemm: batch %d > 65535", batch);
    if (batch > 1 && (sA < 0 || sB < 0 || sC < 0 || o.sA2 < 0 || o.sB2 < 0 || o.sC2 < 0))
        return fail(LHIP_E_SHAPE, "sgemm: negative batch stride");
    if (o.inner <= 0) return fail(LHIP_E_ARG, "sgemm: inner batch count must be > 0");
    if (o.kblocks <= 0) return fail(LHIP_E_ARG, "sgemm: kblocks must be > 0");
    const long long k_all = static_cast<long long>(k) * o.kblocks;
    if (o.kblocks > 1 && k > 0) {
        // One launch where a kernel walks the blocks itself: the three-term
        // kernel (blocks of whole 16-deep stages), or the 16x16-tile one (A not
        // transposed, blocks of whole quads).  Otherwise the blocks are
        // accumulated by successive launches.
        X3Plan p{};
        const bool one = k_all <= 0x7fffffffLL &&
                         (x3_plan(ta, tb, m, n, static_cast<int>(k_all), k, lda, ldb, std::max(ldc, o.ldr), batch, 0, false, &p) ||
                          (!ta && k % 4 == 0 &&
                           tiny_best(ta, tb, m, n, static_cast<int>(k_all), batch, true, true)));
        if (!one) {
            GemmOpts oj = o;
            oj.kblocks = 1;
            for (int j = 0; j < o.kblocks; ++j) {
                if (j == 1) { oj.R = nullptr; oj.ldr = 0; }
                const int rc = sgemm_run(ta, tb, m, n, k, alpha, A + j * o.sAk, lda, sA, B + j * o.sBk, ldb, sB,
                                         j == 0 ? beta : 1.f, C, ldc, sC, batch, oj, stream);
                if (rc != LHIP_OK) return rc;
            }
            return LHIP_OK;
        }
    }
    const bool br = o.kblocks > 1 && k > 0;
    GemmArgs g{};

    g.M = m; g.N = n; g.K = static_cast<int>(br ? k_all : k); g.alpha = alpha; g.beta = beta;
    g.Kb = k; g.sAk = br ? o.sAk : 0; g.sBk = br ? o.sBk : 0;
    g.A = A; g.lda = lda; g.sA = sA; g.sA2 = o.sA2;
    g.B = B; g.ldb = ldb; g.sB = sB; g.sB2 = o.sB2;
    g.C = C; g.ldc = ldc; g.sC = sC; g.sC2 = o.sC2;
    g.R = o.R; g.ldr = o.ldr;
    g.inner = o.inner;
    g.vecA = (k > 0 && lda % 4 == 0 && aligned16(A) && (batch == 1 || (sA % 4 == 0 && o.sA2 % 4 == 0)) &&
              g.sAk % 4 == 0) ? 1 : 0;
    g.vecB = (k > 0 && ldb % 4 == 0 && aligned16(B) && (batch == 1 || (sB % 4 == 0 && o.sB2 % 4 == 0)) &&
              g.sBk % 4 == 0) ? 1 : 0;
    if (k == 0) {
        // C = beta * C through the 16x16-tile kernel
        if (o.splits_out) *o.splits_out = 1;
        g.splits = 1;
        return launch_tiny(ta, tb, g, batch, stream);
    }
    if (!br && !o.splits_out && skinny_ok(ta, tb, m, n, batch, 1) && skinny_best(m, n, k, g.vecB)) {
        g.ws = o.ws;
        g.ws_floats_avail = o.ws ? o.ws_floats : 0;
        return launch_skinny(ta, g, stream);
    }
    if (o.splits_out && (alpha != 1.f || beta != 0.f || batch != 1 || o.R))
        return fail(LHIP_E_ARG, "sgemm: unreduced split-K needs alpha 1, beta 0, batch 1");
    // (the 16x16-tile kernel walks the blocks of a batch-reduce for a plain A only)
    X3Plan x3{};
    // An unreduced split of a small product: one-pass slices on 16x16 tiles, at
    // any K they cover.
    const int cus = st().cu_count > 0 ? st().cu_count : 256;
    const bool tiny_slices = o.splits_out && o.ws && k <= 64 * 64 * kSmallU &&
                             static_cast<long long>(ceil_div(m, 32)) * ceil_div(n, 32) < cus && (m <= 64 || n <= 64);
    if (tiny_slices || (!(br && (ta || k % 4 != 0)) && tiny_best(ta, tb, m, n, g.K, batch, g.vecA, g.vecB)) ||
        !(o.plan ? (x3 = *o.plan, true) : x3_plan(ta, tb, m, n, g.K, br ? k : 0, lda, ldb, std::max(ldc, o.ldr), batch,
                 o.ws ? std::min(o.ws_floats, kX3WsFloats) : 0, !o.splits_out, &x3))) {
        g.splits = o.ws && o.splits_out ? tiny_unreduced_plan(m, n, g.K, o.ws_floats, &g.kchunk) : 1;
        g.ws = o.ws;
        if (o.splits_out) {
            *o.splits_out = g.splits > 1 ? g.splits : 1;
            g.skip_reduce = g.splits > 1 ? 1 : 0;
        }
        return launch_tiny(ta, tb, g, batch, stream);
    }
    if (!br && ks_best(ta, tb, m, n, k, batch, g.vecA, g.vecB)) {
        if (o.splits_out) *o.splits_out = 1;
        return launch_ks(ta, tb, g, batch, stream);
    }
    g.splits = x3.splits;
    g.kchunk = x3.kchunk;
    g.tail = x3.tail;
    g.ws = o.ws;
    if (o.splits_out) {
        *o.splits_out = x3.splits;
        g.skip_reduce = x3.splits > 1 ? 1 : 0;
    }
    return launch_x3(x3.tile, br, ta, tb, g, batch, stream);
}

int sgemm_launch(int ta, int tb, int m, int n, int k, float alpha,
                 const float* A, int lda, const float* B, int ldb, float beta,
                 float* C, int ldc, int batch, long long sA, long long sB, long long sC,
                 hipStream_t stream)
{
    GemmOpts o;
    o.inner = batch > 0 ? batch : 1;
    return sgemm_run(ta, tb, m, n, k, alpha, A, lda, sA, B, ldb, sB, beta, C, ldc, sC, batch, o, stream);
}

// Fixed split-K scratch of lhip_sgemm_noalloc (the array itself is below, at file scope).
constexpr size_t kNoallocScratchBytes = kX3WsFloats * sizeof(float);   // 64 MiB
constexpr int kNoallocMaxDevices = 64;

}  // namespace lhip

// ---- scratch of the allocation-free entry point (lhip_sgemm_noalloc) ----------
// Split-K partials of lhip_sgemm_noalloc live in this file-scope device array
// instead of the library workspace, so that call never allocates.  Each GPU
// holds its own copy for the life of the process.  Host code never uses the
// array's name as an address (on the host it is only a stand-in for the
// symbol): lhip_init resolves its device address once per device with
// hipGetSymbolAddress (noalloc_scratch_init) and every launch takes that
// pointer.  The partials of a split are fully written before the reduce reads
// them, so nothing in the array needs to start at zero.
static __device__ __align__(256) float scratch[lhip::kNoallocScratchBytes / sizeof(float)];

namespace lhip {

static float* g_scratch_dev[kNoallocMaxDevices] = {};

int noalloc_scratch_init(int device)
{
    if (device < 0 || device >= kNoallocMaxDevices)
        return fail(LHIP_E_CAPACITY, "lhip_init: device %d beyond the %d devices the scratch table holds", device,
                    kNoallocMaxDevices);
    if (g_scratch_dev[device]) return LHIP_OK;
    void* p = nullptr;
    const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !p) {
        (void)hipGetLastError();
        return fail(LHIP_E_DEVICE, "lhip_init: hipGetSymbolAddress(scratch) on device %d: %s", device,
                    e != hipSuccess ? hipGetErrorString(e) : "null address");
    }
    g_scratch_dev[device] = static_cast<float*>(p);
    return LHIP_OK;
}

size_t immediate_ws(int transa, int transb, int m, int n, int k, int batch, int lda, int ldb, int ldc, size_t head,
                    X3Plan* plan, bool* planned)
{
    if (planned) *planned = false;
    if (m <= 0 || n <= 0 || k <= 0 || batch <= 0) return 0;
    const bool skinny = skinny_ok(transa, transb, m, n, batch, 1);
    // the smallest products, whose host time counts: 16x16 tiles, never split
    if (k <= 1024 && m > 64 && tiny_best(transa, transb, m, n, k, batch, 0, 0) &&
        static_cast<long long>((m + 31) / 32) * ((n + 31) / 32) * batch < (st().cu_count > 0 ? st().cu_count : 256))
        return 0;
    const size_t doc = documented_partials(transa, transb, m, n, k, batch);
    size_t need = 0;
    X3Plan p{};
    if (skinny) {
        int kchunk = 0;
        const int s = skinny_plan(m, n, k, static_cast<size_t>(1) << 26, &kchunk);
        if (s > 1) need = static_cast<size_t>(s) * m * n;
    }
    bool ok = false;
    if (!(skinny && m <= 16) && !tiny_best(transa, transb, m, n, k, batch, 0, 0)) {
        ok = x3_plan(transa, transb, m, n, k, 0, lda, ldb, ldc, batch, kX3WsFloats, true, &p);
        if (ok) need = std::max(need, p.ws_floats);
    }
    // A recording cannot grow the workspace: products that never needed any
    // are recorded with what is held (unsplit if need be).
    if (st().recording && (head + std::max(doc, need)) * sizeof(float) > st().work_bytes) return doc;
    if (ok && plan) {
        *plan = p;
        *planned = true;
    }
    return std::max(doc, need);
}

}  // namespace lhip

using lhip::fail;
using lhip::st;

extern "C" {

// Immediate calls: split-K partials live in the library workspace (sized here,
// before any launch).
static int sgemm_immediate(int transa, int transb, int m, int n, int k, float alpha, const float* A, int lda,
                           long long sA, const float* B, int ldb, long long sB, float beta, float* C, int ldc,
                           long long sC, int batch)
{
    lhip::GemmOpts o;
    o.inner = batch > 0 ? batch : 1;
    lhip::X3Plan plan;
    bool planned = false;
    o.ws_floats = lhip::immediate_ws(transa, transb, m, n, k, batch, lda, ldb, ldc, 0, &plan, &planned);
    if (planned) o.plan = &plan;
    if (o.ws_floats > 0) {
        int rc = lhip::workspace(o.ws_floats * sizeof(float), reinterpret_cast<void**>(&o.ws));
        if (rc != LHIP_OK) return rc;
    }
    return lhip::sgemm_run(transa, transb, m, n, k, alpha, A, lda, sA, B, ldb, sB, beta, C, ldc, sC, batch, o,
                           st().stream);
}

LHIP_API int lhip_sgemm_noalloc(int transa, int transb, int m, int n, int k, float alpha,
                                const float* A, int lda, const float* B, int ldb, float beta,
                                float* C, int ldc)
{
    LHIP_REQUIRE_READY();
    float* const ptr = lhip::g_scratch_dev[st().device];
    if (!ptr) return fail(LHIP_E_DEVICE, "lhip_sgemm_noalloc: scratch of device %d not resolved", st().device);
    lhip::GemmOpts o;
    const size_t need = m > 0 && n > 0 && k > 0 ? lhip::documented_partials(transa, transb, m, n, k, 1) : 0;
    if (need * sizeof(float) > lhip::kNoallocScratchBytes)
        return fail(LHIP_E_CAPACITY,
                    "lhip_sgemm_noalloc: m=%d n=%d k=%d needs %zu bytes of split-K scratch, beyond its fixed "
                    "%zu bytes; use lhip_sgemm", m, n, k, need * sizeof(float), lhip::kNoallocScratchBytes);
    o.ws = ptr;
    o.ws_floats = lhip::kX3WsFloats;
    return lhip::sgemm_run(transa, transb, m, n, k, alpha, A, lda, 0, B, ldb, 0, beta, C, ldc, 0, 1, o,
                           st().stream);
}

LHIP_API int lhip_sgemm(int transa, int transb, int m, int n, int k, float alpha,
                        const float* A, int lda, const float* B, int ldb, float beta,
                        float* C, int ldc)
{
    LHIP_REQUIRE_READY();
    return sgemm_immediate(transa, transb, m, n, k, alpha, A, lda, 0, B, ldb, 0, beta, C, ldc, 0, 1);
}

LHIP_API int lhip_sgemm_strided_batched(int transa, int transb, int m, int n, int k, float alpha,
                                        const float* A, int lda, long long strideA,
                                        const float* B, int ldb, long long strideB, float beta,
                                        float* C, int ldc, long long strideC, int batch)
{
    LHIP_REQUIRE_READY();
    return sgemm_immediate(transa, transb, m, n, k, alpha, A, lda, strideA, B, ldb, strideB, beta, C, ldc, strideC,
                           batch);
}

LHIP_API int lhip_sgemm_batched_reduce(int transa, int transb, int m, int n, int k, float alpha,
                                       const float* A, int lda, long long strideA,
                                       const float* B, int ldb, long long strideB, float beta,
                                       float* C, int ldc, int count)
{
    LHIP_REQUIRE_READY();
    if (count <= 0) return fail(LHIP_E_ARG, "lhip_sgemm_batched_reduce: count %d must be >= 1", count);
    if (count > 1 && (strideA < 0 || strideB < 0))
        return fail(LHIP_E_SHAPE, "lhip_sgemm_batched_reduce: negative stride");
    lhip::GemmOpts o;
    o.kblocks = count;
    o.sAk = strideA;
    o.sBk = strideB;
    const long long kall = static_cast<long long>(k) * count;
    if (m > 0 && n > 0 && k > 0 && kall <= 0x7fffffffLL) {
        int kchunk = 0;
        const int splits = lhip::splitk_plan(m, n, static_cast<int>(kall), 1, static_cast<size_t>(1) << 26, &kchunk);
        if (splits > 1) {
            o.ws_floats = static_cast<size_t>(splits) * m * n;
            int rc = lhip::workspace(o.ws_floats * sizeof(float), reinterpret_cast<void**>(&o.ws));
            if (rc != LHIP_OK) return rc;
        }
    }
    return lhip::sgemm_run(transa, transb, m, n, k, alpha, A, lda, 0, B, ldb, 0, beta, C, ldc, 0, 1, o, st().stream);
}


}  // extern "C"
