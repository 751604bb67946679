// lhip_gemm_x3.hip -- fp32 GEMM on the bf16 matrix cores, each fp32 operand
// held exactly as the sum of three bf16 terms.
//
// A float x is h + m + l with h = bf16(x), m = bf16(x - h), l = x - h - m: the
// two differences are exact, |m| <= 2^-9 |x| and |l| <= 2^-18 |x|, and l has at
// most 8 significant bits, so nothing is dropped.  Of the nine products of two
// such sums the six largest are formed, each with one
// v_mfma_f32_32x32x16_bf16 accumulating in fp32: l.h, h.l, m.m, m.h, h.m, h.h.
// The three left out are below 2^-27 of a product, under the rounding of the
// fp32 accumulator (2^-25); and with six accumulations per 16 k instead of
// eight (v_mfma_f32_32x32x2_f32) the sum rounds less often.  Measured against
// 64-bit sums, one accumulator, normal operands (relative 2-norm, fp32 MFMA
// and this): K = 16 7.0e-8 and 3.3e-8, 128 2.0e-7 and 1.6e-7, 512 4.2e-7 and
// 3.4e-7, 4096 1.13e-6 and 1.05e-6, 8192 1.75e-6 and 1.41e-6; with the three
// smallest products added the figures do not change.
//
// What this buys: the bf16 cores run 16x the fp32 cores' rate (2.5 PFLOP/s
// against 157 TFLOP/s), so six products at fp32 precision leave a ceiling of
// 419 TFLOP/s.
//
// Values the split cannot carry -- infinities, NaN, values that round to an
// infinite bf16, and non-zero values below 2^-110, whose l would fall under
// bf16's last bit -- are found at no cost in the loop (an operand that is not
// finite leaves a non-finite accumulator; the smallest magnitude is kept while
// converting), and the workgroup then computes its tile again on the fp32
// matrix cores, so such values behave as they always did.
#include <algorithm>
#include <cmath>
#include <type_traits>

#include "lhip_gemm.h"

namespace lhip {
namespace {

typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef float floatx2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float floatx4 __attribute__((ext_vector_type(4)));

// Smallest magnitude the split carries exactly (2^-110), as the fp32 pattern
// shifted left by one (the sign out), less one (so that zero becomes the largest).
constexpr unsigned kX3Tiny = ((127u - 110u) << 24) - 1u;

__device__ __forceinline__ unsigned pack_bf16(float x, float y)
{
    const floatx2 v = {x, y};
    return __builtin_bit_cast(unsigned, __builtin_convertvector(v, bf16x2));
}

// A wave-uniform pointer in scalar registers (the tile arithmetic divides in
// vector registers, which would make every load of the loop carry its base there).
__device__ __forceinline__ const float* uniform(const float* p)
{
    const unsigned long long a = reinterpret_cast<unsigned long long>(p);
    const unsigned lo = __builtin_amdgcn_readfirstlane(static_cast<unsigned>(a));
    const unsigned hi = __builtin_amdgcn_readfirstlane(static_cast<unsigned>(a >> 32));
    return reinterpret_cast<const float*>(static_cast<unsigned long long>(hi) << 32 | lo);
}

// The three bf16 terms of two floats, packed.
__device__ __forceinline__ void split_pair(float x, float y, unsigned& h, unsigned& m, unsigned& l)
{
    h = pack_bf16(x, y);
    x -= __uint_as_float(h << 16);
    y -= __uint_as_float(h & 0xffff0000u);
    m = pack_bf16(x, y);
    x -= __uint_as_float(m << 16);
    y -= __uint_as_float(m & 0xffff0000u);
    l = pack_bf16(x, y);
}

// One operand's ROWS x 16 stage, loaded by NT threads.  The stored operand has
// element (row, k) at X[row * ld + k], or at X[k * ld + row] when KMAJOR.
//
// A unit is KW consecutive k of one row.  Row-contiguous operands load a unit
// with one 16-byte load (four lanes cover a row's 64 bytes); K-major ones load
// a dword per k (consecutive lanes on consecutive rows; with four k per unit,
// lane pairs share a row), so no alignment or width is asked of N or ld.  In LDS each term is a plane of two halves (k 0-7, 8-15)
// of ROWS x 8 bf16: an MFMA fragment is one ds_read_b128 of 32 consecutive
// 16-byte rows per half wave.  The halves are 64 bytes apart modulo
// 128, so 16 lanes of ds_write_b64 (4 rows x 2 halves of row-contiguous units)
// write 128 different bytes of banks; K-major units of eight k write whole
// 16-byte rows.
template <int ROWS, int NT, bool KMAJOR>
struct X3Stage {
    static constexpr int KW = (KMAJOR && ROWS * 2 >= NT) ? 8 : 4;
    static constexpr int U = ROWS * kX3K / KW / NT;
    static constexpr int HALF = ROWS * 16 + 64;
    static constexpr int PLANE = 2 * HALF;
    static constexpr int BYTES = 3 * PLANE;
    static_assert(U >= 1 && U * KW * NT == ROWS * kX3K, "stage/thread mismatch");
    float v[U][KW];
    unsigned off[U];   // byte offset of the unit from the stage's base

    static __device__ __forceinline__ int row_of(int u, int tid)
    {
        return KMAJOR ? (KW == 8 ? (tid + u * NT) % ROWS : ((tid + u * NT) >> 1) % ROWS) : (tid + u * NT) / 4;
    }
    static __device__ __forceinline__ int k_of(int u, int tid)
    {
        return KMAJOR ? (KW == 8 ? (tid + u * NT) / ROWS * 8 : (((tid + u * NT) / (2 * ROWS)) * 2 + (tid & 1)) * 4) : ((tid + u * NT) & 3) * 4;
    }

    // Rows past `rows` are clamped into the operand: they only reach outputs
    // that are not stored.
    __device__ __forceinline__ void init(int rows, int ld, int tid)
    {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int r = min(row_of(u, tid), rows - 1), k = k_of(u, tid);
            off[u] = 4u * (KMAJOR ? static_cast<unsigned>(k) * static_cast<unsigned>(ld) + r
                                  : static_cast<unsigned>(r) * static_cast<unsigned>(ld) + k);
        }
    }

    // Buffer loads: the stage's base in scalar registers, the unit's offset in
    // one vector register, so no load costs vector address arithmetic.
    __device__ __forceinline__ void load(int u, const float* base, int ld)
    {
        const __amdgpu_buffer_rsrc_t rs =
            __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(base), 0, 0x7fffffff, 0x00020000);
        if (KMAJOR) {
#pragma unroll
            for (int e = 0; e < KW; ++e)
                v[u][e] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rs, off[u], 4 * e * ld, 0));
        } else {
            const floatx4 t = __builtin_bit_cast(floatx4, __builtin_amdgcn_raw_buffer_load_b128(rs, off[u], 0, 0));
            v[u][0] = t.x; v[u][1] = t.y; v[u][2] = t.z; v[u][3] = t.w;
        }
    }

    // The last, partial stage: k at or past kvalid read as zero.
    __device__ __forceinline__ void load_tail(int u, const float* __restrict__ base, int ld, int kvalid, int tid)
    {
        const float* p = reinterpret_cast<const float*>(reinterpret_cast<const char*>(base) + off[u]);
        const int k = k_of(u, tid);
#pragma unroll
        for (int e = 0; e < KW; ++e)
            v[u][e] = k + e < kvalid ? p[KMAJOR ? static_cast<size_t>(e) * ld : e] : 0.f;
    }

    // Split unit u and store its three terms; keeps the smallest magnitude seen.
    __device__ __forceinline__ void store(int u, char* lds, int tid, unsigned& tiny) const
    {
        const int r = row_of(u, tid), k = k_of(u, tid);
        char* dst = lds + (k >> 3) * HALF + r * 16 + (k & 7) * 2;
        unsigned t[3][KW / 2];
#pragma unroll
        for (int e = 0; e < KW / 2; ++e) {
            const float x = v[u][2 * e], y = v[u][2 * e + 1];
            split_pair(x, y, t[0][e], t[1][e], t[2][e]);
            tiny = min(tiny, min((__float_as_uint(x) << 1) - 1u, (__float_as_uint(y) << 1) - 1u));
        }
#pragma unroll
        for (int p = 0; p < 3; ++p) {
            if (KW == 8)
                *reinterpret_cast<uint4*>(dst + p * PLANE) = make_uint4(t[p][0], t[p][1], t[p][2 % (KW / 2)], t[p][3 % (KW / 2)]);
            else
                *reinterpret_cast<uint2*>(dst + p * PLANE) = make_uint2(t[p][0], t[p][1]);
        }
    }

    // Unsplit, as [k][ROWS + 1] floats (the fp32 repeat of a tile).
    __device__ __forceinline__ void store_f32(int u, float* lds, int tid) const
    {
        const int r = row_of(u, tid), k = k_of(u, tid);
#pragma unroll
        for (int e = 0; e < KW; ++e) lds[(k + e) * (ROWS + 1) + r] = v[u][e];
    }
};

// BM x BN tile per workgroup; KS wave sets of WM x WN waves, set s taking the
// stages s, s + KS, ... in LDS buffers of its own, the sets' tiles added in set
// order at the end.
template <int BM, int BN, int WM, int WN, int KS, int PF, bool BR, bool TA, bool TB>
__device__ __forceinline__ void x3_tile(const GemmArgs& g, const unsigned kb_magic, const int tm, const int tn,
                                        const int kbeg, const int kend, float* const part)
{
    constexpr int NT = 64 * WM * WN;
    constexpr int FM = BM / WM / 32, FN = BN / WN / 32;
    using SA = X3Stage<BM, NT, TA>;
    using SB = X3Stage<BN, NT, !TB>;
    constexpr int BUF = SA::BYTES + SB::BYTES;
    constexpr int F32 = kX3K * (BM + 1 + BN + 1) * 4;
    constexpr int SET = 2 * BUF > F32 ? 2 * BUF : F32;
    constexpr int RED = (KS - 1) * BM * BN * 4;
    __shared__ __align__(16) char lds_all[KS * SET > RED ? KS * SET : RED];

    const int set = KS > 1 ? __builtin_amdgcn_readfirstlane(threadIdx.x / NT) : 0;
    const int tid = KS > 1 ? threadIdx.x % NT : threadIdx.x;
    const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lr = lane & 31, h = lane >> 5;
    char* lds = lds_all + set * SET;

    const int m0 = tm * BM, n0 = tn * BN;
    const int wm = (wave / WN) * (BM / WM), wn = (wave % WN) * (BN / WN);
    const long long zo = blockIdx.y / g.inner, zi = blockIdx.y % g.inner;
    const int K = kend - kbeg;
    const float* __restrict__ A = g.A + zo * g.sA2 + zi * g.sA + (TA ? m0 : static_cast<long long>(m0) * g.lda) +
                                  (TA ? static_cast<long long>(kbeg) * g.lda : kbeg);
    const float* __restrict__ B = g.B + zo * g.sB2 + zi * g.sB + (TB ? static_cast<long long>(n0) * g.ldb : n0) +
                                  (TB ? kbeg : static_cast<long long>(kbeg) * g.ldb);

    // Stage c starts at k = 16 c of block j = c / (Kb / 16) (batch-reduce; one
    // block otherwise, kb_magic 0); j by a multiplication with
    // ceil(2^32 / (Kb / 16)).
    const int kb_stages = g.Kb / kX3K;
    auto a_base = [&](int c) {
        const int j = kb_magic ? static_cast<int>(__umulhi(static_cast<unsigned>(c), kb_magic)) : 0;
        const long long k = static_cast<long long>(c - j * kb_stages) * kX3K;
        return A + j * g.sAk + (TA ? k * g.lda : k);
    };
    auto b_base = [&](int c) {
        const int j = kb_magic ? static_cast<int>(__umulhi(static_cast<unsigned>(c), kb_magic)) : 0;
        const long long k = static_cast<long long>(c - j * kb_stages) * kX3K;
        return B + j * g.sBk + (TB ? k : k * g.ldb);
    };

    SA ra[PF];
    SB rb[PF];
#pragma unroll
    for (int f = 0; f < PF; ++f) {
        ra[f].init(g.M - m0, g.lda, tid);
        rb[f].init(g.N - n0, g.ldb, tid);
    }
    unsigned tiny = 0xffffffffu;

    // DUAL (the 64x64 tiles, whose registers allow it): h.h in acc, the five
    // small products in a second accumulator, whose roundings are 2^-8 of acc's:
    // one full-size rounding per stage instead of six (K = 1024 on two sets
    // 3.4e-7 -> 1.4e-7).
    constexpr bool DUAL = FM * FN == 1;
    floatx16 acc[FM][FN], low[1][1];
#pragma unroll
    for (int r = 0; r < 16; ++r) low[0][0][r] = 0.f;
    auto clear = [&]() {
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
            for (int j = 0; j < FN; ++j)
#pragma unroll
                for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;
    };
    clear();

    struct Frags { bf16x8 a[3][FM], b[3][FN]; };
    auto read_frags = [&](Frags& f, const char* buf) {
        const char* as = buf + h * SA::HALF + (wm + lr) * 16;
        const char* bs = buf + SA::BYTES + h * SB::HALF + (wn + lr) * 16;
#pragma unroll
        for (int p = 2; p >= 0; --p) {
#pragma unroll
            for (int i = 0; i < FM; ++i) f.a[p][i] = *reinterpret_cast<const bf16x8*>(as + p * SA::PLANE + i * 512);
#pragma unroll
            for (int j = 0; j < FN; ++j) f.b[2 - p][j] = *reinterpret_cast<const bf16x8*>(bs + (2 - p) * SB::PLANE + j * 512);
        }
    };
    auto mma = [&](const Frags& f, int p, int q) {
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
            for (int j = 0; j < FN; ++j) {
                floatx16& c = DUAL && p + q > 0 ? low[0][0] : acc[i][j];
                c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(f.a[p][i], f.b[q][j], c, 0, 0, 0);
            }
    };

    // Loop: while stage t's six products run, the stage t + 1 (loaded one
    // iteration ago) is split into the other LDS buffer and stage t + 2's loads
    // are issued, so a load has a whole iteration to land and the conversion's
    // vector instructions run beside the matrix cores'.  Past its last stage a
    // set reloads that stage into the idle buffer: no branch holds a load.
    const int nst = K / kX3K;            // whole stages of the slice
    const int tail = K - nst * kX3K;
    const int rounds = nst / KS;         // every set has a stage: no branch in the loop
    const int last = nst - 1;
    constexpr int U = SA::U + SB::U;
    if (nst > 0) {
        // the stage the next load_all takes, and where its operands start
        int c = min(set, last);
        const float* pa = uniform(a_base(c));
        const float* pb = uniform(b_base(c));
        const long long step_a = KS * kX3K * (TA ? static_cast<long long>(g.lda) : 1);
        const long long step_b = KS * kX3K * (TB ? 1 : static_cast<long long>(g.ldb));
        auto load_all = [&](int f) {
#pragma unroll
            for (int u = 0; u < SA::U; ++u) ra[f].load(u, pa, g.lda);
#pragma unroll
            for (int u = 0; u < SB::U; ++u) rb[f].load(u, pb, g.ldb);
            const bool more = c + KS <= last;
            if (BR) {
                c = more ? c + KS : c;
                pa = uniform(a_base(c));
                pb = uniform(b_base(c));
            } else {
                c += more ? KS : 0;
                pa += more ? step_a : 0;
                pb += more ? step_b : 0;
            }
        };
        auto put = [&](int f, int u, char* buf) {
            if (u < SA::U) ra[f].store(u < SA::U ? u : 0, buf, tid, tiny);
            else rb[f].store(u < SA::U ? 0 : u - SA::U, buf + SA::BYTES, tid, tiny);
        };
        load_all(0);
        if (PF == 2) load_all(1);   // shares the first stage's round trip
#pragma unroll
        for (int u = 0; u < U; ++u) put(0, u, lds);
        load_all(0);
        __syncthreads();
        auto body = [&](int t, int f) {   // f = (t + 1) % PF
            char* nxt = lds + ((t & 1) ^ 1) * BUF;
            Frags cu;
            read_frags(cu, lds + (t & 1) * BUF);
            mma(cu, 2, 0);
            if (0 < U) put(f, 0, nxt);
            mma(cu, 1, 1);
            if (1 < U) put(f, 1, nxt);
            mma(cu, 0, 2);
            if (2 < U) put(f, 2, nxt);
            mma(cu, 1, 0);
            if (3 < U) put(f, 3, nxt);
            load_all(f);
            mma(cu, 0, 1);
            mma(cu, 0, 0);
            __syncthreads();
        };
        int t = 0;
        if (PF == 1) {
            for (; t < rounds; ++t) body(t, 0);
        } else {
            for (; t + 1 < rounds; t += 2) { body(t, 1); body(t + 1, 0); }
            if (t < rounds) body(t++, 1);
        }
        // the uneven round of the wave sets: the stage is in LDS already
        if (KS > 1 && rounds * KS < nst) {
            if (rounds * KS + set <= last) {
                Frags cu;
                read_frags(cu, lds + (rounds & 1) * BUF);
                mma(cu, 2, 0); mma(cu, 1, 1); mma(cu, 0, 2); mma(cu, 1, 0); mma(cu, 0, 1); mma(cu, 0, 0);
            }
            __syncthreads();
        }
    }
    if (tail) {
        // the partial stage: one set, after the loop
        const bool mine = set == nst % KS;
        if (mine) {
            const float* pa = a_base(nst);
            const float* pb = b_base(nst);
#pragma unroll
            for (int u = 0; u < SA::U; ++u) { ra[0].load_tail(u, pa, g.lda, tail, tid); ra[0].store(u, lds, tid, tiny); }
#pragma unroll
            for (int u = 0; u < SB::U; ++u) { rb[0].load_tail(u, pb, g.ldb, tail, tid); rb[0].store(u, lds + SA::BYTES, tid, tiny); }
        }
        __syncthreads();
        if (mine) {
            Frags f;
            read_frags(f, lds);
            mma(f, 2, 0); mma(f, 1, 1); mma(f, 0, 2); mma(f, 1, 0); mma(f, 0, 1); mma(f, 0, 0);
        }
    }

    if (DUAL) {
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[0][0][r] += low[0][0][r];
    }

    // Anything the split could not carry: the whole tile again in fp32.
    float nonfinite = 0.f;
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) nonfinite = fmaf(acc[i][j][r], 0.f, nonfinite);
    if (__syncthreads_or(nonfinite != 0.f || tiny < kX3Tiny)) {
        clear();
        float* as = reinterpret_cast<float*>(lds);
        float* bs = as + kX3K * (BM + 1);
        const int total = nst + (tail ? 1 : 0);
        for (int t = 0; t * KS < total; ++t) {
            const int c = t * KS + set;
            if (c < total) {
                const int kv = c < nst ? kX3K : tail;
                const float* pa = a_base(c);
                const float* pb = b_base(c);
#pragma unroll
                for (int u = 0; u < SA::U; ++u) { ra[0].load_tail(u, pa, g.lda, kv, tid); ra[0].store_f32(u, as, tid); }
#pragma unroll
                for (int u = 0; u < SB::U; ++u) { rb[0].load_tail(u, pb, g.ldb, kv, tid); rb[0].store_f32(u, bs, tid); }
            }
            __syncthreads();
            if (c < total) {
#pragma unroll 1
                for (int k = 0; k < kX3K; k += 2) {
#pragma unroll
                    for (int i = 0; i < FM; ++i)
#pragma unroll
                        for (int j = 0; j < FN; ++j)
                            acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(
                                as[(k + h) * (BM + 1) + wm + 32 * i + lr], bs[(k + h) * (BN + 1) + wn + 32 * j + lr],
                                acc[i][j], 0, 0, 0);
                }
            }
            __syncthreads();
        }
    }

    if (KS > 1) {
        __syncthreads();
        float* red = reinterpret_cast<float*>(lds_all);
        if (set > 0) {
            float* dst = red + (set - 1) * (BM * BN) + tid;
#pragma unroll
            for (int i = 0; i < FM; ++i)
#pragma unroll
                for (int j = 0; j < FN; ++j)
#pragma unroll
                    for (int r = 0; r < 16; ++r) dst[((i * FN + j) * 16 + r) * NT] = acc[i][j][r];
        }
        __syncthreads();
        if (set > 0) return;
#pragma unroll
        for (int s = 1; s < KS; ++s) {
            const float* src = red + (s - 1) * (BM * BN) + tid;
#pragma unroll
            for (int i = 0; i < FM; ++i)
#pragma unroll
                for (int j = 0; j < FN; ++j)
#pragma unroll
                    for (int r = 0; r < 16; ++r) acc[i][j][r] += src[((i * FN + j) * 16 + r) * NT];
        }
    }

    // acc[i][j][r]: row wm + 32 i + 8 (r / 4) + 4 h + r % 4, column wn + 32 j + lr.
    // The destination is a buffer that ends with the tile's last element, so
    // rows past M fall outside it and are dropped, and columns past N are sent
    // there: one address add and one store per element, no branches, and the
    // code of a tile stays small next to what runs before and after it.
    const long long coff = zo * g.sC2 + zi * g.sC;
    const int rows = min(g.M - m0, BM);
    auto tile_rsrc = [&](const float* base, int ld) {
        return __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(uniform(base + static_cast<long long>(m0) * ld + n0)), 0,
                                                 4 * ((rows - 1) * ld + min(g.N - n0, BN)), 0x00020000);
    };
    auto offset = [&](int j, int ld) {
        return wn + 32 * j + lr < g.N - n0 ? 4 * ((wm + 4 * h) * ld + wn + 32 * j + lr) : static_cast<int>(0x80000000);
    };
    auto store = [&](const __amdgpu_buffer_rsrc_t& rs, float v, int off) {
        __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, v), rs, off, 0, 0);
    };
    // a slice's raw sums go to its partials ([slice][batch][M][N], or a whole
    // tile when only the last tiles are split); the ordered reduce applies
    // alpha, beta and R
    const bool slice = part != nullptr, whole = slice && g.tail > 0;
    const int ld = whole ? BN : slice ? g.N : g.ldc;
    const float alpha = slice ? 1.f : g.alpha;
    const __amdgpu_buffer_rsrc_t rd =
        whole ? __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(uniform(part)), 0, 4 * BM * BN, 0x00020000)
              : tile_rsrc(slice ? part : g.C + coff, ld);
    if (slice || g.beta == 0.f) {
#pragma unroll
        for (int j = 0; j < FN; ++j) {
            const int vd = offset(j, ld);
#pragma unroll
            for (int i = 0; i < FM; ++i)
#pragma unroll
                for (int r = 0; r < 16; ++r)
                    store(rd, alpha * acc[i][j][r], vd + 4 * (32 * i + 8 * (r >> 2) + (r & 3)) * ld);
        }
    } else {
        const int ldr = g.R ? g.ldr : g.ldc;
        const __amdgpu_buffer_rsrc_t rr = tile_rsrc((g.R ? g.R : g.C) + coff, ldr);
#pragma unroll
        for (int j = 0; j < FN; ++j) {
            const int vd = offset(j, ld), vr = offset(j, ldr);
#pragma unroll
            for (int i = 0; i < FM; ++i) {
                float t[16];
#pragma unroll
                for (int r = 0; r < 16; ++r)
                    t[r] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(
                        rr, vr + 4 * (32 * i + 8 * (r >> 2) + (r & 3)) * ldr, 0, 0));
#pragma unroll
                for (int r = 0; r < 16; ++r)
                    store(rd, alpha * acc[i][j][r] + g.beta * t[r], vd + 4 * (32 * i + 8 * (r >> 2) + (r & 3)) * ld);
            }
        }
    }
}

template <int BM, int BN, int WM, int WN, int KS, int PF, bool BR, bool TA, bool TB>
__global__ void __launch_bounds__(64 * WM * WN * KS)
sgemm_x3_kernel(const GemmArgs g, const unsigned kb_magic)
{
    // One call of the tile below, so that its code is there once.  With a tail
    // the whole tiles come first (one round of workgroups or more), then the
    // slices of the rest, which share the CUs with them.
    int pid = blockIdx.x, npid = gridDim.x, kbeg = blockIdx.z * g.kchunk, kend = min(g.K, kbeg + g.kchunk);
    float* part = nullptr;
    if (g.tail > 0) {
        const int whole = g.tiles_m * g.tiles_n - g.tail, e = pid - whole;
        if (e < 0) {
            npid = whole;
            kend = g.K;
        } else {
            const int s = e / g.tail, t = e - s * g.tail;
            pid = whole + t;
            npid = 1;
            kbeg = s * g.kchunk;
            kend = min(g.K, kbeg + g.kchunk);
            part = g.ws + static_cast<size_t>(e) * (BM * BN);
        }
    } else if (g.splits > 1) {
        part = g.ws + (static_cast<long long>(blockIdx.z) * gridDim.y + blockIdx.y) * (static_cast<long long>(g.M) * g.N);
    }
    int tm, tn;
    tile_coords(pid, npid, g.tiles_m, g.tiles_n, tm, tn);
    x3_tile<BM, BN, WM, WN, KS, PF, BR, TA, TB>(g, kb_magic, tm, tn, kbeg, kend, part);
}

// The ordered sum of the split tiles: C = alpha * sum_s part[s] + beta * R, four
// columns per thread (tiles are whole rows of float4; C and R take dword-aligned
// ones), eight slices in flight.
typedef float floatx4u __attribute__((ext_vector_type(4), aligned(4)));

template <int BT>
__global__ void __launch_bounds__(256) x3_tail_reduce(const GemmArgs g)
{
    constexpr int PER = BT * BT / 4;
    const int i = blockIdx.x * 256 + threadIdx.x;
    const int t = i / PER, q = i - t * PER;
    int tm, tn;
    tile_coords(g.tiles_m * g.tiles_n - g.tail + t, 1, g.tiles_m, g.tiles_n, tm, tn);
    const int row = tm * BT + q / (BT / 4), col = tn * BT + 4 * (q % (BT / 4));
    if (row >= g.M || col >= g.N) return;
    const floatx4* src = reinterpret_cast<const floatx4*>(g.ws) + static_cast<size_t>(t) * PER + q;
    const size_t step = static_cast<size_t>(g.tail) * PER;
    floatx4 sum = {0.f, 0.f, 0.f, 0.f};
    for (int s = 0; s < g.splits; s += 8) {
        floatx4 v[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) v[u] = src[min(s + u, g.splits - 1) * step];
#pragma unroll
        for (int u = 0; u < 8; ++u)
            if (s + u < g.splits) sum += v[u];
    }
    float* dst = g.C + static_cast<long long>(row) * g.ldc + col;
    const float* r = g.R ? g.R + static_cast<long long>(row) * g.ldr + col : dst;
    if (col + 4 <= g.N) {
        floatx4 o = g.alpha * sum;
        if (g.beta != 0.f) o += g.beta * static_cast<floatx4>(*reinterpret_cast<const floatx4u*>(r));
        *reinterpret_cast<floatx4u*>(dst) = o;
    } else {
        for (int c = 0; col + c < g.N; ++c) dst[c] = g.beta != 0.f ? g.alpha * sum[c] + g.beta * r[c] : g.alpha * sum[c];
    }
}

// Grouped C_g = A_g^T . B_g over the same K (the weight gradients of a training
// step in one launch): workgroup id -> (group, tile) through the groups'
// first-tile table, XCD-contiguous so that an XCD works on neighbouring tiles.
struct X3GroupArgs {
    const float* A[kGroupedMax];
    const float* B[kGroupedMax];
    float* C[kGroupedMax];
    int lda[kGroupedMax], ldb[kGroupedMax], ldc[kGroupedMax], M[kGroupedMax], N[kGroupedMax];
    int tile0[kGroupedMax + 1], tiles_m[kGroupedMax];
    int ngroups, K;
};

template <int BT, int WM, int WN, int KS>
__global__ void __launch_bounds__(64 * WM * WN * KS)
sgemm_x3_grouped_kernel(const X3GroupArgs ga)
{
    const int pid = static_cast<int>(blockIdx.x % 8) * static_cast<int>(gridDim.x / 8) + static_cast<int>(blockIdx.x / 8);
    if (pid >= ga.tile0[ga.ngroups]) return;
    int e = 0;
    while (pid >= ga.tile0[e + 1]) ++e;
    GemmArgs g{};
    g.M = ga.M[e]; g.N = ga.N[e]; g.K = ga.K; g.Kb = ga.K; g.alpha = 1.f;
    g.A = ga.A[e]; g.lda = ga.lda[e];
    g.B = ga.B[e]; g.ldb = ga.ldb[e];
    g.C = ga.C[e]; g.ldc = ga.ldc[e];
    g.inner = 1; g.splits = 1; g.kchunk = ga.K;
    const int t = pid - ga.tile0[e];
    x3_tile<BT, BT, WM, WN, KS, 2, false, true, false>(g, 0, t % ga.tiles_m[e], t / ga.tiles_m[e], 0, ga.K, nullptr);
}

template <int BM, int BN, int WM, int WN, int KS, int PF, bool BR = false>
int launch_cfg_x3(int ta, int tb, GemmArgs g, int batch, hipStream_t stream)
{
    g.tiles_m = ceil_div(g.M, BM);
    g.tiles_n = ceil_div(g.N, BN);
    const long long nwg = static_cast<long long>(g.tiles_m) * g.tiles_n;
    if (nwg > 0x7fffffffLL) return fail(LHIP_E_CAPACITY, "sgemm: %lld workgroups exceed the grid limit", nwg);
    if (g.splits <= 1) { g.splits = 1; g.kchunk = g.K; g.ws = nullptr; }
    const int cpb = g.Kb / kX3K;
    const unsigned magic = g.Kb == g.K ? 0u : static_cast<unsigned>(((1ull << 32) + cpb - 1) / cpb);
    const dim3 grid = g.tail > 0 ? dim3(static_cast<unsigned>(nwg - g.tail + static_cast<long long>(g.tail) * g.splits), 1, 1)
                                 : dim3(static_cast<unsigned>(nwg), batch, g.splits);
    const dim3 block(64 * WM * WN * KS, 1, 1);
    if (!ta && !tb) klaunch(sgemm_x3_kernel<BM, BN, WM, WN, KS, PF, BR, false, false>, grid, block, 0, stream, g, magic);
    else if (ta && !tb) klaunch(sgemm_x3_kernel<BM, BN, WM, WN, KS, PF, BR, true, false>, grid, block, 0, stream, g, magic);
    else if (!ta && tb) klaunch(sgemm_x3_kernel<BM, BN, WM, WN, KS, PF, BR, false, true>, grid, block, 0, stream, g, magic);
    else klaunch(sgemm_x3_kernel<BM, BN, WM, WN, KS, PF, BR, true, true>, grid, block, 0, stream, g, magic);
    const int rc = check_launch("sgemm (x3): kernel launch");
    if (rc == LHIP_OK && g.tail > 0) {
        klaunch(x3_tail_reduce<BM>, g.tail * (BM * BN / 4 / 256), 256, 0, stream, g);
        return check_launch("sgemm (x3): reduce");
    }
    if (rc != LHIP_OK || g.splits <= 1 || g.skip_reduce) return rc;
    return launch_reduce(g, batch, stream);
}

// The tiles, and what each costs on a CU (us, least squares over 2000 timed
// launches of 68 products, all three layouts, ragged and aligned; the fit is
// within 10% of the median launch): `fixed` for the launch, prologue and
// epilogue, `alone` per 16-deep stage while every CU has one workgroup or
// none, `shared` per stage and workgroup once CUs have more (0: not used then).
struct X3Tile {
    int rows;   // the tile is square
    double fixed, alone, shared;
};
constexpr X3Tile kX3Tiles[] = {
    {256, 10.0, 1.68, 1.90},   // 8 waves of 128x64: 53-57% of the bf16 peak at 4096^3 (220-237 TFLOP/s x 6), where power limits it
    {128, 6.0, 0.53, 0.62},    // 8 waves of 64x32, two workgroups per CU
    {128, 8.0, 0.455, 0.0},    // 2 wave sets of 64x64 waves, one workgroup per CU
    {64, 5.5, 0.25, 0.225},    // 2 wave sets of 32x32 waves
    {64, 7.0, 0.195, 0.0},     // 4 wave sets, one workgroup per CU
};

}  // namespace

// The cheapest tile and split by the figures above: a product's stages run one
// workgroup after another on the fullest CU; a split adds the reduce launch and
// its traffic.  Against the best of all tiles and splits the choice lost 2% on
// average over the 68 products, at most 19%.
bool x3_plan(int ta, int tb, int m, int n, int k, int kb, int lda, int ldb, int ldc, int batch, size_t ws_floats,
             bool tail_ok, X3Plan* out)
{
    if (kb % kX3K != 0) return false;
    const int cus = st().cu_count > 0 ? st().cu_count : 256;
    const double mnb = static_cast<double>(m) * n * batch;
    static constexpr int kSplits[] = {1, 2, 3, 4, 6, 8, 12, 16, 24, 32, 48, 64, 96, 128};
    const double per_cus = 1.0 / cus;
    double best = 0.0;
    bool found = false;
    for (int t = 0; t < static_cast<int>(sizeof(kX3Tiles) / sizeof(kX3Tiles[0])); ++t) {
        const X3Tile& c = kX3Tiles[t];
        // byte offsets inside a stage stay below 2^31: rows apart in an operand
        // read along its rows, k apart in a K-major one
        const long long ra = ta ? 16 : c.rows, rb = tb ? c.rows : 16;
        if (ra * lda >= 1LL << 29 || rb * ldb >= 1LL << 29 || static_cast<long long>(c.rows) * std::max(ldc, n) >= 1LL << 29)
            continue;
        const double tiles = static_cast<double>(ceil_div(m, c.rows)) * ceil_div(n, c.rows) * batch;
        for (int s : kSplits) {
            if (s > 1 && (kb > 0 || k < 64 * s || s * mnb > static_cast<double>(ws_floats))) break;
            const double per_cu = tiles * s * per_cus, full = per_cu <= 4.0 ? std::ceil(per_cu) : per_cu + 0.5;
            if (full > 1.0 && (c.shared == 0.0 || s * mnb > 64e6)) break;
            const int stages = static_cast<int>((static_cast<unsigned>(k) + 16u * s - 1u) / (16u * s));
            double us = c.fixed + stages * (full <= 1.0 ? c.alone : c.shared * full);
            if (s > 1) us += 4.0 + (s + 1) * mnb * (4e-6 / 3.5);   // reduce at 3.5 TB/s
            if (!found || us < best) {
                found = true;
                best = us;
                *out = {t, s, stages * kX3K, 0, 0};
            }
        }
        // Tiles a little past a whole round of CUs: the rounds run whole, the
        // rest is split so that it fills the CUs once more for a fraction of a
        // tile's time.
        const long long rest = static_cast<long long>(tiles) % cus, rounds = static_cast<long long>(tiles) / cus;
        if (!tail_ok || batch != 1 || kb > 0 || c.shared == 0.0 || rounds < 1 || rounds > 8 || rest == 0) continue;
        const int s = static_cast<int>(std::min<long long>({cus / rest, k / 64, 32LL}));
        if (s < 2) continue;
        const int stages = ceil_div(k, kX3K * s);
        const double part = static_cast<double>(s) * rest * c.rows * c.rows;
        if (part > static_cast<double>(ws_floats)) continue;
        const double us = c.fixed + k / kX3K * (rounds == 1 ? c.alone : c.shared * rounds) + stages * c.shared + 5.0 +
                          part * (8e-6 / 3.5);
        if (!found || us < best) {
            found = true;
            best = us;
            *out = {t, s, stages * kX3K, static_cast<int>(rest), 0};
        }
    }
    if (!found) return false;
    // slices are whole stages, so there may be fewer than asked for
    if (out->splits > 1) out->splits = ceil_div(k, out->kchunk);
    if (out->splits > 1) {
        const int rows = kX3Tiles[out->tile].rows;
        out->ws_floats = out->tail > 0 ? static_cast<size_t>(out->splits) * out->tail * rows * rows
                                       : static_cast<size_t>(out->splits) * m * n * batch;
    } else {
        out->splits = 1;
        out->kchunk = k;
        out->tail = 0;
    }
    return true;
}

int launch_x3(int tile, bool br, int ta, int tb, const GemmArgs& g, int batch, hipStream_t stream)
{
    auto go = [&](auto brc) {
        constexpr bool BR = decltype(brc)::value;
        switch (tile) {
        case 0: return launch_cfg_x3<256, 256, 2, 4, 1, 1, BR>(ta, tb, g, batch, stream);
        case 1: return launch_cfg_x3<128, 128, 2, 4, 1, 2, BR>(ta, tb, g, batch, stream);
        case 2: return launch_cfg_x3<128, 128, 2, 2, 2, 2, BR>(ta, tb, g, batch, stream);
        case 3: return launch_cfg_x3<64, 64, 2, 2, 2, 2, BR>(ta, tb, g, batch, stream);
        default: return launch_cfg_x3<64, 64, 2, 2, 4, 2, BR>(ta, tb, g, batch, stream);
        }
    };
    return br ? go(std::true_type{}) : go(std::false_type{});
}

// 128x128 tiles once they fill the CUs (each then costs 0.62 us per stage and
// workgroup), 64x64 tiles on two wave sets below that.
int launch_x3_grouped_tn(const GroupedTN* g, int ngroups, int K, hipStream_t stream)
{
    const int cus = st().cu_count > 0 ? st().cu_count : 256;
    auto count = [&](int tile) {
        long long n = 0;
        for (int i = 0; i < ngroups; ++i) n += static_cast<long long>(ceil_div(g[i].M, tile)) * ceil_div(g[i].N, tile);
        return n;
    };
    const int tile = 4 * count(128) >= 3LL * cus ? 128 : 64;
    const long long tiles = count(tile);
    if (tiles > 0x7ffffff0LL) return fail(LHIP_E_CAPACITY, "sgemm_grouped_tn: too many tiles");
    X3GroupArgs ga{};
    int first = 0;
    for (int i = 0; i < ngroups; ++i) {
        ga.A[i] = g[i].A; ga.B[i] = g[i].B; ga.C[i] = g[i].C;
        ga.lda[i] = g[i].lda; ga.ldb[i] = g[i].ldb; ga.ldc[i] = g[i].ldc;
        ga.M[i] = g[i].M; ga.N[i] = g[i].N;
        ga.tile0[i] = first;
        ga.tiles_m[i] = ceil_div(g[i].M, tile);
        first += ga.tiles_m[i] * ceil_div(g[i].N, tile);
    }
    ga.tile0[ngroups] = first;
    ga.ngroups = ngroups;
    ga.K = K;
    const unsigned grid = (static_cast<unsigned>(first) + 7u) / 8u * 8u;
    if (tile == 128) klaunch(sgemm_x3_grouped_kernel<128, 2, 4, 1>, grid, 512, 0, stream, ga);
    else klaunch(sgemm_x3_grouped_kernel<64, 2, 2, 2>, grid, 512, 0, stream, ga);
    return check_launch("sgemm_grouped_tn (x3)");
}

}  // namespace lhip
