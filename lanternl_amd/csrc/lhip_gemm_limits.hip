// lhip_gemm_limits.hip -- the split-K partials a product is documented to need.
//
// Two refusals of the ABI are stated in terms of these sizes: lhip_sgemm_noalloc
// refuses a product whose partials exceed its fixed array, and a product
// recorded into a program is refused when the library workspace would have to
// grow for them.  Callers plan for these limits (which shapes to warm up before
// recording, which to send to lhip_sgemm), so they are kept as they are while
// the kernels' own slices are planned from measured rates (x3_plan), always
// within the fixed array.
#include <algorithm>

#include "lhip_gemm.h"

namespace lhip {
namespace {

// 33..64 rows with long K and wide N: one 64-row tile band of 64x64 tiles on
// four wave sets, split over K so that tiles x slices fill the CUs (M = 64,
// K = N = 4096: 64 tiles x 4 slices, 31.8 us against 45 us on the skinny MFMA
// form and its reduce).
bool ks_split_ok(int m, int n, int k, int batch)
{
    return batch == 1 && m > 32 && m <= 64 && n >= 1024 && k >= 2048;
}

int ks_split_plan(int m, int n, int k, size_t ws_floats, int* kchunk_out)
{
    const int cus = st().cu_count > 0 ? st().cu_count : 256;
    const long long tiles = ceil_div(n, 64);
    long long s = std::max<long long>(1, cus / tiles);
    s = std::min<long long>(s, k / 512);
    s = std::min<long long>(s, 16);
    const long long mn = static_cast<long long>(m) * n;
    s = std::min<long long>(s, static_cast<long long>(ws_floats / mn));
    if (s < 2) return 1;
    const int kchunk = ceil_div(ceil_div(k, static_cast<int>(s)), 32) * 32;
    *kchunk_out = kchunk;
    return ceil_div(k, kchunk);
}

// Below the 64x64-tile threshold, the 32x32 small kernel is used unless K is
// long AND both output dimensions exceed 64: its 32-wide tiles re-read A N/32
// times and B M/32 times, which for long K costs more L2/MALL traffic than
// the 64x64 tiles (+ split-K) save in latency.
bool use_small_kernel(int m, int n, int k) { return k <= 2048 || m <= 64 || n <= 64; }

// 256x256 tiles split over K (one batch): when the tiles alone would fill
// between a quarter and all of the CUs (e.g. 2048^3: 64 tiles), each tile's K
// is cut into slices of at least 512 so that tiles x slices covers the CUs;
// the slices are summed in order by the reduce.  K % 32 == 0 keeps every
// slice whole.  Returns the slice count (1: not this path).
int split256_plan(int m, int n, int k, int batch, size_t ws_floats, int* kchunk_out)
{
    const int cus = st().cu_count > 0 ? st().cu_count : 256;
    const long long tiles = static_cast<long long>(ceil_div(m, 256)) * ceil_div(n, 256);
    if (batch != 1 || tiles >= cus || 4 * tiles < cus || k % 32 != 0) return 1;
    long long s = (cus + tiles - 1) / tiles;
    s = std::min<long long>(s, k / 512);
    const long long mn = static_cast<long long>(m) * n;
    if (mn > 0) s = std::min<long long>(s, static_cast<long long>(ws_floats / mn));
    if (s < 2) return 1;
    const int kchunk = ceil_div(ceil_div(k, static_cast<int>(s)), 32) * 32;
    const int splits = ceil_div(k, kchunk);
    if (splits < 2) return 1;
    *kchunk_out = kchunk;
    return splits;
}

// The 256x256-tile kernel on 128x128 tiles: when there are fewer 256x256
// tiles than CUs but at least ~3/4 of a CU's worth of 128x128 tiles, unless
// the 256x256 tiles split over K into slices of 1024 or more (long K: the
// big tiles' 84% beat the small ones' 79% at 2048x2048x8192).  Measured:
// 2048^3 151.8 (256x256 in 4 slices of 512) -> 143.1 us; the C3 logits
// 512x32000x128 57.3 -> 51.0 us; C3 dW 128x32000x512 52.4 -> 45.7 us.
// Few 128x128 tiles (at most an eighth of the CUs) over a long K: the same
// kernel split over K into one slice per CU's worth of tiles, slices of 448+
// (C3 dhidden 512x128x32000: 4 tiles x 64 slices of 512, 53-57 -> 48 us; a
// split count that leaves CUs idle or doubles up measured slower).  Batch 1.
int big128_split_plan(int m, int n, int k, size_t ws_floats, int* kchunk_out)
{
    const int cus = st().cu_count > 0 ? st().cu_count : 256;
    if (m <= 64 || n <= 64) return 1;
    const long long t128 = static_cast<long long>(ceil_div(m, 128)) * ceil_div(n, 128);
    if (8 * t128 > cus) return 1;
    const long long s = cus / t128;
    const int kchunk = static_cast<int>(ceil_div(ceil_div(static_cast<long long>(k), s), 32LL) * 32);
    if (kchunk < 448) return 1;
    const int splits = ceil_div(k, kchunk);
    if (splits < 2 || static_cast<size_t>(splits) * m * n > ws_floats) return 1;
    *kchunk_out = kchunk;
    return splits;
}

bool big128_ok(int m, int n, int batch, int s256, int kc256)
{
    const int cus = st().cu_count > 0 ? st().cu_count : 256;
    const long long t256 = static_cast<long long>(ceil_div(m, 256)) * ceil_div(n, 256) * batch;
    const long long t128 = static_cast<long long>(ceil_div(m, 128)) * ceil_div(n, 128) * batch;
    return t256 < cus && 4 * t128 >= 3LL * cus && !(s256 > 1 && kc256 >= 1024);
}

// K per split slice from which a split 64x64-tile product runs on four wave sets.
constexpr int kKsSliceMin = 1024;

}  // namespace

int splitk_plan(int m, int n, int k, int batch, size_t ws_floats, int* kchunk_out)
{
    const int cus = st().cu_count > 0 ? st().cu_count : 256;
    const long long tiles64 = static_cast<long long>(ceil_div(m, 64)) * ceil_div(n, 64) * batch;
    const long long big_tiles = static_cast<long long>(ceil_div(m, 128)) * ceil_div(n, 128) * batch;
    if (big_tiles >= cus || tiles64 >= cus) return 1;
    const long long mnb = static_cast<long long>(m) * n * batch;
    const long long tiles32 = static_cast<long long>(ceil_div(m, 32)) * ceil_div(n, 32) * batch;
    long long tiles, min_k;
    int unit;
    if (use_small_kernel(m, n, k)) {
        // 32x32 tiles, K shared by four waves: split only long K (each wave
        // walks K/4 serially; below 1024 the extra reduce launch costs more
        // than the shorter walk saves)
        if (k < 1024) return 1;
        tiles = static_cast<long long>(ceil_div(m, 32)) * ceil_div(n, 32) * batch;
        unit = 32;
        min_k = 256;
        // 16x16 tiles (fewer 32x32 tiles than CUs) take long K unsplit: their
        // passes are software-pipelined, which beats a split plus its reduce
        if (tiles < cus) return 1;
    } else {
        // 64x64 tiles, 32-deep K tiles walked by one workgroup
        tiles = tiles64;
        unit = 32;
        min_k = 128;
        // slices of 1024 or more K at one workgroup per CU run on four wave
        // sets (ks_slices), which beats two single-set workgroups per CU
        const long long s1 = (cus + tiles - 1) / tiles;
        if (k / s1 >= kKsSliceMin) {
            long long s = std::min<long long>(s1, 64);
            if (mnb > 0) s = std::min<long long>(s, static_cast<long long>(ws_floats / mnb));
            if (s >= 2) {
                const int kchunk = ceil_div(ceil_div(k, s), 32) * 32;
                const int splits = ceil_div(k, kchunk);
                if (splits >= 2) {
                    *kchunk_out = kchunk;
                    return splits;
                }
            }
        }
    }
    long long s = (2LL * cus + tiles - 1) / tiles;          // aim at ~2 workgroups per CU
    s = std::min<long long>(s, k / min_k);
    s = std::min<long long>(s, 64);
    if (mnb > 0) s = std::min<long long>(s, static_cast<long long>(ws_floats / mnb));
    if (s < 2) return 1;
    const int kchunk = ceil_div(ceil_div(k, s), unit) * unit;
    const int splits = ceil_div(k, kchunk);
    if (splits < 2) return 1;
    *kchunk_out = kchunk;
    return splits;
}

size_t documented_partials(int transa, int transb, int m, int n, int k, int batch)
{
    const size_t cap = static_cast<size_t>(1) << 26;
    int kchunk = 0, splits = 1;
    const bool skinny = !transb && m <= 64 && n >= 256 && batch == 1;
    if (ks_split_ok(m, n, k, batch)) {
        splits = ks_split_plan(m, n, k, cap, &kchunk);
        if (splits <= 1 && skinny) splits = skinny_plan(m, n, k, cap, &kchunk);
    } else if (skinny) {
        splits = skinny_plan(m, n, k, cap, &kchunk);
    } else {
        splits = split256_plan(m, n, k, batch, cap, &kchunk);
        if (big128_ok(m, n, batch, splits, kchunk)) splits = 1;
        else if (splits <= 1) {
            splits = batch == 1 ? big128_split_plan(m, n, k, cap, &kchunk) : 1;
            if (splits <= 1) splits = splitk_plan(m, n, k, batch, cap, &kchunk);
        }
    }
    return splits > 1 ? static_cast<size_t>(splits) * m * n * batch : 0;
}

}  // namespace lhip
