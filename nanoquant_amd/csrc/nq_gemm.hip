// Prefill path (>= 128 tokens): one-bit weights x 16-bit activations on the MFMA units of gfx950.
//
//   C[t, j] = s_out[j] * sum_k (x[t, k] * s_in[k]) * sgn(W[j, k])
//
// Replaces Marlin_impl / marlin_cuda_template of the reference (src/nanoquant/kernel/cuda/
// gemm_kernel.cu:278-932) in function only.  The tile itself is in nq_tile.h; this file says which tiles a launch is cut
// into.  Up to 16 problems on the same tokens share a launch; there is no split of k between workgroups, so no scratch.
#include <cmath>

#include "nq_common.h"
#include "nq_kernels.h"
#include "nq_mfma.h"
#include "nq_tile.h"

namespace nq {

// Workgroups of all problems one behind the other: workgroup b belongs to the problem p with first[p] <= b < first[p + 1].
// A linear by itself has kernels of its own (N = 1): finding the problem is a round trip to the kernel arguments ahead of the
// first load (2048 x 2048 on 128 tokens, both GEMMs in a graph: 9.95 us with the kernels of 16, 9.3 with these).
constexpr int kGroupMax = 16;   // 16 problems of 64 bytes: well inside the 4 KB of kernel arguments
template <int N>
struct GemmGroup {
    GemmArgs a[N];
    int first[N + 1];
};

// Workgroups go to the 8 XCDs round-robin by id and first[p] is a multiple of 8, so (id - first[p]) mod 8 is the XCD; the
// mapping keeps the workgroups that share an activation slab on one XCD (one L2) where the number of token blocks gy allows
// it: gy a multiple of 8 (or large): XCD = token block mod 8; gy = 1, 2, 4: XCD x owns token block x mod gy and every
// (8/gy)-th row block; otherwise row blocks run fastest.  group_blocks() is the host's count for the same mapping.
__host__ __device__ inline int group_mode(int gy) { return (gy % 8 == 0 || gy >= 32) ? 0 : (8 % gy == 0) ? 1 : 2; }
static int group_blocks(int gx, int gy) {
    const int mode = group_mode(gy);
    if (mode == 0) return gx * ((gy + 7) / 8 * 8);
    if (mode == 1) { const int sub = 8 / gy; return (gx + sub - 1) / sub * 8; }
    return (gx * gy + 7) / 8 * 8;
}

// Row block and token block of workgroup `local` of a problem; false: none.
template <int TT>
__device__ __forceinline__ bool tile_of(const GemmArgs& a, int local, int& bx, int& by) {
    const int gx = a.gx, gy = (a.T + 32 * TT - 1) / (32 * TT);
    const int mode = group_mode(gy);
    if (mode == 0) {
        const int slot = local >> 3;
        by = (slot / gx) * 8 + (local & 7);
        bx = slot % gx;
    } else if (mode == 1) {
        const int sub = 8 / gy, xcd = local & 7;
        by = xcd % gy;
        bx = (local >> 3) * sub + xcd / gy;
    } else {
        bx = local % gx;
        by = local / gx;
    }
    return bx < gx && by < gy;
}

template <int DT, bool SCALED, int TT, int RT, int WR, int WK, int NB, int N>
__global__ __launch_bounds__(64 * WR * WK, 2) void gemm_tile_kernel(GemmGroup<N> g) {
    extern __shared__ __attribute__((aligned(16))) uint16_t tile_lds[];
    const int b = blockIdx.x;
    // first[i] of the unused entries is the grid size, so no count is needed; all of first[] comes with one load
    int p = 0;
#pragma unroll
    for (int i = 1; i < N; ++i) p += b >= g.first[i] ? 1 : 0;
    const GemmArgs a = g.a[p];
    int bx, by;
    if (!tile_of<TT>(a, N > 1 ? b - g.first[p] : b, bx, by)) return;
    // Half a tile or less is left of the tokens: a tile of half the tokens, whose sums are the same.  In us, whole tiles / so:
    // 3072 -> 11008 rows on 333 tokens 34.1 / 29.5 on 64 x 256, 30.6 / 27.9 on 64 x 128; 2048 -> 4096 on 2080 tokens 46.5 / 38.6 on
    // 128 x 256; 3072 -> 11008 on 4112 tokens 233 / 222.
    if constexpr (TT > 1) {
        if (a.T - 32 * TT * by <= 16 * TT) return Tile<DT, SCALED, TT / 2, RT, WR, WK, NB>::run(a, bx, 2 * by, tile_lds);
    }
    Tile<DT, SCALED, TT, RT, WR, WK, NB>::run(a, bx, by, tile_lds);
}

// Sums of terms: the first `heads` entries are one per output, next[p] is the entry of the term behind p (or -1).
struct GemmSums {
    GemmGroup<kGroupMax> g;
    int next[kGroupMax];
};
template <int DT, int TT, int RT, int WR, int WK, int NB>
__global__ __launch_bounds__(64 * WR * WK, 2) void gemm_tile_sum_kernel(GemmSums s) {
    extern __shared__ __attribute__((aligned(16))) uint16_t tile_lds[];
    const int b = blockIdx.x;
    int p = 0;
#pragma unroll
    for (int i = 1; i < kGroupMax; ++i) p += b >= s.g.first[i] ? 1 : 0;
    int bx, by;
    if (!tile_of<TT>(s.g.a[p], b - s.g.first[p], bx, by)) return;
    if constexpr (TT > 1) {
        if (s.g.a[p].T - 32 * TT * by <= 16 * TT) return Tile<DT, false, TT / 2, RT, WR, WK, NB>::run_sum(s.g.a, s.next, p, bx, 2 * by, tile_lds);
    }
    Tile<DT, false, TT, RT, WR, WK, NB>::run_sum(s.g.a, s.next, p, bx, by, tile_lds);
}

// ---- host side --------------------------------------------------------------------------------
// The tiles a launch can be cut into, and what one costs.  Few-token tiles: 32 tokens x 32 RT rows, four wavefronts that split
// k (the sums of a linear are the same whatever RT).  Block tiles: 64 or 128 tokens x 128 or 256 rows, every wavefront walks
// the whole k (the same sums for all three).  Sizes that were tried and are nowhere ahead by more than 3 %: 32 x 128 and 64 x 64
// with split k, 64 x 512.  64 x 128 split over two or four k groups gains up to 15 % on 2 % of the shapes.
//
// Time of a launch in us = start + round * (rounds of resident workgroups) + sum over the rounds of (k tiles per wavefront) *
// tile[workgroups per compute unit in that round - 1], fitted to 1346 launches (32 to 4096 tokens, k of 1 to 43 tiles, 256 to 22016
// rows, weights from memory): the middle 90 % of the fits are within -20 .. +15 %, and the size that the estimate picks is 2 %
// slower than the best one on average, 11 % in the worst twentieth.
struct TileCost {
    float start, round, tile[4];     // tile[i] = 0: i + 1 workgroups do not fit a compute unit
};
struct TileVariant {
    int tt, rt, wr, wk, nb;
    int sum_fit;                     // gemm_tile_sum_kernel: workgroups that fit a compute unit (0: none of this size), and what
    float sum_start;                 // it takes beyond the costs below where a single round of them does it all
    TileCost cost[2];                // without and with s_in
};
constexpr int kFewTiles = 3, kVariantCount = 6;      // the first kFewTiles entries are few-token tiles
constexpr TileVariant kVariants[kVariantCount] = {
    {1, 1, 1, 4, 4, 2, 0.f, {{2.27f, 0.89f, {0.75f, 1.77f}}, {2.01f, 1.62f, {0.72f, 1.63f}}}},
    {1, 2, 1, 4, 4, 2, 0.f, {{2.30f, 1.22f, {1.10f, 2.44f}}, {1.94f, 2.00f, {1.01f, 2.33f}}}},
    {1, 3, 1, 4, 3, 2, 0.f, {{2.46f, 1.30f, {1.60f, 3.38f}}, {1.57f, 2.59f, {1.46f, 3.21f}}}},
    {2, 1, 4, 1, 4, 4, 0.f, {{1.35f, 2.84f, {0.69f, 1.63f, 2.83f, 3.60f}}, {2.19f, 1.50f, {0.90f, 1.74f, 2.81f, 3.90f}}}},
    {2, 2, 4, 1, 4, 2, 2.f, {{0.84f, 4.08f, {1.14f, 3.04f, 4.89f}}, {0.f, 4.27f, {1.33f, 3.05f, 4.96f}}}},
    {4, 2, 4, 1, 4, 0, 0.f, {{0.f, 6.09f, {2.18f, 5.76f}}, {0.f, 5.73f, {2.33f, 5.57f}}}},
};

struct GemmShapes {
    int count, T;
    const int *K, *R;
    bool scaled, sums;               // sums: for gemm_tile_sum_kernel
    double cus;                      // compute units
};
// The costs are of a device of 256, which also stands in where there is none to ask.
static double device_units() {
    const int n = compute_units();
    return n > 0 ? n : 256;
}

static int tile_gx(const TileVariant& v, int R) { return (R + 32 * v.rt * v.wr - 1) / (32 * v.rt * v.wr); }
static int tile_gy(const TileVariant& v, int T) { return (T + 32 * v.tt - 1) / (32 * v.tt); }

static double tile_time(const TileVariant& v, const GemmShapes& s) {
    const TileCost& c = v.cost[s.scaled];
    const int gy = tile_gy(v, s.T);
    // a last token block of half the tokens or less costs 0.6 of one (the signs are read and decoded all the same)
    const double whole = v.tt > 1 && s.T - (gy - 1) * 32 * v.tt <= 16 * v.tt ? (gy - 0.4) / gy : 1.0;
    double blocks = 0, work = 0;                 // whole workgroups; their k tiles per wavefront, summed
    int longest = 0;
    for (int p = 0; p < s.count; ++p) {
        const double n = whole * group_blocks(tile_gx(v, s.R[p]), gy);
        const int tiles = (s.K[p] / kTileK + v.wk - 1) / v.wk;
        blocks += n;
        work += n * tiles;
        longest = tiles > longest ? tiles : longest;
    }
    int fit = 0;
    while (fit < (s.sums ? v.sum_fit : 4) && c.tile[fit] > 0.f) ++fit;
    const double mean = work / blocks;
    auto walk = [&](double workgroups, double* rounds) {
        const long per_cu = (long)std::ceil(workgroups / s.cus), full = per_cu / fit, rest = per_cu % fit;
        *rounds = (double)full + (rest ? 1 : 0);
        const double all = mean * ((double)full * c.tile[fit - 1] + (rest ? c.tile[rest - 1] : 0.f));
        // The longest problem's workgroups start first and share their compute units with those of mean length (4096 and 11008 ->
        // 3072 rows on 768 tokens: 164, not 116, on 128 x 256; panels 128).
        const long beside = per_cu < fit ? per_cu : fit;
        const double one = mean * c.tile[beside - 1] + ((double)longest - mean) * c.tile[0];
        return all > one ? all : one;
    };
    double rounds, real_rounds;
    const double time = walk(blocks, &rounds), real = walk(blocks / whole, &real_rounds);
    // half the way to what as many whole workgroups would take: the cut ones still share compute units
    return c.start + (s.sums && real_rounds <= 1.0 ? v.sum_start : 0.f) + c.round * 0.5 * (rounds + real_rounds) + 0.5 * (time + real);
}

static int best_tile(const GemmShapes& s, int begin, int end, double* time) {
    int best = begin;
    *time = tile_time(kVariants[begin], s);
    for (int i = begin + 1; i < end; ++i) {
        const double t = tile_time(kVariants[i], s);
        if (t < *time) { *time = t; best = i; }
    }
    return best;
}

// Few-token or block tiles.  The two add in different orders, so where the choice is left to the estimate the last bits of a linear
// depend on what shares the launch.  They do not up to kSameBitsTokens tokens (few-token tiles, unless the caller allows
// others from kAnyTileFrom tokens on: there a launch of many rows gains up to a third, 3072 -> 22016 rows on 128 tokens 27 -> 21
// us) nor, in a group, above kFewMaxTokens (block tiles; few-token ones would be ahead for few rows only, 4096 -> 256 rows on 3000 tokens 20 / 13).  What
// few-token tiles read again counts once per INPUT: terms with inputs of their own (every second GEMM, whose inputs are the h)
// bring as many token rows as so many times the tokens, and beyond some 1800 of them block tiles are the faster ones.
// The estimate's own error is a few per cent, hence the margins.
constexpr int kSameBitsTokens = 160, kAnyTileFrom = 100, kFewMaxTokens = 1536;
constexpr long kFewMaxInputs = 1800;

static bool inputs_too_many(int count, const void* const* x, int T, const int* K) {
    long tiles = 0;
    int longest = 0;
    for (int p = 0; p < count; ++p) {
        longest = K[p] / kTileK > longest ? K[p] / kTileK : longest;
        bool seen = false;
        for (int q = 0; q < p; ++q) seen = seen || x[q] == x[p];
        if (!seen) tiles += K[p] / kTileK;
    }
    return (long)T * tiles > kFewMaxInputs * longest;
}

static int choose_tile(const void* const* x, const GemmShapes& s, int use, double* time) {
    double few_time = 0, block_time = 0;
    const int few = best_tile(s, 0, kFewTiles, &few_time), block = best_tile(s, kFewTiles, kVariantCount, &block_time);
    bool take_few = few_time < 0.95 * block_time;
    if (s.T <= kSameBitsTokens) take_few = use != kGemmAnyTile || s.T < kAnyTileFrom || block_time >= 0.9 * few_time;
    else if (use != kGemmAlone && (s.T > kFewMaxTokens || inputs_too_many(s.count, x, s.T, s.K))) take_few = false;
    *time = take_few ? few_time : block_time;
    return take_few ? few : block;
}

double gemm_tiles_time(int count, const void* const* x, int T, const int* K, const int* R, bool scaled) {
    double time = 0;
    choose_tile(x, GemmShapes{count, T, K, R, scaled, false, device_units()}, kGemmAnyTile, &time);
    return time;
}

template <int DT, bool SCALED, int V, int N>
static hipError_t launch_tiles(const GemmGroup<N>& g, int blocks, hipStream_t stream) {
    constexpr TileVariant v = kVariants[V];
    using S = TileShape<v.tt, v.rt, v.wr, v.wk, v.nb>;
    auto kern = gemm_tile_kernel<DT, SCALED, v.tt, v.rt, v.wr, v.wk, v.nb, N>;
    static PerDeviceFlag raised;                 // per kernel and device
    const int dev = current_device();
    if (S::kLds > 64 * 1024 && !raised.test(dev)) {
        hipError_t e = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)S::kLds);
        if (e != hipSuccess) return e;
        raised.set(dev);
    }
    hipLaunchKernelGGL(kern, dim3(blocks), dim3(S::kThreads), S::kLds, stream, g);
    return hipGetLastError();
}
template <int DT, bool SCALED, int N>
static hipError_t launch_tiles(int v, const GemmGroup<N>& g, int blocks, hipStream_t stream) {
    static_assert(kVariantCount == 6, "one case per entry");
    switch (v) {
        case 0: return launch_tiles<DT, SCALED, 0, N>(g, blocks, stream);
        case 1: return launch_tiles<DT, SCALED, 1, N>(g, blocks, stream);
        case 2: return launch_tiles<DT, SCALED, 2, N>(g, blocks, stream);
        case 3: return launch_tiles<DT, SCALED, 3, N>(g, blocks, stream);
        case 4: return launch_tiles<DT, SCALED, 4, N>(g, blocks, stream);
        default: return launch_tiles<DT, SCALED, 5, N>(g, blocks, stream);
    }
}

template <int N>
static hipError_t launch_group(int pick, int dtype, int count, const void* const* x, const uint32_t* const* tiles,
                               const void* const* s_in, const void* const* s_out, const void* const* bias, void* const* y,
                               int T, const int* K, const int* R, hipStream_t stream) {
    // Longest k first: the workgroups that run longest start first, the short ones fill in behind them.
    int order[N];
    for (int p = 0; p < count; ++p) order[p] = p;
    for (int i = 1; i < count; ++i)
        for (int j = i; j > 0 && K[order[j]] > K[order[j - 1]]; --j) { const int t = order[j]; order[j] = order[j - 1]; order[j - 1] = t; }
    GemmGroup<N> g;
    int blocks = 0;
    for (int p = 0; p < N; ++p) {
        const int q = order[p < count ? p : count - 1];
        GemmArgs& a = g.a[p];
        a.x = x[q]; a.tiles = (const uint4*)tiles[q];
        a.s_in = (const uint16_t*)(s_in ? s_in[q] : nullptr); a.s_out = (const uint16_t*)(s_out ? s_out[q] : nullptr);
        a.bias = (const uint16_t*)(bias ? bias[q] : nullptr);
        a.y = y[q];
        a.T = T; a.K = K[q]; a.R = R[q];
        a.gx = tile_gx(kVariants[pick], R[q]);
        g.first[p] = blocks;
        if (p < count) blocks += group_blocks(a.gx, tile_gy(kVariants[pick], T));
    }
    g.first[N] = blocks;
    const bool scaled = g.a[0].s_in != nullptr;
    if (dtype == 0) return scaled ? launch_tiles<0, true, N>(pick, g, blocks, stream) : launch_tiles<0, false, N>(pick, g, blocks, stream);
    return scaled ? launch_tiles<1, true, N>(pick, g, blocks, stream) : launch_tiles<1, false, N>(pick, g, blocks, stream);
}

// A launch with problems of more than kGemmMaxK columns: one problem after the other, those token by token, every token a problem
// of its own on the smallest tile (offsets of its further, missing tokens may wrap round: what they read is not stored).
static hipError_t launch_apart(int dtype, int count, const void* const* x, const uint32_t* const* tiles, const void* const* s_in,
                               const void* const* s_out, const void* const* bias, void* const* y, int T, const int* K, const int* R,
                               int use, hipStream_t stream) {
    for (int p = 0; p < count; ++p)
        if (K[p] >= kGemmEndK) return hipErrorInvalidValue;
    for (int p = 0; p < count; ++p) {
        const void* si = s_in ? s_in[p] : nullptr;
        const void* so = s_out ? s_out[p] : nullptr;
        const void* bs = bias ? bias[p] : nullptr;
        if (K[p] <= kGemmMaxK) {
            const hipError_t e = gemm_onebit_group(dtype, 1, x + p, tiles + p, &si, &so, &bs, y + p, T, K + p, R + p, use, stream);
            if (e != hipSuccess) return e;
            continue;
        }
        for (int t = 0; t < T; t += kGroupMax) {
            const int tokens = T - t < kGroupMax ? T - t : kGroupMax;
            const void *xs[kGroupMax], *sis[kGroupMax], *sos[kGroupMax], *bss[kGroupMax];
            const uint32_t* ws[kGroupMax];
            void* ys[kGroupMax];
            int Ks[kGroupMax], Rs[kGroupMax];
            for (int j = 0; j < tokens; ++j) {
                xs[j] = (const uint16_t*)x[p] + (size_t)(t + j) * K[p];
                ys[j] = (uint16_t*)y[p] + (size_t)(t + j) * R[p];
                ws[j] = tiles[p]; sis[j] = si; sos[j] = so; bss[j] = bs;
                Ks[j] = K[p]; Rs[j] = R[p];
            }
            const hipError_t e = launch_group<kGroupMax>(0, dtype, tokens, xs, ws, sis, sos, bss, ys, 1, Ks, Rs, stream);
            if (e != hipSuccess) return e;
        }
    }
    return hipSuccess;
}

// GEMMs of several problems on the same token count in one launch; every problem: K % 256 == 0, R % 32 == 0, and
// either all have input scales or none (checked by the caller).
hipError_t gemm_onebit_group(int dtype, int count, const void* const* x, const uint32_t* const* tiles,
                             const void* const* s_in, const void* const* s_out, const void* const* bias, void* const* y,
                             int T, const int* K, const int* R, int use, hipStream_t stream) {
    if (count < 1 || count > kGroupMax) return hipErrorInvalidValue;
    for (int p = 0; p < count; ++p)
        if (K[p] > kGemmMaxK) return launch_apart(dtype, count, x, tiles, s_in, s_out, bias, y, T, K, R, use, stream);
    double time = 0;
    const int pick = choose_tile(x, GemmShapes{count, T, K, R, s_in && s_in[0], false, device_units()}, use, &time);
    if (count == 1) return launch_group<1>(pick, dtype, count, x, tiles, s_in, s_out, bias, y, T, K, R, stream);
    return launch_group<kGroupMax>(pick, dtype, count, x, tiles, s_in, s_out, bias, y, T, K, R, stream);
}

// ---- sums of terms ------------------------------------------------------------------------------
// The tiles whose accumulators fit the registers twice.
constexpr int kSumVariantCount = 5;

template <int DT, int V>
static hipError_t launch_sums(const GemmSums& s, int blocks, hipStream_t stream) {
    constexpr TileVariant v = kVariants[V];
    using S = TileShape<v.tt, v.rt, v.wr, v.wk, v.nb>;
    auto kern = gemm_tile_sum_kernel<DT, v.tt, v.rt, v.wr, v.wk, v.nb>;
    static PerDeviceFlag raised;
    const int dev = current_device();
    if (S::kLds > 64 * 1024 && !raised.test(dev)) {
        hipError_t e = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)S::kLds);
        if (e != hipSuccess) return e;
        raised.set(dev);
    }
    hipLaunchKernelGGL(kern, dim3(blocks), dim3(S::kThreads), S::kLds, stream, s);
    return hipGetLastError();
}
template <int DT>
static hipError_t launch_sums(int v, const GemmSums& s, int blocks, hipStream_t stream) {
    static_assert(kSumVariantCount == 5, "one case per entry");
    switch (v) {
        case 0: return launch_sums<DT, 0>(s, blocks, stream);
        case 1: return launch_sums<DT, 1>(s, blocks, stream);
        case 2: return launch_sums<DT, 2>(s, blocks, stream);
        case 3: return launch_sums<DT, 3>(s, blocks, stream);
        default: return launch_sums<DT, 4>(s, blocks, stream);
    }
}

// The outputs of a launch of sums: one per term that no other term's next[] names, longest k first.
struct SumHeads {
    int count, longest;                                // outputs; most terms of one
    int at[kGroupMax], K[kGroupMax], R[kGroupMax];     // first term, k summed over the terms, rows
    int split_k[kGroupMax];                            // the same sum of whole rounds of four wavefronts that split k
    bool head[kGroupMax];
};
static SumHeads sum_heads(int count, const int* next, const int* K, const int* R) {
    SumHeads h;
    h.count = h.longest = 0;
    for (int i = 0; i < count; ++i) h.head[i] = true;
    for (int i = 0; i < count; ++i)
        if (next[i] >= 0) h.head[next[i]] = false;
    for (int i = 0; i < count; ++i) {
        if (!h.head[i]) continue;
        int k = 0, split = 0, terms = 0;
        for (int t = i; t >= 0; t = next[t], ++terms) {
            k += K[t];
            split += (K[t] + 4 * kTileK - 1) / (4 * kTileK) * (4 * kTileK);
        }
        h.longest = h.longest > terms ? h.longest : terms;
        int j = h.count++;
        for (; j > 0 && h.K[j - 1] < k; --j) {
            h.at[j] = h.at[j - 1]; h.K[j] = h.K[j - 1]; h.R[j] = h.R[j - 1]; h.split_k[j] = h.split_k[j - 1];
        }
        h.at[j] = i; h.K[j] = k; h.R[j] = R[i]; h.split_k[j] = split;
    }
    return h;
}
// A sum costs about what one problem of its terms' k costs, and some 1.5 us for every further term, whose ring is filled anew;
// but of 64 x 256 tiles, whose accumulators it holds twice (196 registers), only two workgroups fit a compute unit, and in a
// single round of them nobody multiplies while a ring is filled.  The pick is 0.3 % slower than the best tile on average and 9 %
// at worst, over 160 pairs of stages (100 to 4096 tokens, seven linears of two models); priced as the plain kernel 0.7 and 12 %
// ({q, k, v} of Qwen3-8B at 0.9 bits on 333 tokens: both stages 37.5 us on 64 x 256, 33.6 on 64 x 128).
// Where k is split between wavefronts a term of one k tile takes as long as one of four: counted by its own k, two terms of
// 256 -> 64 rows on 8192 tokens took such a tile, 20.3 us with the first stage; 17.4 apart and added, 16.6 on the tile taken now.
static int choose_sum_tile(const SumHeads& h, int T, double* time) {
    double few_time = 0, block_time = 0;
    const double cus = device_units();
    const int few = best_tile(GemmShapes{h.count, T, h.split_k, h.R, false, true, cus}, 0, kFewTiles, &few_time);
    const int block = best_tile(GemmShapes{h.count, T, h.K, h.R, false, true, cus}, kFewTiles, kSumVariantCount, &block_time);
    const bool take_few = few_time < 0.95 * block_time;
    *time = (take_few ? few_time : block_time) + 1.5 * (h.longest - 1);
    return take_few ? few : block;
}
double gemm_sums_time(int count, const int* next, int T, const int* K, const int* R) {
    double time = 0;
    for (int i = 0; i < count; ++i)
        if (K[i] > kGemmMaxK) return 1e30;
    choose_sum_tile(sum_heads(count, next, K, R), T, &time);
    return time;
}

// y of every term that no other term's next[] names = the sum of the GEMMs along next[] (-1: the last); no input scales, the
// same R along a chain, K % 256 == 0, R % 32 == 0, next[i] > i (checked by the caller).
hipError_t gemm_onebit_sums(int dtype, int count, const int* next, const void* const* x, const uint32_t* const* tiles,
                            const void* const* s_out, const void* const* bias, void* const* y, int T, const int* K, const int* R,
                            hipStream_t stream) {
    if (count < 1 || count > kGroupMax) return hipErrorInvalidValue;
    for (int i = 0; i < count; ++i)
        if (K[i] > kGemmMaxK) return hipErrorInvalidValue;
    const SumHeads h = sum_heads(count, next, K, R);
    double time = 0;
    const int pick = choose_sum_tile(h, T, &time);
    int slot[kGroupMax];
    for (int j = 0; j < h.count; ++j) slot[h.at[j]] = j;
    for (int i = 0, free = h.count; i < count; ++i)
        if (!h.head[i]) slot[i] = free++;
    GemmSums s;
    for (int i = 0; i < kGroupMax; ++i) {
        const int q = i < count ? i : 0, to = i < count ? slot[i] : i;
        GemmArgs& a = s.g.a[to];
        a.x = x[q]; a.tiles = (const uint4*)tiles[q];
        a.s_in = nullptr; a.s_out = (const uint16_t*)s_out[q]; a.bias = (const uint16_t*)bias[q];
        a.y = y[q];
        a.T = T; a.K = K[q]; a.R = R[q];
        a.gx = tile_gx(kVariants[pick], R[q]);
        s.next[to] = i < count && next[i] >= 0 ? slot[next[i]] : -1;
    }
    int blocks = 0;
    for (int j = 0; j <= kGroupMax; ++j) {
        s.g.first[j] = blocks;
        if (j < h.count) blocks += group_blocks(s.g.a[j].gx, tile_gy(kVariants[pick], T));
    }
    return dtype == 0 ? launch_sums<0>(pick, s, blocks, stream) : launch_sums<1>(pick, s, blocks, stream);
}

int gemm_tile_size(int use, int count, const void* const* x, int T, const int* K, const int* R, bool scaled) {
    double time = 0;
    const TileVariant& v = kVariants[choose_tile(x, GemmShapes{count, T, K, R, scaled, false, device_units()}, use, &time)];
    return (32 * v.tt) << 16 | 32 * v.rt * v.wr;
}
int gemm_sums_tile_size(int count, const int* next, int T, const int* K, const int* R) {
    double time = 0;
    const TileVariant& v = kVariants[choose_sum_tile(sum_heads(count, next, K, R), T, &time)];
    return (32 * v.tt) << 16 | 32 * v.rt * v.wr;
}

int gemm_group_max() { return kGroupMax; }

}  // namespace nq
