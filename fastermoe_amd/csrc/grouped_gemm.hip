// Grouped GEMM over ragged expert segments for gfx950 (MI355X, CDNA4).
//
// One launch covers every expert: the row segments travel in the kernel
// arguments, a workgroup finds its (expert, row tile, column tile) by a binary
// search over the tile prefix, and there is no per-expert launch, no host loop
// over streams and no host synchronisation.
//
// Three products share one kernel template:
//   forward  Y[seg]  = X[seg] . W_e^T      rows ragged, contraction = in
//   dgrad    dX[seg] = dY[seg] . W_e       rows ragged, contraction = out
//   wgrad    dW_e    = dY[seg]^T . X[seg]  contraction ragged (the segment)
//
// This file holds the host side: segment tables, launch plans per product and per
// chunk and the stand-alone bias-gradient kernel that the kernel of gemm_any.hip (fp64, and fp32 with feature
// sizes that are not a multiple of 16 bytes) needs.  The MFMA
// kernel itself (tiling, LDS layouts, software pipeline, epilogues) is in
// gemm_kernel.hpp and is instantiated once per element type and product by
// gemm_inst.hip.
#include "gemm_ring.hpp"
#include "gemm_skinny.hpp"
#include "profile.hpp"

#include <algorithm>
#include <cstdlib>
#include <cstring>
#include <initializer_list>
#include <mutex>
#include <vector>

namespace fmoe {
using namespace gemm;
namespace {

// ---- bias gradient: column sums per expert segment ---------------------------------
// Thread (c, g) adds rows g, g+4, ... of column c in order; the four partial sums
// are then added in a fixed order, so the result is reproducible.
template <typename T, typename Acc>
__global__ __launch_bounds__(kThreads) void bias_grad_kernel(const T *__restrict__ gy, T *__restrict__ gb,
                                                             int64_t out_feat, const SegmentTable tab,
                                                             int accumulate_first) {
    __shared__ Acc part[4][64];
    const int ei = blockIdx.y;
    const int expert = tab.first_expert + ei;
    const int c = blockIdx.x * 64 + (threadIdx.x & 63);
    const int g = threadIdx.x >> 6;
    Acc acc = 0;
    if (c < out_feat)
        for (int r = tab.seg[ei] + g; r < tab.seg[ei + 1]; r += 4) acc += (Acc)gy[(int64_t)r * out_feat + c];
    part[g][threadIdx.x & 63] = acc;
    __syncthreads();
    if (g == 0 && c < out_feat) {
        Acc s = ((part[0][threadIdx.x] + part[1][threadIdx.x]) + part[2][threadIdx.x]) + part[3][threadIdx.x];
        T *dst = gb + (int64_t)expert * out_feat + c;
        if (accumulate_first && ei == 0) s += (Acc)*dst;
        *dst = (T)s;
    }
}

// ---- host side ---------------------------------------------------------------------------

struct Plan {
    int first, last;       // experts [first, last] covered (last < first: nothing)
    bool accumulate_first; // the first covered expert began before row_lo
};

// Row segments of experts [e0, e1] clipped to [row_lo, row_hi): seg[i] is the
// clipped start of expert e0+i, seg[n] the clipped end of expert e1.
void fill_table(SegmentTable *tab, const int64_t *counts, int e0, int e1, int64_t row_lo, int64_t row_hi,
                int block_rows) {
    auto clip = [&](int64_t r) { return r < row_lo ? row_lo : (r > row_hi ? row_hi : r); };
    int64_t start = 0;
    for (int e = 0; e < e0; ++e) start += counts[e];
    tab->n = e1 - e0 + 1;
    tab->first_expert = e0;
    int tiles = 0;
    for (int e = e0; e <= e1; ++e) {
        const int64_t end = start + counts[e];
        const int64_t lo = clip(start), hi = clip(end);
        tab->seg[e - e0] = (int32_t)lo;
        tab->seg[e - e0 + 1] = (int32_t)hi;
        tab->tile[e - e0] = tiles;
        tiles += (int)ceil_div(hi - lo, block_rows);
        start = end;
    }
    tab->tile[tab->n] = tiles;
}

// Tile of a launch.  Weight gradients of 16-bit types: 256 x 256 (one workgroup per compute unit) unless that gives too few tiles
// to occupy the chip: then 128 x 256, and when even those number fewer than two per compute unit, 128 x 128 (two workgroups per
// compute unit).  Row-ragged products: rows_16bit_tile, rows_f32_tile.  fp32 has no tiles 256 wide (128 x 128 came within 4 % of 256 x 256 where
// that was ahead); its weight gradients: f32_wgrad_tile.
// FMOE_GEMM_TILE=256x256|128x256|128x128 forces one shape (for tests and measurements; fp32 takes 128x128 for the first two); for fp32
// also 64x64, for the row-ragged products 128x128+ (one workgroup per compute unit) and, 16-bit types alone, 64x128.
struct TileShape {
    int bm, bn;
    int loaders = kLoadersCompute;
    bool many = false;   // enough 256 x 256 tiles for the persistent kernel
};
bool is_16bit(int dtype) { return dtype == FMOE_BF16 || dtype == FMOE_F16; }
bool forced_tile(int dtype, bool rows, TileShape *tile) {
    const char *e = getenv("FMOE_GEMM_TILE");
    if (!e) return false;
    const bool f32 = dtype == FMOE_F32;
    if (!strcmp(e, "256x256")) *tile = f32 ? TileShape{128, 128} : TileShape{256, 256};
    else if (!strcmp(e, "128x256")) *tile = f32 ? TileShape{128, 128} : TileShape{128, 256};
    else if (!strcmp(e, "128x128")) *tile = {128, 128, rows && is_16bit(dtype) ? kLoadersShared : kLoadersCompute};
    else if (!strcmp(e, "128x128+") && rows) *tile = {128, 128, kLoadersAlone};
    else if (!strcmp(e, "64x128") && rows && is_16bit(dtype)) *tile = {64, 128, kLoadersAlone};
    else if (!strcmp(e, "64x64") && f32) *tile = {64, 64};
    else return false;
    return true;
}

// Weight gradients in fp32 (no contraction is split): 128 x 128, or 64 x 64 where the compute unit with the most tile area then has less by
// more than the 30 % that their operands' extra reads cost.  us for 64 x 64 / 128 x 128: 8 experts of
// 576 x 512, 1600 rows: 22 / 25; 4 of 768 x 512, 25552: 197 / 258; 16 of 1472 x 704, 9893: 167 / 149; 8 of 2048 x 4096, 8192: 951 / 729.
TileShape f32_wgrad_tile(int64_t experts, int64_t out_feat, int64_t in_feat) {
    const int64_t units = device_compute_units();
    const int64_t low = ceil_div(experts * ceil_div(out_feat, 64) * ceil_div(in_feat, 64), units) * 64 * 64;
    const int64_t high = ceil_div(experts * ceil_div(out_feat, 128) * ceil_div(in_feat, 128), units) * 128 * 128;
    return 130 * low < 100 * high ? TileShape{64, 64} : TileShape{128, 128};
}

constexpr TileShape kManyTiles{256, 256, kLoadersCompute, true};
TileShape pick_tile(int64_t tiles_256) {
    if (tiles_256 >= 512) return kManyTiles;
    return tiles_256 >= 256 ? TileShape{128, 256} : TileShape{128, 128};
}

// Row-ragged products in 16 bits with fewer than 512 tiles of 256 x 256: the shape with the least time by this estimate.  A round of tiles
// that fills a share f of the chip's places takes start + slabs (alone + shared f) us, the accumulators' way out included; the last round
// may be a partial one.  The weights' way from memory comes on top, as far as the rounds do not hide it.  The constants are fitted to 300
// products of 4 to 128 experts, 90 to 14000 rows and 512 to 8192 features, a tenth of a launch's time off on average, with weights that
// change from call to call, as in a model.  (Repeated on the same ones up to 256 MB of them stay in the memory-side cache, and low tiles,
// which read them more often, look better than they are: constants fitted like that picked shapes that took 1.042 times what the best of
// the five does on 120 other products, these 1.035, and 0.90 times what 128 x 128 tiles below 256 tiles of 256 x 256 and 128 x 256 from
// there on did.) us for 64 x 128 / 128 x 128 alone / 128 x 128 shared / 128 x 256 / 256 x 256 (and 128 x 128 without loading waves): 8
// experts of 4096 -> 1024, 1024 rows: 33 / 37 / 38 / 37 / 48 (37); 16 of 768 -> 3072, 2000: 49 / 43 / 40 / 41 / 29 (37); of 3072 -> 768: 42
// / 38 / 40 / 52 / 65 (41); 8 of 2048 -> 2048, 1600: 38 / 26 / 29 / 34 / 47 (30); 8 of 1024 -> 1024, 4000: 27 / 26 / 21 / 21 / 29 (24); 12
// of 2112 -> 2112, 5000: 103 / 83 / 72 / 67 / 54 (77); 8 of 2048 -> 1024, 8192: 65 / 58 / 58 / 58 / 48 (60); 64 of 2048 -> 8192, 509: 516 /
// 397 / 399 / 377 / 429 (377).
struct RowShape {
    TileShape tile;
    int per_unit;                        // workgroups on a compute unit
    double start, alone, shared, stream; // us, us per slab, TB/s (of what the rounds do not hide)
};
constexpr RowShape kRowShapes[] = {
    {{64, 128, kLoadersAlone}, 1, 3.2, 0.18, 0.14, 6.2},     {{128, 128, kLoadersAlone}, 1, 3.4, 0.31, 0.26, 30},
    {{128, 128, kLoadersShared}, 2, 4.5, 0.25, 0.83, 17},    {{128, 256, kLoadersCompute}, 1, 4.4, 0.48, 0.45, 24},
    {{256, 256, kLoadersCompute}, 1, 7.4, 0.81, 0.50, 40},
};
template <typename RowTiles> TileShape rows_16bit_tile(RowTiles row_tiles, double weight_bytes, int64_t n_cols, int64_t contraction) {
    const double slabs = (double)ceil_div(contraction, 64);
    const int64_t units = device_compute_units();
    double best = 0;
    TileShape pick{};
    for (const RowShape &s : kRowShapes) {
        const int64_t tiles = row_tiles(s.tile.bm) * ceil_div(n_cols, s.tile.bn), places = units * s.per_unit;
        const int64_t full = tiles / places, rest = tiles % places;
        double us = (double)full * (s.start + slabs * (s.alone + s.shared));
        if (rest) {
            const TailSplit split = s.tile.bm == 64 ? TailSplit{0, 1, 0} : plan_tail_split((int)std::min<int64_t>(tiles, INT32_MAX), (int)slabs, (int)units);
            if (split.k_split > 1 && full == 0)   // (and two short kernels after it)
                us += 8 + s.start + split.split_slabs * (s.alone + s.shared * (double)(rest * split.k_split) / (double)places);
            else
                us += s.start + slabs * (s.alone + s.shared * (double)rest / (double)places);
        }
        // (a few large tiles cannot ask for the weights fast enough)
        const double share = s.tile.bn == 256 ? std::min(1.0, (double)tiles * 1.6 / (double)units) : 1.0;
        us += weight_bytes * 1e-6 / (s.stream * share);
        if (pick.bm == 0 || us < best) { best = us; pick = s.tile; }
    }
    return pick;
}

// The same for fp32 (products out of bf16 parts: Split8 in gemm_kernel.hpp; slabs of 32 elements).  A compute unit takes its m tiles
// per_unit at a time, each such round start + slabs (alone + shared m / per_unit) us long, and as long as the fullest unit has tiles; the
// parts of a tail whose contraction is shared come after them.  Fitted to 220 products of 4 to 128 experts, 64 to 32768 rows and 512 to
// 13056 features, then moved to where the shape picked is the best one most often: repeated on the same weights it takes 1.01 times what
// that does, with weights that change from call to call (120 other products) 1.02 times, 64 x 64 alone 1.18, 128 x 128 two to a unit 1.07,
// one to a unit 1.08 times.  Repeated, us for the three (and before, on the fp32 MFMA): 4 experts of 640 -> 512, 251 rows: 18 / 33 / 29; 4
// of 832 -> 3328, 547: 55 / 46 / 42; 32 of 640 -> 1344, 2635: 63 / 59 / 61; 8 of 1024 -> 512, 8192: 79 / 92 / 92 (98); 8 of 2048 -> 4096,
// 8192: 1063 / 787 / 816 (1095).
struct F32RowShape {
    TileShape tile;
    int per_unit;
    double start, alone, shared, tail, stream; // us, us per slab, us, TB/s
};
constexpr F32RowShape kF32RowShapes[] = {
    {{64, 64}, 4, 1.4, 0.32, 2.07, 0, 2.4}, {{128, 128}, 2, 4.0, 0.03, 2.47, 19, 4.4}, {{128, 128, kLoadersAlone}, 1, 4.3, 0.24, 0.96, 14, 3.3},
};
template <typename RowTiles> TileShape rows_f32_tile(RowTiles row_tiles, double weight_bytes, int64_t n_cols, int64_t contraction) {
    const int64_t slabs = ceil_div(contraction, kSlabBytes / 4), units = device_compute_units();
    double best = 0;
    TileShape pick{};
    for (const F32RowShape &s : kF32RowShapes) {
        const int64_t tiles = row_tiles(s.tile.bm) * ceil_div(n_cols, s.tile.bn);
        const TailSplit split = s.tile.bm == 64 ? TailSplit{(int)std::min<int64_t>(tiles, INT32_MAX), 1, 0}
                                                : plan_tail_split((int)std::min<int64_t>(tiles, INT32_MAX), (int)slabs, (int)units);
        const int64_t fullest = ceil_div(split.main_tiles, units), rounds = fullest / s.per_unit, rest = fullest % s.per_unit;
        auto round = [&](int64_t m) { return s.start + (double)slabs * (s.alone + s.shared * (double)m / s.per_unit); };
        double us = (double)rounds * round(s.per_unit) + (rest ? round(rest) : 0);
        if (split.k_split > 1) us += s.tail + split.split_slabs * (s.alone + s.shared / s.per_unit);
        us = std::max(us + 3, weight_bytes * 1e-6 / s.stream + 4);
        if (pick.bm == 0 || us < best) { best = us; pick = s.tile; }
    }
    return pick;
}

// The activation code the kernels see.  For results that are rounded to a 16-bit type GELU and its
// derivative come from polynomials (gemm_kernel.hpp); FMOE_GELU_ERF=1 selects the erf formula of
// the 32-bit path for them too (|error| <= 1.5e-7 instead of 4e-5 .. 1.4e-4, at about twice the
// epilogue's arithmetic).
int kernel_activation(int activation) {
    if (activation == FMOE_ACT_GELU) {
        const char *e = getenv("FMOE_GELU_ERF");
        if (e && e[0] == '1') return gemm::kActGeluErf;
    }
    return activation;
}

// ragged rows: tiles_256 counts every expert's rows rounded up to whole 256-row tiles
TileShape pick_rows_tile(const int64_t *counts, int64_t n_expert, int64_t row_lo, int64_t row_hi, int64_t n_cols,
                         int64_t contraction, int dtype) {
    TileShape forced;
    if (forced_tile(dtype, true, &forced)) return forced;
    auto row_tiles = [&](int height) {
        int64_t start = 0, tiles = 0;
        for (int64_t e = 0; e < n_expert; ++e) {
            const int64_t end = start + counts[e];
            const int64_t lo = start < row_lo ? row_lo : start, hi = end > row_hi ? row_hi : end;
            if (hi > lo) tiles += ceil_div(hi - lo, height);
            start = end;
        }
        return tiles;
    };
    const double weights = (double)row_tiles(INT32_MAX) * (double)n_cols * (double)contraction;   // (of experts with rows)
    if (dtype == FMOE_F32) return rows_f32_tile(row_tiles, weights * 4, n_cols, contraction);
    if (row_tiles(256) * ceil_div(n_cols, 256) >= 512) return kManyTiles;
    return rows_16bit_tile(row_tiles, weights * 2, n_cols, contraction);
}

// ragged rows over a device table: the host does not know the counts; rows_cap rows spread over
// the experts make about rows_cap / 256 whole tiles plus a partial one for every other expert
TileShape pick_rows_tile_estimate(int64_t rows_cap, int64_t n_expert, int64_t n_cols, int64_t contraction, int dtype) {
    TileShape forced;
    if (forced_tile(dtype, true, &forced)) return forced;
    const int64_t whole = rows_cap / 256;
    const int64_t tiles = (whole + std::min<int64_t>(n_expert, std::max<int64_t>(whole, 1)) / 2) * ceil_div(n_cols, 256);
    if (dtype != FMOE_F32 && tiles >= 512) return kManyTiles;
    // every expert that can have a row, with its share of the rows and half a tile past the whole ones
    const int64_t live = std::max<int64_t>(1, std::min(n_expert, rows_cap));
    auto row_tiles = [&](int height) {
        return (int64_t)((double)live * std::max(1.0, (double)rows_cap / ((double)live * height) + 0.5) + 0.5);
    };
    const double weights = (double)live * (double)n_cols * (double)contraction;
    return dtype == FMOE_F32 ? rows_f32_tile(row_tiles, weights * 4, n_cols, contraction) : rows_16bit_tile(row_tiles, weights * 2, n_cols, contraction);
}

// Row tiles of gemm_unaligned.hip, 64 or 128 rows high: the low ones where the high ones would leave part of the
// chip idle (two workgroups fit a unit, so 512 tiles is one round).
TileShape pick_unaligned_tile(const int64_t *counts, int64_t n_expert, int64_t row_lo, int64_t row_hi, int64_t n_cols) {
    int64_t start = 0, row_tiles = 0;
    for (int64_t e = 0; e < n_expert; ++e) {
        const int64_t end = start + counts[e];
        const int64_t lo = start < row_lo ? row_lo : start, hi = end > row_hi ? row_hi : end;
        if (hi > lo) row_tiles += ceil_div(hi - lo, 128);
        start = end;
    }
    return row_tiles * ceil_div(n_cols, 128) >= 512 ? TileShape{128, 128} : TileShape{64, 128};
}
TileShape unaligned_tile_estimate(int64_t rows_cap, int64_t n_expert, int64_t n_cols) {
    const int64_t row_tiles = rows_cap / 128 + std::min(n_expert, rows_cap) / 2;
    return row_tiles * ceil_div(n_cols, 128) >= 512 ? TileShape{128, 128} : TileShape{64, 128};
}

// weight gradient: C is [out, in] per expert
TileShape pick_wgrad_tile(int64_t n_experts_written, int64_t out_feat, int64_t in_feat, int dtype) {
    TileShape forced;
    if (forced_tile(dtype, false, &forced)) return forced;
    if (dtype == FMOE_F32) return f32_wgrad_tile(n_experts_written, out_feat, in_feat);
    return pick_tile(n_experts_written * ceil_div(out_feat, 256) * ceil_div(in_feat, 256));
}

double table_flop(const SegmentTable &tab, int64_t in_feat, int64_t out_feat) {
    return 2.0 * (double)(tab.seg[tab.n] - tab.seg[0]) * (double)in_feat * (double)out_feat;
}

int check_counts(const char *who, const int64_t *counts, int64_t n_expert, int64_t row_lo, int64_t row_hi,
                 int64_t *total) {
    FMOE_REQUIRE(counts != nullptr, "%s: expert_count_host is NULL", who);
    FMOE_REQUIRE(n_expert >= 1, "%s: n_expert=%lld", who, (long long)n_expert);
    int64_t s = 0;
    for (int64_t e = 0; e < n_expert; ++e) {
        FMOE_REQUIRE(counts[e] >= 0, "%s: expert_count[%lld]=%lld is negative", who, (long long)e,
                     (long long)counts[e]);
        s += counts[e];
    }
    if (s > (int64_t)INT32_MAX || n_expert > (int64_t)(1 << 24))
        return fail(FMOE_ELIMIT, "%s: %lld rows / %lld experts exceed the supported range", who, (long long)s,
                    (long long)n_expert);
    FMOE_REQUIRE(row_lo >= 0 && row_lo <= row_hi && row_hi <= s, "%s: row range [%lld,%lld) outside [0,%lld]", who,
                 (long long)row_lo, (long long)row_hi, (long long)s);
    *total = s;
    return FMOE_OK;
}

// experts that own at least one row of [row_lo, row_hi)
Plan plan_rows(const int64_t *counts, int64_t n_expert, int64_t row_lo, int64_t row_hi) {
    Plan p{0, -1, false};
    int64_t start = 0;
    bool any = false;
    for (int e = 0; e < (int)n_expert; ++e) {
        const int64_t end = start + counts[e];
        if (end > row_lo && start < row_hi && end > start) {
            if (!any) { p.first = e; p.accumulate_first = start < row_lo; any = true; }
            p.last = e;
        }
        start = end;
    }
    return p;
}

// experts this chunk must WRITE in a ragged-K product: those with rows in the
// chunk, plus row-less experts positioned inside it.
Plan plan_contraction(const int64_t *counts, int64_t n_expert, int64_t row_lo, int64_t row_hi, bool last_chunk) {
    Plan p{0, -1, false};
    int64_t start = 0;
    bool any = false;
    for (int e = 0; e < (int)n_expert; ++e) {
        const int64_t end = start + counts[e];
        const bool has_rows = end > start && end > row_lo && start < row_hi;
        const bool empty_here = end == start && ((start >= row_lo && start < row_hi) || (last_chunk && start == row_hi));
        if (has_rows || empty_here) {
            if (!any) { p.first = e; p.accumulate_first = has_rows && start < row_lo; any = true; }
            p.last = e;
        }
        start = end;
    }
    return p;
}

template <typename T> bool fast_ok(std::initializer_list<const void *> ptrs, std::initializer_list<int64_t> dims) {
    constexpr int CE = 16 / (int)sizeof(T);
    for (const void *p : ptrs)
        if (p && !aligned16(p)) return false;
    // a row must be a whole number of 16-byte chunks, and 256 rows must stay inside the
    // 2 GiB a buffer offset can address
    for (int64_t d : dims)
        if (d % CE != 0 || d * (int64_t)sizeof(T) > (int64_t)(1 << 22)) return false;
    return true;
}

enum Product { kFwd = 0, kDgrad = 1, kWgrad = 2 };

struct SplitBuffer {
    int device;
    hipStream_t stream;
    float *ptr;
    size_t bytes;
};
std::mutex g_split_mutex;
std::vector<SplitBuffer> g_split_buffers;
int g_compute_units[16] = {};

template <int PRODUCT>
int dispatch(GemmParams &prm, int dtype, int epi, bool fast, hipStream_t stream) {
    // Shapes off the 16-byte grid: 16-bit types in gemm_unaligned.hip, the others and double precision on the
    // element-checked kernel of gemm_any.hip.  bf16 on that one and on gemm_unaligned.hip, forward / data gradient /
    // weight gradient: 1554 rows, 12 experts of 500 x 1302: 89 / 170 / 64 and 15 / 24 / 21 us; 16 rows, 8 experts of
    // 1000 x 2001: 93 / 178 / 26 and 17 / 32 / 20; 8192 rows, 8 experts of 2047 x 4093: 3063 / 2800 / 2116 and 203 / 228 / 218.
    if (!fast && is_16bit(dtype)) return launch_mfma_unaligned(prm, dtype, PRODUCT, epi, stream);
    if (!fast || dtype == FMOE_F64) return launch_mfma_any(prm, dtype, PRODUCT, epi, stream);
    switch (dtype * 3 + PRODUCT) {
        case FMOE_BF16 * 3 + kFwd: return launch_mfma_bf16_fwd(prm, epi, stream);
        case FMOE_BF16 * 3 + kDgrad: return launch_mfma_bf16_dgrad(prm, epi, stream);
        case FMOE_BF16 * 3 + kWgrad: return launch_mfma_bf16_wgrad(prm, epi, stream);
        case FMOE_F16 * 3 + kFwd: return launch_mfma_f16_fwd(prm, epi, stream);
        case FMOE_F16 * 3 + kDgrad: return launch_mfma_f16_dgrad(prm, epi, stream);
        case FMOE_F16 * 3 + kWgrad: return launch_mfma_f16_wgrad(prm, epi, stream);
        case FMOE_F32 * 3 + kFwd: return launch_mfma_f32_fwd(prm, epi, stream);
        case FMOE_F32 * 3 + kDgrad: return launch_mfma_f32_dgrad(prm, epi, stream);
        case FMOE_F32 * 3 + kWgrad: return launch_mfma_f32_wgrad(prm, epi, stream);
    }
    return fail(FMOE_EINVAL, "unknown dtype %d", dtype);
}

// Whether a launch over a device table goes to the persistent kernel of gemm_ring.hpp: 16-bit types and enough
// tiles for 256 x 256 ones (and no tile shape forced).  There it was at least level on every product
// measured: 4 to 9 % faster at K = 4096, 7 to 14 % at K = 1024, 26 to 37 % on weight gradients of 64 to 256 rows per
// expert.  Not built for 32-bit types, whose tiles are no larger than 128 x 128.
bool use_ring(const TileShape &tile, int dtype) {
    return tile.many && is_16bit(dtype);
}

// Whether a forward launch over a device table goes to gemm_skinny.hip (no tile shape forced).  The host does not know the counts: an
// expert with more than 32 rows has its weights read again, from the caches, so the lines lie where a skewed gate loses little.
// 16-bit types: at most four rows per expert on average, or twelve where the weights make less than two rounds of 128 x 128 tiles (512 at a
// time), whose last round is then badly filled.  us on the tiles and here, weights from memory: 128 experts of 1088 x 4352, 1 row
// each: 177 / 123; 256 of 2048 x 1024, 2: 184 / 140, of 1024 x 2048: 203 / 146; 64 of 1664 x 3328, 2.7: 154 / 108; 64 of 1408 x 1408, 3.6: 59 /
// 39; 128 of 1280 x 1280, 3.5, a third of the rows one expert's: 26 / 29; 256 of 1536 x 1536, 8, a fifth of them one's: 82 / 117 (even counts at
// 8: 64 of 2048 x 8192 384 / 333, 256 of 1088 x 2176 258 / 227).  Fewer tiles: 8 of 4096 x 14336, 8 rows: 187 / 138; 8 of 14336 x 4096, 8 / 12:
// 176 / 146, 176 / 156; 12 of 512 x 1792, 12: 11.3 / 8.1; 16 of 768 x 3072, 12, at random / shares 1 / rank^1.2: 23.4 / 19.5, 24.1 / 20.5; of 3072
// x 768: 31.5 / 21.8, 34.7 / 29.1; 32 of 768 x 3072, 13, a third of them one's: 41 / 36, of 3072 x 768: 36 / 41; 32 of 1024 x 1024, 15: 19.7 / 20.1.
// What the lines cost where a gate sends all rows to one expert (weights read again per 32 rows, where one round of tiles has them once): 8 of 4096 x
// 14336, 96 rows: 39 / 89; 32 of 768 x 3072, 384: 13 / 18; 256 of 2048 x 1024, 1024: 23 / 32; 64 of 4096 x 1024, 256: 39 / 32.
// float32: at most 24 rows per expert on average, 12 of contractions from 4096 on and 32 of shorter ones where the 128 x 128 tiles would
// number less than half the compute units; as many as two passes take in all (64) whatever the contraction.  64 experts of 1216 x 1216, 1 row
// each: 105 / 44; 8 of 1792 x 6272, 1.5: 140 / 46; 32 of 1024 x 3584, 16: 194 / 102; 64 of 1280 x 1280, 14, a third of the rows one's: 116 / 82; 256
// of 1408 x 704, 24: 402 / 300; 12 of 2432 x 1216, 27: 80 / 42; 32 of 1024 x 1024, 32: 51 / 51; 8 of 2048 x 8192, 48: 225 / 232; 8 of 8192 x 2048, 24,
// at random / skewed: 190 / 119, 193 / 156.
bool use_skinny(int64_t rows_cap, int64_t n_expert, int64_t in_feat, int64_t out_feat, int dtype) {
    if ((!is_16bit(dtype) && dtype != FMOE_F32) || getenv("FMOE_GEMM_TILE")) return false;
    if (dtype == FMOE_F32) {
        if (in_feat >= 4096 && rows_cap > 64) return rows_cap <= 12 * n_expert;
        return rows_cap <= 24 * n_expert || (rows_cap <= 32 * n_expert && n_expert * ceil_div(out_feat, 128) * 2 < device_compute_units());
    }
    return rows_cap <= 4 * n_expert || (rows_cap <= 12 * n_expert && n_expert * ceil_div(out_feat, 128) < 1024);
}

// Whether the tiled kernels read the weights of a row-ragged launch over a device table past the caches (16-bit types): where the average
// expert has one row tile, so that most weights are read once.  Experts of several row tiles, whose next tile then finds nothing
// in L2, lose what that costs; the line lies where an even spread rarely makes a second tile.  us through the caches and past them, weights
// from memory, forward (the data gradients gain as much): 256 experts of 768 -> 3072, 9.5 rows each: 275 / 251; 64 of 2048 -> 1024, 30: 72 / 67; 32 of
// 3328 -> 3328, 96, a fifth of the rows one's: 204 / 183; 32 of 2048 -> 4096, 106: 164 / 152; 16 of 2560 -> 2560, 216 (tiles of 256): 80 / 73; past
// the line 128 of 1664 -> 832, 136 (tiles of 128): 136 / 151; 12 of 3328 -> 960, 264: 53 / 66; 4 of 4352 -> 1088, 320: 35 / 40.  Where all rows are
// one expert's: 128 of 2048 -> 2048, 40 on average: 53 / 65; 64 of 2048 -> 8192, 16: 37 / 40.  (The
// persistent kernel's launches have more row tiles: all their weights past the caches cost 64 experts with shares 1 / rank^1.2 of 16384 rows 7 %.)
// Weights that the memory-side cache (256 MiB) can hold together with the layer's other linear stay as they were: loads past the caches
// drop them from it, and the next product that reads them waits for memory (16 experts of 768 x 3072, 2000 rows, a training step
// after another: forward of the second linear 24.6 us, 37.9 after a data gradient that read past the caches and took no less time itself).
constexpr int64_t kHeldWeightBytes = (int64_t)128 << 20;
bool reads_weights_once(const TileShape &tile, int64_t rows_cap, int64_t n_expert, int64_t in_feat, int64_t out_feat, int dtype) {
    return is_16bit(dtype) && rows_cap * 7 <= n_expert * tile.bm * 6 && n_expert * in_feat * out_feat * 2 > kHeldWeightBytes;
}

// Whether the kernel for few rows reads the weights through the caches, of an expert with at most 32 rows too: unless the caller says that nothing
// will read them again soon, or the memory-side cache could not hold them.  A decoding step gains by it (us through the caches and past
// them: 8 experts of 1024 x 4096, 8 rows 17.3 / 14.6; 32 of 1024 x 1024, 128 rows 14.7 / 13.7; 16 of 768 x 3072, 192 rows 18.3 / 16.6), a training
// step's data gradients then wait for memory (all of its products: 16 of 768 x 3072, 192 rows 132 / 143, data gradients 42 / 54; 64 of 1024 x
// 512, 512 rows 112 / 116; 128 of 512 x 768, 512 rows 150 / 156; float32: 64 of 512 x 512, 1024 rows 126 / 134, of 512 x 1024 203 / 216).
bool caches_few_row_weights(const LinearForwardArgs &a, int64_t n_expert) {
    return !a.dev_weights_once && n_expert * a.in_feat * a.out_feat * dtype_bytes(a.dtype) <= kHeldWeightBytes;
}

// The kernel of a row-ragged launch over a device table, and the workspace it can make use of.
enum class DevKernel { kTiles, kSkinny, kRing };
struct DevRoute {
    DevKernel kernel;
    TileShape tile;
};
DevRoute forward_route(int64_t rows_cap, int64_t n_expert, int64_t in_feat, int64_t out_feat, int dtype, int epilogue,
                       int activation, bool keep_pre, bool gathers) {
    const TileShape tile = pick_rows_tile_estimate(rows_cap, n_expert, out_feat, in_feat, dtype);
    if (use_skinny(rows_cap, n_expert, in_feat, out_feat, dtype)) return {DevKernel::kSkinny, tile};
    // (what the persistent kernel is built for; the erf formula, "none" and ReLU with a saved pre-activation are rare)
    const bool ring_act = epilogue == kEpiStore || activation == FMOE_ACT_GELU || (activation == FMOE_ACT_RELU && !keep_pre);
    return {use_ring(tile, dtype) && !gathers && ring_act ? DevKernel::kRing : DevKernel::kTiles, tile};
}
DevRoute dgrad_route(int64_t rows_cap, int64_t n_expert, int64_t in_feat, int64_t out_feat, int dtype, int epilogue, int activation) {
    const TileShape tile = pick_rows_tile_estimate(rows_cap, n_expert, in_feat, out_feat, dtype);
    const bool ring_act = epilogue == kEpiStore || activation == FMOE_ACT_GELU || activation == FMOE_ACT_RELU;
    return {use_ring(tile, dtype) && ring_act ? DevKernel::kRing : DevKernel::kTiles, tile};
}
int64_t route_workspace_bytes(const DevRoute &route, int64_t contraction, int dtype) {
    const int eb = dtype_bytes(dtype);
    const int n_slabs = (int)std::min<int64_t>(ceil_div(contraction, kSlabBytes / eb), 1 << 24);
    // (contractions that the tiles would not split pay on neither kernel: 48 slabs and a tail of two tiles per XCD on the
    // persistent one take 187 us cut and not cut)
    if (route.kernel == DevKernel::kSkinny || !tail_split_possible(n_slabs)) return 0;
    const int64_t tile_bytes = (int64_t)route.tile.bm * route.tile.bn * (int64_t)sizeof(float);
    if (route.kernel == DevKernel::kRing) return ring_split_possible(n_slabs) ? ring_ws_tiles(ring_workgroups()) * tile_bytes : 0;
    // (a split never has more parts than compute units, and 64 x 64 tiles are never split)
    return route.tile.bm == 64 ? 0 : device_compute_units() * tile_bytes;
}
// the caller's workspace where it is one, else null: the launch is not split
float *route_workspace(const DevRoute &route, int64_t contraction, int dtype, void *ws, int64_t ws_bytes) {
    const int64_t need = route_workspace_bytes(route, contraction, dtype);
    return ws != nullptr && need > 0 && ws_bytes >= need && (reinterpret_cast<uintptr_t>(ws) & 15u) == 0 ? (float *)ws : nullptr;
}

template <int PRODUCT>
int dispatch_ring(const GemmParams &g, int dtype, int epi, hipStream_t stream) {
    RingParams prm{};
    prm.P = g.P; prm.Q = g.Q; prm.C = g.C; prm.bias = g.bias; prm.bias_grad = g.bias_grad; prm.aux = g.aux;
    prm.ldp = g.ldp; prm.ldq = g.ldq; prm.ldc = g.ldc;
    prm.p_expert_stride = g.p_expert_stride; prm.c_expert_stride = g.c_expert_stride; prm.bias_expert_stride = g.bias_expert_stride;
    prm.n_cols = g.n_cols; prm.n_rows = g.n_rows; prm.k_extent = g.k_extent;
    prm.tiles_n = (int)ceil_div(g.n_cols, kRingTile);
    prm.tiles_m = PRODUCT == kWgrad ? (int)ceil_div(g.n_rows, kRingTile) : 0;
    prm.dev_tab = g.dev_tab;
    prm.n_expert = g.tab.n;
    prm.dev_map_off = (int32_t)segtab::map256_off(g.tab.n);
    const int64_t order = segtab::order_off(g.dev_rows_cap, g.tab.n);
    const int64_t tiles = PRODUCT == kWgrad ? (int64_t)g.tab.n * prm.tiles_m * prm.tiles_n
                                            : segtab::cap_tiles(g.dev_rows_cap, g.tab.n, kRingTile) * prm.tiles_n;
    if (order + 4 * (int64_t)g.tab.n > (int64_t)INT32_MAX || tiles > (int64_t)INT32_MAX - 65536)
        return fail(FMOE_ELIMIT, "grouped GEMM: %lld tiles exceed the supported range", (long long)tiles);
    prm.dev_order_off = (int32_t)order;
    prm.split_ws = g.dev_split_ws;
    ProfileScope prof(g.profile_class, g.profile_work, stream);
    if (dtype == FMOE_BF16)
        return PRODUCT == kFwd ? launch_ring_bf16_fwd(prm, epi, g.activation, stream)
               : PRODUCT == kDgrad ? launch_ring_bf16_dgrad(prm, epi, g.activation, stream) : launch_ring_bf16_wgrad(prm, epi, g.activation, stream);
    return PRODUCT == kFwd ? launch_ring_f16_fwd(prm, epi, g.activation, stream)
           : PRODUCT == kDgrad ? launch_ring_f16_dgrad(prm, epi, g.activation, stream) : launch_ring_f16_wgrad(prm, epi, g.activation, stream);
}

bool is_fast(int dtype, std::initializer_list<const void *> ptrs, std::initializer_list<int64_t> dims) {
    switch (dtype) {
        case FMOE_BF16: return fast_ok<__bf16>(ptrs, dims);
        case FMOE_F16: return fast_ok<_Float16>(ptrs, dims);
        case FMOE_F32: return fast_ok<float>(ptrs, dims);
    }
    return false;
}

}  // namespace

namespace gemm {

int device_compute_units() {
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 16) return 256;
    std::lock_guard<std::mutex> lock(g_split_mutex);
    if (g_compute_units[dev] == 0) {
        int n = 0;
        if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0) n = 256;
        g_compute_units[dev] = n;
    }
    return g_compute_units[dev];
}

// One buffer per (device, stream): launches on one stream run in order, so they can share it;
// launches on different streams may overlap and get their own.
float *split_workspace(hipStream_t stream, size_t bytes) {
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) return nullptr;
    std::lock_guard<std::mutex> lock(g_split_mutex);
    for (SplitBuffer &b : g_split_buffers) {
        if (b.device != dev || b.stream != stream) continue;
        return b.bytes >= bytes ? b.ptr : nullptr;
    }
    if (g_split_buffers.size() >= 32) return nullptr;  // a process that keeps creating streams: stop splitting
    // a split launch never has more parts than compute units, each a tile of at most 256 x 256
    // floats: sized for that once, the buffer fits every later request
    int cus = 0;
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus <= 0) cus = 256;
    size_t want = (size_t)cus * 256 * 256 * sizeof(float);
    if (want < bytes) want = bytes;
    float *ptr = nullptr;
    if (hipMalloc((void **)&ptr, want) != hipSuccess) { (void)hipGetLastError(); return nullptr; }
    g_split_buffers.push_back(SplitBuffer{dev, stream, ptr, want});
    return ptr;
}

}  // namespace gemm

bool linear_forward_can_gather(const LinearForwardArgs &a) {
    if (a.dtype == FMOE_F64 || dtype_bytes(a.dtype) == 0) return false;
    if (!is_fast(a.dtype, {a.x, a.w, a.y, a.aux, a.bias}, {a.in_feat, a.out_feat})) return false;
    // (the loader divides 31-bit indices: every index that names a row must fit)
    if (a.x_index_div < 1 || a.x_index_div > (int64_t)INT32_MAX || a.x_total_rows < 0 ||
        a.x_total_rows > (int64_t)INT32_MAX / a.x_index_div)
        return false;
    return a.x_total_rows * a.in_feat * (int64_t)dtype_bytes(a.dtype) < ((int64_t)1 << 31);
}

// checks shared by the launches over a device table; fills the parts of prm that say so
int device_table_launch(const char *who, GemmParams &prm, const int32_t *dev_tab, int64_t rows_cap, int64_t n_expert,
                        bool taken) {
    FMOE_REQUIRE(taken, "%s: a launch over a device segment table needs a 16- or 32-bit float type, 16-byte aligned tensors and feature "
                       "sizes that are multiples of 16 bytes (in a layer's call 16-bit types need the type only)", who);
    FMOE_REQUIRE(n_expert >= 1 && n_expert <= (int64_t)(1 << 24) && rows_cap >= 0 && rows_cap <= (int64_t)INT32_MAX - 65536,
                 "%s: n_expert=%lld rows_cap=%lld", who, (long long)n_expert, (long long)rows_cap);
    FMOE_REQUIRE((reinterpret_cast<uintptr_t>(dev_tab) & 15u) == 0, "%s: the segment table must be 16-byte aligned", who);
    prm.dev_tab = dev_tab;
    prm.dev_rows_cap = rows_cap;
    prm.tab.n = (int32_t)n_expert;
    prm.tab.first_expert = 0;
    return FMOE_OK;
}

int64_t linear_dev_workspace_bytes(int64_t contraction, int dtype) {
    const int eb = dtype_bytes(dtype);
    if (eb == 0 || dtype == FMOE_F64 || contraction < 1) return 0;
    // the most that any launch of this contraction can use: the largest tiles, for 16-bit types also on the persistent kernel
    if (dtype == FMOE_F32) return route_workspace_bytes({DevKernel::kTiles, {128, 128}}, contraction, dtype);
    return std::max(route_workspace_bytes({DevKernel::kTiles, {256, 256}}, contraction, dtype),
                    route_workspace_bytes({DevKernel::kRing, kManyTiles}, contraction, dtype));
}

int grouped_linear_forward(const LinearForwardArgs &a, const int64_t *counts, int64_t n_expert, int64_t row_lo,
                           int64_t row_hi, hipStream_t stream) {
    if (a.dev_tab != nullptr) {
        FMOE_REQUIRE(a.in_feat >= 1 && a.out_feat >= 1 && a.in_feat < (1 << 30) && a.out_feat < (1 << 30),
                     "linear_forward: in_feat=%lld out_feat=%lld", (long long)a.in_feat, (long long)a.out_feat);
        if (a.dev_rows_cap == 0) return FMOE_OK;
        FMOE_REQUIRE(a.x && a.w && a.y, "linear_forward: NULL tensor");
        const bool fast = is_fast(a.dtype, {a.x, a.w, a.y, a.aux, a.bias}, {a.in_feat, a.out_feat});
        FMOE_REQUIRE(a.x_row_index == nullptr || linear_forward_can_gather(a),
                     "linear_forward: rows cannot be gathered in the loader for this shape");
        GemmParams prm{};
        const bool any_grid = !fast && a.dev_any_grid && is_16bit(a.dtype) && a.x_row_index == nullptr;
        if (int rc = device_table_launch("linear_forward", prm, a.dev_tab, a.dev_rows_cap, n_expert, fast || any_grid)) return rc;
        prm.activation = kernel_activation(a.activation);
        const DevRoute route = any_grid ? DevRoute{DevKernel::kTiles, unaligned_tile_estimate(a.dev_rows_cap, n_expert, a.out_feat)}
                                        : forward_route(a.dev_rows_cap, n_expert, a.in_feat, a.out_feat, a.dtype, a.epilogue, prm.activation,
                                                        a.aux != nullptr, a.x_row_index != nullptr);
        prm.block_m = route.tile.bm; prm.block_n = route.tile.bn; prm.loaders = route.tile.loaders;
        prm.weights_once = fast && reads_weights_once(route.tile, a.dev_rows_cap, n_expert, a.in_feat, a.out_feat, a.dtype);
        prm.profile_class = kProfGemmFwd; prm.profile_work = 2.0 * (double)a.dev_rows_cap * (double)a.in_feat * (double)a.out_feat;
        prm.P = a.w; prm.Q = a.x; prm.C = a.y; prm.bias = a.bias; prm.aux = a.aux;
        prm.q_row_index = a.x_row_index; set_row_index_divisor(prm, a.x_index_div); prm.q_total_rows = a.x_total_rows;
        prm.ldp = a.in_feat; prm.ldq = a.in_feat; prm.ldc = a.out_feat;
        prm.p_expert_stride = a.in_feat * a.out_feat;
        prm.bias_expert_stride = a.out_feat;
        prm.n_cols = (int)a.out_feat; prm.k_extent = (int)a.in_feat;
        if (any_grid) return dispatch<kFwd>(prm, a.dtype, a.epilogue, false, stream);
        prm.dev_split_ws = route_workspace(route, a.in_feat, a.dtype, a.dev_workspace, a.dev_workspace_bytes);
        if (route.kernel == DevKernel::kSkinny) {
            SkinnyParams sk{};
            sk.w = a.w; sk.x = a.x; sk.bias = a.bias; sk.y = a.y; sk.aux = a.aux;
            sk.dev_tab = a.dev_tab;
            sk.row_index = a.x_row_index; sk.x_total_rows = a.x_total_rows;
            sk.div_mul = prm.q_div_mul; sk.div_shift = prm.q_div_shift;
            sk.n_cols = prm.n_cols; sk.k_extent = prm.k_extent; sk.activation = prm.activation;
            sk.weights_cached = caches_few_row_weights(a, n_expert);
            ProfileScope prof(prm.profile_class, prm.profile_work, stream);
            return launch_skinny(sk, a.dtype, a.dev_rows_cap, n_expert, stream);
        }
        if (route.kernel == DevKernel::kRing) return dispatch_ring<kFwd>(prm, a.dtype, a.epilogue, stream);
        return dispatch<kFwd>(prm, a.dtype, a.epilogue, fast, stream);
    }
    int64_t total;
    if (int rc = check_counts("linear_forward", counts, n_expert, row_lo, row_hi, &total)) return rc;
    FMOE_REQUIRE(a.in_feat >= 1 && a.out_feat >= 1 && a.in_feat < (1 << 30) && a.out_feat < (1 << 30),
                 "linear_forward: in_feat=%lld out_feat=%lld", (long long)a.in_feat, (long long)a.out_feat);
    if (row_hi == row_lo) return FMOE_OK;
    FMOE_REQUIRE(a.x && a.w && a.y, "linear_forward: NULL tensor");
    const Plan plan = plan_rows(counts, n_expert, row_lo, row_hi);
    const bool fast = is_fast(a.dtype, {a.x, a.w, a.y, a.aux, a.bias}, {a.in_feat, a.out_feat});
    FMOE_REQUIRE(a.x_row_index == nullptr || linear_forward_can_gather(a),
                 "linear_forward: rows cannot be gathered in the loader for this shape");
    const TileShape tile = !fast && is_16bit(a.dtype) ? pick_unaligned_tile(counts, n_expert, row_lo, row_hi, a.out_feat)
                                                      : pick_rows_tile(counts, n_expert, row_lo, row_hi, a.out_feat, a.in_feat, a.dtype);
    for (int e0 = plan.first; e0 <= plan.last; e0 += kMaxGroupExperts) {
        const int e1 = std::min(plan.last, e0 + kMaxGroupExperts - 1);
        GemmParams prm{};
        prm.block_m = tile.bm; prm.block_n = tile.bn; prm.loaders = tile.loaders;
        fill_table(&prm.tab, counts, e0, e1, row_lo, row_hi, tile.bm);
        prm.profile_class = kProfGemmFwd; prm.profile_work = table_flop(prm.tab, a.in_feat, a.out_feat);
        prm.P = a.w; prm.Q = a.x; prm.C = a.y; prm.bias = a.bias; prm.aux = a.aux;
        prm.q_row_index = a.x_row_index; set_row_index_divisor(prm, a.x_index_div); prm.q_total_rows = a.x_total_rows;
        prm.ldp = a.in_feat; prm.ldq = a.in_feat; prm.ldc = a.out_feat;
        prm.p_expert_stride = a.in_feat * a.out_feat;
        prm.bias_expert_stride = a.out_feat;
        prm.n_cols = (int)a.out_feat; prm.k_extent = (int)a.in_feat;
        prm.activation = kernel_activation(a.activation);
        if (int rc = dispatch<kFwd>(prm, a.dtype, a.epilogue, fast, stream)) return rc;
    }
    return FMOE_OK;
}

int grouped_linear_dgrad(const LinearDgradArgs &a, const int64_t *counts, int64_t n_expert, int64_t row_lo,
                         int64_t row_hi, hipStream_t stream) {
    if (a.dev_tab != nullptr) {
        FMOE_REQUIRE(a.in_feat >= 1 && a.out_feat >= 1 && a.in_feat < (1 << 30) && a.out_feat < (1 << 30),
                     "linear_dgrad: in_feat=%lld out_feat=%lld", (long long)a.in_feat, (long long)a.out_feat);
        if (a.dev_rows_cap == 0) return FMOE_OK;
        FMOE_REQUIRE(a.gy && a.w && a.gx, "linear_dgrad: NULL tensor");
        const bool fast = is_fast(a.dtype, {a.gy, a.w, a.gx, a.aux}, {a.in_feat, a.out_feat});
        GemmParams prm{};
        const bool any_grid = !fast && a.dev_any_grid && is_16bit(a.dtype);
        if (int rc = device_table_launch("linear_dgrad", prm, a.dev_tab, a.dev_rows_cap, n_expert, fast || any_grid)) return rc;
        prm.activation = kernel_activation(a.activation);
        const DevRoute route = any_grid ? DevRoute{DevKernel::kTiles, unaligned_tile_estimate(a.dev_rows_cap, n_expert, a.in_feat)}
                                        : dgrad_route(a.dev_rows_cap, n_expert, a.in_feat, a.out_feat, a.dtype, a.epilogue, prm.activation);
        prm.block_m = route.tile.bm; prm.block_n = route.tile.bn; prm.loaders = route.tile.loaders;
        prm.weights_once = fast && reads_weights_once(route.tile, a.dev_rows_cap, n_expert, a.in_feat, a.out_feat, a.dtype);
        prm.profile_class = kProfGemmDgrad; prm.profile_work = 2.0 * (double)a.dev_rows_cap * (double)a.in_feat * (double)a.out_feat;
        prm.P = a.w; prm.Q = a.gy; prm.C = a.gx; prm.aux = const_cast<void *>(a.aux);
        prm.ldp = a.in_feat; prm.ldq = a.out_feat; prm.ldc = a.in_feat;
        prm.p_expert_stride = a.in_feat * a.out_feat;
        prm.n_cols = (int)a.in_feat; prm.k_extent = (int)a.out_feat;
        if (any_grid) return dispatch<kDgrad>(prm, a.dtype, a.epilogue, false, stream);
        prm.dev_split_ws = route_workspace(route, a.out_feat, a.dtype, a.dev_workspace, a.dev_workspace_bytes);
        if (route.kernel == DevKernel::kRing) return dispatch_ring<kDgrad>(prm, a.dtype, a.epilogue, stream);
        return dispatch<kDgrad>(prm, a.dtype, a.epilogue, fast, stream);
    }
    int64_t total;
    if (int rc = check_counts("linear_dgrad", counts, n_expert, row_lo, row_hi, &total)) return rc;
    FMOE_REQUIRE(a.in_feat >= 1 && a.out_feat >= 1 && a.in_feat < (1 << 30) && a.out_feat < (1 << 30),
                 "linear_dgrad: in_feat=%lld out_feat=%lld", (long long)a.in_feat, (long long)a.out_feat);
    if (row_hi == row_lo) return FMOE_OK;
    FMOE_REQUIRE(a.gy && a.w && a.gx, "linear_dgrad: NULL tensor");
    const Plan plan = plan_rows(counts, n_expert, row_lo, row_hi);
    const bool fast = is_fast(a.dtype, {a.gy, a.w, a.gx, a.aux}, {a.in_feat, a.out_feat});
    const TileShape tile = !fast && is_16bit(a.dtype) ? pick_unaligned_tile(counts, n_expert, row_lo, row_hi, a.in_feat)
                                                      : pick_rows_tile(counts, n_expert, row_lo, row_hi, a.in_feat, a.out_feat, a.dtype);
    for (int e0 = plan.first; e0 <= plan.last; e0 += kMaxGroupExperts) {
        const int e1 = std::min(plan.last, e0 + kMaxGroupExperts - 1);
        GemmParams prm{};
        prm.block_m = tile.bm; prm.block_n = tile.bn; prm.loaders = tile.loaders;
        fill_table(&prm.tab, counts, e0, e1, row_lo, row_hi, tile.bm);
        prm.profile_class = kProfGemmDgrad; prm.profile_work = table_flop(prm.tab, a.in_feat, a.out_feat);
        prm.P = a.w; prm.Q = a.gy; prm.C = a.gx; prm.aux = const_cast<void *>(a.aux);
        prm.ldp = a.in_feat; prm.ldq = a.out_feat; prm.ldc = a.in_feat;
        prm.p_expert_stride = a.in_feat * a.out_feat;
        prm.n_cols = (int)a.in_feat; prm.k_extent = (int)a.out_feat;
        prm.activation = kernel_activation(a.activation);
        if (int rc = dispatch<kDgrad>(prm, a.dtype, a.epilogue, fast, stream)) return rc;
    }
    return FMOE_OK;
}

int grouped_linear_wgrad(const LinearWgradArgs &a, const int64_t *counts, int64_t n_expert, int64_t row_lo,
                         int64_t row_hi, bool last_chunk, hipStream_t stream) {
    if (a.dev_tab != nullptr) {
        FMOE_REQUIRE(a.in_feat >= 1 && a.out_feat >= 1 && a.in_feat < (1 << 30) && a.out_feat < (1 << 30),
                     "linear_wgrad: in_feat=%lld out_feat=%lld", (long long)a.in_feat, (long long)a.out_feat);
        FMOE_REQUIRE(a.gw && (a.dev_rows_cap == 0 || (a.gy && a.x)), "linear_wgrad: NULL tensor");
        // (with no rows at all the pointers may be NULL: every expert's contraction is empty and nothing is read)
        const bool fast = is_fast(a.dtype, {a.gy, a.x, a.gw}, {a.in_feat, a.out_feat});
        const TileShape tile = pick_wgrad_tile(n_expert, a.out_feat, a.in_feat, a.dtype);
        GemmParams prm{};
        const bool any_grid = !fast && a.dev_any_grid && is_16bit(a.dtype);
        if (int rc = device_table_launch("linear_wgrad", prm, a.dev_tab, a.dev_rows_cap, n_expert, fast || any_grid)) return rc;
        prm.block_m = tile.bm; prm.block_n = tile.bn; prm.loaders = tile.loaders;
        prm.profile_class = kProfGemmWgrad; prm.profile_work = 2.0 * (double)a.dev_rows_cap * (double)a.in_feat * (double)a.out_feat;
        prm.P = a.x; prm.Q = a.gy; prm.C = a.gw; prm.bias_grad = a.gb;
        prm.ldp = a.in_feat; prm.ldq = a.out_feat; prm.ldc = a.in_feat;
        prm.c_expert_stride = a.in_feat * a.out_feat;
        prm.n_cols = (int)a.in_feat; prm.n_rows = (int)a.out_feat;
        prm.accumulate_first = 0;
        if (!any_grid && use_ring(tile, a.dtype)) return dispatch_ring<kWgrad>(prm, a.dtype, kEpiStore, stream);
        return dispatch<kWgrad>(prm, a.dtype, kEpiStore, fast, stream);
    }
    int64_t total;
    if (int rc = check_counts("linear_wgrad", counts, n_expert, row_lo, row_hi, &total)) return rc;
    FMOE_REQUIRE(a.in_feat >= 1 && a.out_feat >= 1 && a.in_feat < (1 << 30) && a.out_feat < (1 << 30),
                 "linear_wgrad: in_feat=%lld out_feat=%lld", (long long)a.in_feat, (long long)a.out_feat);
    FMOE_REQUIRE(a.gw && (total == 0 || (a.gy && a.x)), "linear_wgrad: NULL tensor");
    const Plan plan = plan_contraction(counts, n_expert, row_lo, row_hi, last_chunk);
    const bool fast = is_fast(a.dtype, {a.gy, a.x, a.gw}, {a.in_feat, a.out_feat});
    const TileShape tile = pick_wgrad_tile(plan.last - plan.first + 1, a.out_feat, a.in_feat, a.dtype);
    for (int e0 = plan.first; e0 <= plan.last; e0 += kMaxGroupExperts) {
        const int e1 = std::min(plan.last, e0 + kMaxGroupExperts - 1);
        GemmParams prm{};
        prm.block_m = tile.bm; prm.block_n = tile.bn; prm.loaders = tile.loaders;
        fill_table(&prm.tab, counts, e0, e1, row_lo, row_hi, tile.bm);
        prm.profile_class = kProfGemmWgrad; prm.profile_work = table_flop(prm.tab, a.in_feat, a.out_feat);
        prm.P = a.x; prm.Q = a.gy; prm.C = a.gw; prm.bias_grad = fast || is_16bit(a.dtype) ? a.gb : nullptr;
        prm.ldp = a.in_feat; prm.ldq = a.out_feat; prm.ldc = a.in_feat;
        prm.c_expert_stride = a.in_feat * a.out_feat;
        prm.n_cols = (int)a.in_feat; prm.n_rows = (int)a.out_feat;
        prm.accumulate_first = (e0 == plan.first && plan.accumulate_first) ? 1 : 0;
        if (int rc = dispatch<kWgrad>(prm, a.dtype, kEpiStore, fast, stream)) return rc;
    }
    // the 16- and 32-bit MFMA kernels fold the bias gradient into their first column tiles; gemm_any.hip does not
    if (a.gb && !fast && !is_16bit(a.dtype))
        return grouped_bias_grad(a.gy, a.gb, a.out_feat, a.dtype, counts, n_expert, row_lo, row_hi, last_chunk, stream);
    return FMOE_OK;
}

int grouped_bias_grad(const void *gy, void *gb, int64_t out_feat, int dtype, const int64_t *counts,
                      int64_t n_expert, int64_t row_lo, int64_t row_hi, bool last_chunk, hipStream_t stream) {
    int64_t total;
    if (int rc = check_counts("bias_grad", counts, n_expert, row_lo, row_hi, &total)) return rc;
    FMOE_REQUIRE(gb && (total == 0 || gy) && out_feat >= 1, "bias_grad: bad argument");
    const Plan plan = plan_contraction(counts, n_expert, row_lo, row_hi, last_chunk);
    for (int e0 = plan.first; e0 <= plan.last; e0 += kMaxGroupExperts) {
        const int e1 = std::min(plan.last, e0 + kMaxGroupExperts - 1);
        SegmentTable tab;
        fill_table(&tab, counts, e0, e1, row_lo, row_hi, 256);
        const int acc_first = (e0 == plan.first && plan.accumulate_first) ? 1 : 0;
        dim3 grid((unsigned)ceil_div(out_feat, 64), (unsigned)tab.n);
        ProfileScope prof(kProfBiasGrad, (double)(tab.seg[tab.n] - tab.seg[0]) * out_feat * dtype_bytes(dtype), stream);
        switch (dtype) {
            case FMOE_BF16: bias_grad_kernel<__bf16, float><<<grid, kThreads, 0, stream>>>((const __bf16 *)gy, (__bf16 *)gb, out_feat, tab, acc_first); break;
            case FMOE_F16: bias_grad_kernel<_Float16, float><<<grid, kThreads, 0, stream>>>((const _Float16 *)gy, (_Float16 *)gb, out_feat, tab, acc_first); break;
            case FMOE_F32: bias_grad_kernel<float, float><<<grid, kThreads, 0, stream>>>((const float *)gy, (float *)gb, out_feat, tab, acc_first); break;
            case FMOE_F64: bias_grad_kernel<double, double><<<grid, kThreads, 0, stream>>>((const double *)gy, (double *)gb, out_feat, tab, acc_first); break;
            default: return fail(FMOE_EINVAL, "bias_grad: unknown dtype %d", dtype);
        }
        FMOE_LAUNCH_CHECK();
    }
    return FMOE_OK;
}

}  // namespace fmoe

using namespace fmoe;

extern "C" int fmoe_gemm_tail_plan(int64_t total_tiles, int64_t contraction_slabs, int compute_units, int64_t *plan_host) {
    FMOE_REQUIRE(plan_host && total_tiles >= 0 && total_tiles < (int64_t)INT32_MAX && contraction_slabs >= 0 &&
                     contraction_slabs < (int64_t)INT32_MAX && compute_units >= 0,
                 "fmoe_gemm_tail_plan: bad argument");
    const gemm::TailSplit ts = gemm::plan_tail_split((int)total_tiles, (int)contraction_slabs,
                                                     compute_units > 0 ? compute_units : gemm::device_compute_units());
    plan_host[0] = ts.main_tiles;
    plan_host[1] = ts.k_split;
    plan_host[2] = ts.split_slabs;
    return FMOE_OK;
}

extern "C" int fmoe_linear_forward(const void *x, const void *w, const void *bias, void *y,
                                   const int64_t *expert_count_host, int64_t n_expert, int64_t in_feat,
                                   int64_t out_feat, int dtype, void *stream) {
    FMOE_REQUIRE(dtype_bytes(dtype) != 0, "fmoe_linear_forward: unknown dtype %d", dtype);
    int64_t total;
    if (int rc = check_counts("fmoe_linear_forward", expert_count_host, n_expert, 0, 0, &total)) return rc;
    LinearForwardArgs a{x, w, bias, y, nullptr, in_feat, out_feat, dtype, kEpiStore, FMOE_ACT_NONE};
    return grouped_linear_forward(a, expert_count_host, n_expert, 0, total, (hipStream_t)stream);
}

extern "C" int fmoe_linear_act_forward(const void *x, const void *w, const void *bias, void *pre, void *y,
                                       const int64_t *expert_count_host, int64_t n_expert, int64_t in_feat,
                                       int64_t out_feat, int dtype, int activation, void *stream) {
    FMOE_REQUIRE(dtype_bytes(dtype) != 0, "fmoe_linear_act_forward: unknown dtype %d", dtype);
    FMOE_REQUIRE(activation >= FMOE_ACT_NONE && activation <= FMOE_ACT_GELU, "fmoe_linear_act_forward: activation %d",
                 activation);
    int64_t total;
    if (int rc = check_counts("fmoe_linear_act_forward", expert_count_host, n_expert, 0, 0, &total)) return rc;
    LinearForwardArgs a{x, w, bias, y, pre, in_feat, out_feat, dtype, kEpiBiasAct, activation};
    return grouped_linear_forward(a, expert_count_host, n_expert, 0, total, (hipStream_t)stream);
}

extern "C" int fmoe_linear_dact_backward(const void *grad_y, const void *w, const void *pre, void *grad_x,
                                         const int64_t *expert_count_host, int64_t n_expert, int64_t in_feat,
                                         int64_t out_feat, int dtype, int activation, void *stream) {
    FMOE_REQUIRE(dtype_bytes(dtype) != 0, "fmoe_linear_dact_backward: unknown dtype %d", dtype);
    FMOE_REQUIRE(activation >= FMOE_ACT_NONE && activation <= FMOE_ACT_GELU,
                 "fmoe_linear_dact_backward: activation %d", activation);
    int64_t total;
    if (int rc = check_counts("fmoe_linear_dact_backward", expert_count_host, n_expert, 0, 0, &total)) return rc;
    FMOE_REQUIRE(activation == FMOE_ACT_NONE || total == 0 || pre != nullptr, "fmoe_linear_dact_backward: pre is NULL");
    const bool has_act = activation != FMOE_ACT_NONE;
    LinearDgradArgs d{grad_y, w, grad_x, has_act ? pre : nullptr, in_feat, out_feat, dtype,
                      has_act ? kEpiDAct : kEpiStore, activation};
    return grouped_linear_dgrad(d, expert_count_host, n_expert, 0, total, (hipStream_t)stream);
}

extern "C" int fmoe_linear_backward(const void *grad_y, const void *x, const void *w, void *grad_x, void *grad_w,
                                    void *grad_b, const int64_t *expert_count_host, int64_t n_expert,
                                    int64_t in_feat, int64_t out_feat, int dtype, void *stream) {
    FMOE_REQUIRE(dtype_bytes(dtype) != 0, "fmoe_linear_backward: unknown dtype %d", dtype);
    int64_t total;
    if (int rc = check_counts("fmoe_linear_backward", expert_count_host, n_expert, 0, 0, &total)) return rc;
    hipStream_t st = (hipStream_t)stream;
    if (grad_x) {
        LinearDgradArgs d{grad_y, w, grad_x, nullptr, in_feat, out_feat, dtype, kEpiStore, FMOE_ACT_NONE};
        if (int rc = grouped_linear_dgrad(d, expert_count_host, n_expert, 0, total, st)) return rc;
    }
    if (grad_w) {
        LinearWgradArgs g{grad_y, x, grad_w, grad_b, in_feat, out_feat, dtype};
        if (int rc = grouped_linear_wgrad(g, expert_count_host, n_expert, 0, total, true, st)) return rc;
    } else if (grad_b) {
        if (int rc = grouped_bias_grad(grad_y, grad_b, out_feat, dtype, expert_count_host, n_expert, 0, total, true, st))
            return rc;
    }
    return FMOE_OK;
}

// ---- the same products over a segment table in device memory ---------------------------------

extern "C" int fmoe_linear_dev_supported(int64_t in_feat, int64_t out_feat, int dtype) {
    const int eb = dtype_bytes(dtype);
    if (eb == 0 || dtype == FMOE_F64 || in_feat < 1 || out_feat < 1) return 0;
    const int64_t ce = 16 / eb;
    return (in_feat % ce == 0 && out_feat % ce == 0 && in_feat * eb <= (1 << 22) && out_feat * eb <= (1 << 22)) ? 1 : 0;
}

extern "C" int fmoe_linear_act_dev_reads_rows(int64_t rows_cap, int64_t n_expert, int64_t in_feat, int64_t out_feat, int dtype,
                                              int activation, int keep_pre) {
    if (!fmoe_linear_dev_supported(in_feat, out_feat, dtype) || rows_cap < 1 || n_expert < 1) return 0;
    const bool plain = activation == FMOE_ACT_NONE && !keep_pre;
    return forward_route(rows_cap, n_expert, in_feat, out_feat, dtype, plain ? kEpiStore : kEpiBiasAct, kernel_activation(activation),
                         keep_pre != 0, false).kernel == DevKernel::kRing ? 1 : 0;
}

extern "C" int fmoe_linear_dev_reads_rows(int64_t rows_cap, int64_t n_expert, int64_t in_feat, int64_t out_feat, int dtype) {
    return fmoe_linear_act_dev_reads_rows(rows_cap, n_expert, in_feat, out_feat, dtype, FMOE_ACT_NONE, 0);
}

extern "C" int64_t fmoe_linear_forward_dev_workspace_bytes(int64_t rows_cap, int64_t n_expert, int64_t in_feat, int64_t out_feat,
                                                           int dtype, int activation, int keep_pre, int gathers) {
    if (!fmoe_linear_dev_supported(in_feat, out_feat, dtype) || rows_cap < 1 || n_expert < 1) return 0;
    const bool plain = activation == FMOE_ACT_NONE && !keep_pre;
    return route_workspace_bytes(forward_route(rows_cap, n_expert, in_feat, out_feat, dtype, plain ? kEpiStore : kEpiBiasAct,
                                               kernel_activation(activation), keep_pre != 0, gathers != 0), in_feat, dtype);
}

extern "C" int64_t fmoe_linear_dgrad_dev_workspace_bytes(int64_t rows_cap, int64_t n_expert, int64_t in_feat, int64_t out_feat,
                                                         int dtype, int activation) {
    if (!fmoe_linear_dev_supported(in_feat, out_feat, dtype) || rows_cap < 1 || n_expert < 1) return 0;
    return route_workspace_bytes(dgrad_route(rows_cap, n_expert, in_feat, out_feat, dtype,
                                             activation == FMOE_ACT_NONE ? kEpiStore : kEpiDAct, kernel_activation(activation)),
                                 out_feat, dtype);
}

extern "C" int64_t fmoe_linear_dev_workspace_bytes(int64_t contraction, int dtype) {
    return linear_dev_workspace_bytes(contraction, dtype);
}

extern "C" int fmoe_linear_forward_dev(const void *x, const int64_t *x_row_index, int64_t x_index_div,
                                       int64_t x_total_rows, const void *w, const void *bias, void *pre, void *y,
                                       const void *segment_table, int64_t n_expert, int64_t rows_cap, int64_t in_feat,
                                       int64_t out_feat, int dtype, int activation, void *workspace,
                                       int64_t workspace_bytes, void *stream) {
    FMOE_REQUIRE(dtype_bytes(dtype) != 0, "fmoe_linear_forward_dev: unknown dtype %d", dtype);
    FMOE_REQUIRE(activation >= FMOE_ACT_NONE && activation <= FMOE_ACT_GELU, "fmoe_linear_forward_dev: activation %d",
                 activation);
    FMOE_REQUIRE(segment_table != nullptr, "fmoe_linear_forward_dev: NULL segment table");
    FMOE_REQUIRE(x_row_index == nullptr || (x_index_div >= 1 && x_total_rows >= 0),
                 "fmoe_linear_forward_dev: x_index_div=%lld x_total_rows=%lld", (long long)x_index_div, (long long)x_total_rows);
    const bool plain = activation == FMOE_ACT_NONE && pre == nullptr;
    LinearForwardArgs a{x, w, bias, y, pre, in_feat, out_feat, dtype, plain ? kEpiStore : kEpiBiasAct, activation};
    a.x_row_index = x_row_index;
    a.x_index_div = x_row_index ? x_index_div : 1;
    a.x_total_rows = x_row_index ? x_total_rows : 0;
    a.dev_tab = (const int32_t *)segment_table;
    a.dev_rows_cap = rows_cap;
    a.dev_workspace = workspace;
    a.dev_workspace_bytes = workspace_bytes;
    return grouped_linear_forward(a, nullptr, n_expert, 0, rows_cap, (hipStream_t)stream);
}

extern "C" int fmoe_linear_dgrad_dev(const void *grad_y, const void *w, const void *pre, void *grad_x,
                                     const void *segment_table, int64_t n_expert, int64_t rows_cap, int64_t in_feat,
                                     int64_t out_feat, int dtype, int activation, void *workspace,
                                     int64_t workspace_bytes, void *stream) {
    FMOE_REQUIRE(dtype_bytes(dtype) != 0, "fmoe_linear_dgrad_dev: unknown dtype %d", dtype);
    FMOE_REQUIRE(activation >= FMOE_ACT_NONE && activation <= FMOE_ACT_GELU, "fmoe_linear_dgrad_dev: activation %d",
                 activation);
    FMOE_REQUIRE(segment_table != nullptr, "fmoe_linear_dgrad_dev: NULL segment table");
    FMOE_REQUIRE(activation == FMOE_ACT_NONE || rows_cap == 0 || pre != nullptr, "fmoe_linear_dgrad_dev: pre is NULL");
    const bool has_act = activation != FMOE_ACT_NONE;
    LinearDgradArgs d{grad_y, w, grad_x, has_act ? pre : nullptr, in_feat, out_feat, dtype,
                      has_act ? kEpiDAct : kEpiStore, activation};
    d.dev_tab = (const int32_t *)segment_table;
    d.dev_rows_cap = rows_cap;
    d.dev_workspace = workspace;
    d.dev_workspace_bytes = workspace_bytes;
    return grouped_linear_dgrad(d, nullptr, n_expert, 0, rows_cap, (hipStream_t)stream);
}

extern "C" int fmoe_linear_wgrad_dev(const void *grad_y, const void *x, void *grad_w, void *grad_b,
                                     const void *segment_table, int64_t n_expert, int64_t rows_cap, int64_t in_feat,
                                     int64_t out_feat, int dtype, void *stream) {
    FMOE_REQUIRE(dtype_bytes(dtype) != 0, "fmoe_linear_wgrad_dev: unknown dtype %d", dtype);
    FMOE_REQUIRE(segment_table != nullptr, "fmoe_linear_wgrad_dev: NULL segment table");
    LinearWgradArgs g{grad_y, x, grad_w, grad_b, in_feat, out_feat, dtype};
    g.dev_tab = (const int32_t *)segment_table;
    g.dev_rows_cap = rows_cap;
    return grouped_linear_wgrad(g, nullptr, n_expert, 0, rows_cap, true, (hipStream_t)stream);
}
