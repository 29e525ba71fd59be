// Grouped GEMM over a device-resident segment table with one persistent workgroup per compute unit,
// 16-bit element types (gfx950).  Included by gemm_ring_inst.hip (one translation unit per element
// type and product) and, for the host interface, by grouped_gemm.hip.
//
// The kernel of gemm_kernel.hpp computes one 256 x 256 tile per workgroup.  With 160 KiB of LDS a compute
// unit holds one workgroup, so nothing runs there while a tile's first slabs are on their way (5 us
// from the last store of one tile to the first product of the next), and a contraction of 16 slabs
// (23 us of products) or of an expert's few rows pays for that on every tile.  Here a workgroup walks a list
// of tiles as ONE stream of slabs: the loads run two slabs ahead of the products across tile borders, so
// that while a tile is stored the next one's first slabs land.
//
// Same tile, wave layout, LDS images, swizzles and four-phase slab schedule as gemm_kernel.hpp; what differs:
//   * the epilogue is staged through the Q buffer of the slab just finished (4 KiB per wave, 16 rows
//     at a time) instead of through all of LDS, whose other buffers hold the next tile's slabs;
//   * a tile of 128 rows or fewer leaves the waves of its lower half out of the products;
//   * the tiles are dealt to the workgroups beforehand: row-ragged products in bands of row
//     tiles shared by the XCDs; the weight gradient expert by expert in descending order of their rows (the table's
//     order list), back and forth over the workgroups, so that every workgroup gets its share of long and
//     short contractions, and by cost where that leaves them uneven (ring_deal); the gradients of experts without
//     rows are filled with zeros outside the stream (ring_fill);
//   * the bias gradient is one more column of products (a block of ones times the output gradient).
#pragma once
#include "gemm_kernel.hpp"

namespace fmoe {
namespace gemm {

struct RingParams {
    const void *P;     // column operand
    const void *Q;     // row operand
    void *C;
    const void *bias;  // per expert [n_cols] or null
    void *bias_grad;   // ragged K: per expert [n_rows] column sums of Q, or null
    void *aux;         // see Epilogue
    int64_t ldp, ldq, ldc;     // leading dimensions in elements
    int64_t p_expert_stride, c_expert_stride, bias_expert_stride;
    int32_t n_cols, n_rows, k_extent, tiles_n, tiles_m;
    const int32_t *dev_tab;    // segtab layout
    int32_t dev_map_off, dev_order_off, n_expert;
    // Ragged rows: the accumulators of tiles whose contraction is shared by several workgroups (null: none is shared),
    // ring_ws_tiles() tiles of floats; ws_wgs workgroups run the launch (the number the second kernel plans with).
    float *split_ws;
    int32_t ws_wgs;
};

// A workgroup's work item: a tile, or (partial) a range of a tile's slabs.
template <typename T> struct RingTile {
    const T *P, *Q;           // at the item's first contraction element
    int64_t c_off;
    int expert, K;            // contraction elements of the item
    int p_valid, q_valid, n0, m0;
    int first_slab, ws_slot;  // partial items: place in the contraction, and where the accumulators go
    bool partial;
};

// How the tiles of one XCD are dealt to its `per` workgroups (ragged rows).  Whole rounds first; the `tail` tiles of
// a last, partial round are cut along the contraction into split_wgs equal runs of slabs, one per workgroup
// (a run may end one tile and begin the next).  Measured with 4096 columns, whole rounds and a tail of 2 / 8 / 16 / 24
// tiles per XCD, not cut and cut: 64 slabs 241 / 245 / 254 / 265 and 216 / 237 / 257 / 266 us, 128 slabs 466 / 470 /
// 487 / 523 and 401 / 429 / 475 / 520, 224 slabs 847 / 863 / 893 / 947 and 715 / 771 / 847 / 987: the accumulators' way
// through memory grows with the tail (two parts from nearly every workgroup at 24), and a short tail alone on the chip
// clocks higher.  So tails of at most half the workgroups are cut, and only where that saves 40 slabs (at 48 slabs
// a tail of 2 takes 187 us either way).  At most 8 runs to a tile.
struct RingPlan {
    int full, tail, split_wgs;   // split_wgs == 0: not cut
};
constexpr int kRingMaxParts = 8, kRingSplitSaves = 40;
__host__ __device__ inline RingPlan ring_plan(int tiles, int per, int n_slabs, bool may_split) {
    RingPlan p{tiles / per, tiles % per, 0};
    if (!may_split || p.tail == 0 || p.tail * 2 > per) return p;
    const int wgs = p.tail * kRingMaxParts < per ? p.tail * kRingMaxParts : per;
    if (n_slabs - (p.tail * n_slabs + wgs - 1) / wgs >= kRingSplitSaves) p.split_wgs = wgs;
    return p;
}
// whether any tile count makes ring_plan cut a contraction of n_slabs slabs
inline bool ring_split_possible(int n_slabs) { return n_slabs - (n_slabs + kRingMaxParts - 1) / kRingMaxParts >= kRingSplitSaves; }
// Where the part of run j that lies in tail tile i goes, in tiles of floats: from one part to the next j, i or both go up
// by one, so the parts of an XCD (`per` runs at most, over at most per / 2 tiles) fit in per + per / 2 places.
__host__ __device__ inline int ring_ws_slot(int xcd, int per, int run, int tail_tile) { return xcd * (per + per / 2) + run + tail_tile; }
inline int64_t ring_ws_tiles(int wgs) { return (int64_t)(wgs / 8 + wgs / 8 / 2) * 8; }
// the run that holds slab x of the tail's tail * n_slabs slabs; run j is [j * total / wgs, (j + 1) * total / wgs)
__device__ __forceinline__ int ring_run_of(int x, int total, int wgs) { return ((x + 1) * wgs - 1) / total; }

// tile `rem` of `tm_total` row tiles x tiles_n column tiles, in groups of kGroupM row tiles per column tile
__device__ __forceinline__ void ring_tile_coords(int rem, int tiles_n, int tm_total, int &mt, int &nt) {
    // (the compiler divides in vector registers; what depends on the quotient belongs in scalar ones)
    const int gspan = kGroupM * tiles_n;
    const int grp = __builtin_amdgcn_readfirstlane(rem / gspan);
    const int gsz = min(kGroupM, tm_total - grp * kGroupM);
    const int in_grp = rem - grp * gspan;
    nt = __builtin_amdgcn_readfirstlane(in_grp / gsz);
    mt = grp * kGroupM + (in_grp - nt * gsz);
}

// The tiles of a row-ragged launch by XCD (each has its own L2).  Bands of kRingBand row tiles go to the eight XCDs in
// equal parts, one group of kGroupM row tiles each, so that all of them sweep the same experts' columns at the same time
// and a weight slab that one of them has fetched is in the memory-side cache for the others (with a
// contiguous eighth of all row tiles per XCD each works on experts of its own: 65536 rows over 8 experts of
// 4096 x 14336, K = 14336: 5716 us, in bands 5340).  The rows past the last whole band are dealt in contiguous eighths of their tiles.
constexpr int kRingBand = 8 * kGroupM;
struct RingShare {
    int per_band, bands, rest_tiles, per_xcd;   // tiles of an XCD per band, bands, tiles past them, an XCD's share of those
    __device__ __forceinline__ RingShare(int tm_total, int tiles_n)
        : per_band(kGroupM * tiles_n), bands(tm_total / kRingBand), rest_tiles((tm_total % kRingBand) * tiles_n),
          per_xcd((rest_tiles + 7) >> 3) {}
    __device__ __forceinline__ int tiles(int xcd) const {
        return bands * per_band + max(0, min(per_xcd, rest_tiles - xcd * per_xcd));
    }
    // row tile and column tile of the XCD's tile i
    __device__ __forceinline__ void coords(int xcd, int i, int tm_total, int tiles_n, int &mt, int &nt) const {
        const int band = __builtin_amdgcn_readfirstlane(i / per_band);
        if (band < bands) {
            ring_tile_coords(i - band * per_band, tiles_n, kGroupM, mt, nt);
            mt += band * kRingBand + xcd * kGroupM;
        } else {
            ring_tile_coords(xcd * per_xcd + i - bands * per_band, tiles_n, tm_total - bands * kRingBand, mt, nt);
            mt += bands * kRingBand;
        }
    }
};

constexpr int kRingThreads = 512, kRingWaves = 8;
constexpr int kRingTile = 256;
constexpr int kRingSlab = kRingTile * kSlabBytes;   // 32 KiB
constexpr int kRingPBufs = 3, kRingQBase = kRingPBufs * kRingSlab;
constexpr int kRingLds = (kRingPBufs + 2) * kRingSlab;
typedef int ring_i32x4 __attribute__((ext_vector_type(4)));

// How the tiles of a weight gradient are dealt: `rounds` back-and-forth rounds over all workgroups, then the `count` tiles from
// `first` on (rounds == 0: rounds alone).
struct RingDeal {
    int rounds, first, count;
};
constexpr int kDealTileCost = 3;   // what a tile costs beside its slabs, in slabs (its epilogue, 4 to 5 us)
constexpr int kDealSpread = 16;    // slabs by which the first round's tiles have to differ: planning takes 5 to 8 us, four or five slabs
constexpr int kDealRounds = 8;     // most rounds before the rest is dealt by cost
constexpr int kDealExperts = 1024, kDealGroups = 512;   // most experts and workgroups it is planned for
__device__ __forceinline__ int ring_tile_cost(int rows) { return max(1, (rows + 63) >> 6) + kDealTileCost; }
// tile of a back-and-forth round
__device__ __forceinline__ int ring_zigzag(int round, int grid, int w) { return round * grid + ((round & 1) ? grid - 1 - w : w); }
struct DealLds {
    int cost[kDealExperts], pre[kDealExperts + 1];     // per expert of the order list, and its exclusive prefix
    int wave_sum[8], round_max[kDealRounds + 1][8];    // (the last: all rounds)
    int64_t wave_room[8], room[kDealGroups + 1];       // exclusive prefix of what the workgroups are below the mean
};

// Rounds alone give every workgroup as many tiles as any other, and where some experts have much more rows than the rest and
// few tiles (fewer than there are workgroups, so that the first round mixes long tiles with short ones) the workgroups with the
// long ones finish last.  There the first rounds, as many as make the longest list shortest, are followed by runs of
// the remaining tiles cut by cost, for each workgroup as long as its rounds are below the mean.  us with one workgroup
// per tile / rounds alone / this: 64 experts of 1456 x 1256, 12926 rows by a Zipf law: 143 / 157 / 133; 16 of 1472 x 2944,
// 75724: 651 / 776 / 632; 128 of 640 x 2560, 14719: 193 / 207 / 181; 32 of 544 x 8040, all 39094 rows in one: 773 / 889 / 773.
// Every workgroup plans the whole launch from the table, with the same numbers.  Simulated over sizes and
// routings, the longest list is 1.05 times the mean (or the longest tile) on average; 1.15 with rounds alone, 1.03 if
// every tile went to the least loaded workgroup.
__device__ __forceinline__ RingDeal ring_deal(const RingParams &prm, int n, int tiles_per_expert, int total, int grid, int w, DealLds &lds) {
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;   // (n: experts with rows)
    const int rounds = total / grid, rest = total - rounds * grid;
    const RingDeal rounds_alone{0, 0, 0};
    const int *order = prm.dev_tab + prm.dev_order_off;   // {expert, first row, rows, 0}
    for (int e = t; e < n; e += 512) lds.cost[e] = ring_tile_cost(order[4 * e + 2]);
    __syncthreads();
    // thread t: the prefix up to experts 2 t and 2 t + 1
    const int c0 = 2 * t < n ? lds.cost[2 * t] : 0, c1 = 2 * t + 1 < n ? lds.cost[2 * t + 1] : 0;
    int v = c0 + c1;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const int up = __shfl_up(v, off, 64);
        if (lane >= off) v += up;
    }
    if (lane == 63) lds.wave_sum[wave] = v;
    // thread t: the list of workgroup t
    int load = 0;
    for (int k = 0; k <= rounds; ++k) {
        if (t < grid && (k < rounds || ring_zigzag(k, grid, t) < total)) load += lds.cost[ring_zigzag(k, grid, t) / tiles_per_expert];
        if (k < kDealRounds || k == rounds) {
            int m = load;
#pragma unroll
            for (int off = 1; off < 64; off <<= 1) m = max(m, __shfl_xor(m, off, 64));
            if (lane == 0) {
                if (k < kDealRounds) lds.round_max[k][wave] = m;
                if (k == rounds) lds.round_max[kDealRounds][wave] = m;
            }
        }
    }
    __syncthreads();
    for (int u = 0; u < wave; ++u) v += lds.wave_sum[u];
    if (2 * t <= n) lds.pre[2 * t] = v - c0 - c1;
    if (2 * t + 1 <= n) lds.pre[2 * t + 1] = v - c1;
    if (t == 511 && n == kDealExperts) lds.pre[n] = v;
    __syncthreads();
    const int64_t all = (int64_t)lds.pre[n] * tiles_per_expert;
    const int mean = (int)((all + grid - 1) / grid);
    auto longest = [&](int k) {
        int m = 0;
#pragma unroll
        for (int u = 0; u < 8; ++u) m = max(m, lds.round_max[k][u]);
        return m;
    };
    int best = INT32_MAX, k_best = 0;
    for (int k = 1; k <= kDealRounds && k * grid < total; ++k) {
        const int est = max(longest(k - 1), mean + lds.cost[k * grid / tiles_per_expert] / 2);
        if (est < best) {
            best = est;
            k_best = k;
        }
    }
    // (by a sixteenth at least: runs by cost share less of their operands than rounds do)
    if (k_best == 0 || (int64_t)longest(kDealRounds) * 16 <= (int64_t)best * 17) return rounds_alone;
    // what each workgroup is below the mean after k_best rounds, and its prefix
    int64_t room = 0;
    if (t < grid) {
        int have = 0;
        for (int k = 0; k < k_best; ++k) have += lds.cost[ring_zigzag(k, grid, t) / tiles_per_expert];
        room = max(0, mean - have);
    }
    int64_t r = room;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const int64_t up = __shfl_up((long long)r, off, 64);
        if (lane >= off) r += up;
    }
    if (lane == 63) lds.wave_room[wave] = r;
    __syncthreads();
    for (int u = 0; u < wave; ++u) r += lds.wave_room[u];
    lds.room[t + 1] = r;
    if (t == 0) lds.room[0] = 0;
    __syncthreads();
    const int n0 = k_best * grid;
    const int64_t base = (int64_t)lds.pre[n0 / tiles_per_expert] * tiles_per_expert +
                         (int64_t)lds.cost[n0 / tiles_per_expert] * (n0 % tiles_per_expert);
    const int64_t total_room = lds.room[grid], left = all - base;
    const double scale = (double)left / (double)total_room;
    // the first tile whose middle lies at or past the cost that belongs to `room` (the same number on both sides of a border)
    auto first_tile = [&](int64_t room_before) {
        const int64_t at = base + (room_before == total_room ? left : (int64_t)((double)room_before * scale));
        int lo = 0, hi = n;   // pre[lo] <= at / tiles_per_expert < pre[hi]
        while (hi - lo > 1) {
            const int mid = (lo + hi) >> 1;
            if ((int64_t)lds.pre[mid] * tiles_per_expert <= at) lo = mid; else hi = mid;
        }
        const int c = lds.cost[lo];
        const int64_t past = 2 * at - c - 2 * (int64_t)lds.pre[lo] * tiles_per_expert;
        const int64_t i = past <= 0 ? 0 : (past + 2 * c - 1) / (2 * c);
        return max(n0, lo * tiles_per_expert + (int)min(i, (int64_t)tiles_per_expert));
    };
    const int first = first_tile(lds.room[w]), end = w == grid - 1 ? total : first_tile(lds.room[w + 1]);
    return RingDeal{k_best, first, max(0, end - first)};
}

// Experts of the order list whose weight gradients are dealt as tiles: those with rows, or all (see ring_fill).
__device__ __forceinline__ int ring_live(const RingParams &prm, int grid) {
    const int live = prm.dev_tab[segtab::kLive], tpe = prm.tiles_m * prm.tiles_n;
    const bool whole = prm.n_rows % kRingTile == 0 && prm.n_cols % kRingTile == 0;
    const bool nearly = 16 * (int64_t)prm.n_rows * prm.n_cols >= 15 * (int64_t)tpe * kRingTile * kRingTile;
    return nearly && (4 * live > prm.n_expert || (whole && prm.n_expert * tpe >= 16 * grid)) ? prm.n_expert : live;
}

// Weight and bias gradients of the other experts, those of the order list from ring_live() on: zeros, 128 KiB at a time over all
// workgroups.  As a tile such a piece would cost what a tile with a slab does, 5 us, however little of it has to be stored.  Waiting
// for the stores of a piece together keeps the memory's queues short.  us with one workgroup per tile / as tiles / like this:
// 5 rows over 128 experts of 96 x 3264: 22 / 35 / 17; 8 over 12 of 1248 x 2144: 15 / 20 / 15; 100 over 128 of 2000 x 2000:
// 292 / 265 / 192; 7 over 32 of 1024 x 4096: 35 / 43 / 39.  Where tiles are (nearly) full they stay tiles if most experts have rows,
// which leaves little to fill (64 over 16 of 1000 x 4000: 30 / 29 / 31), or if they are full and many, which go out through LDS as
// fast (100 over 128 of 2048 x 2048: 178 / 179 / 187).
template <typename T> __device__ __forceinline__ void ring_fill(const RingParams &prm, int place) {
    constexpr int kStores = 16, kPieceVecs = kStores * kRingThreads;
    const int t = threadIdx.x, grid = gridDim.x, n_live = ring_live(prm, grid);
    const int64_t vecs = prm.c_expert_stride / 8;   // (an expert's gradient is dense, and both of its sizes are multiples of 8)
    const int pieces = (int)((vecs + kPieceVecs - 1) / kPieceVecs);
    const int total = (prm.n_expert - n_live) * pieces;   // (pieces of 128 KiB in memory, or one per expert: an int holds them)
    // (the pieces go on where the tiles ended, so that workgroups with a tile less begin)
    const int dealt = (int)((int64_t)n_live * prm.tiles_m * prm.tiles_n % grid);
    for (int q = place >= dealt ? place - dealt : place + grid - dealt; q < total; q += grid) {
        const int i = q / pieces;
        const int64_t v0 = (int64_t)(q - i * pieces) * kPieceVecs, expert = prm.dev_tab[prm.dev_order_off + 4 * (n_live + i)];
        u32x4 *dst = (u32x4 *)((T *)prm.C + expert * prm.c_expert_stride);
#pragma unroll
        for (int j = 0; j < kStores; ++j) {
            const int64_t v = v0 + j * kRingThreads + t;
            if (v < vecs) dst[v] = u32x4{0, 0, 0, 0};
        }
        if (v0 == 0 && prm.bias_grad != nullptr)
            for (int r = t; r < prm.n_rows; r += kRingThreads) ((T *)prm.bias_grad)[expert * prm.n_rows + r] = (T)0.f;
        __builtin_amdgcn_s_waitcnt(0x0f70);   // vmcnt(0)
        __syncthreads();
    }
}

// acc[x][y][i] is C(row 64 wm + 16 y + lb, column 128 wn + 16 x + 4 hq + i).  Sixteen rows at a time go
// through 4 KiB of LDS (16-byte chunk c of row r at c ^ r) and out as whole 256-byte row pieces.
// (NY block rows, from block row y0 of the wave's 64 rows on: acc[x][y] is block row y0 + y.)
template <typename T, int EPI, int ACT, bool AUX, bool BIAS_GRAD, int NY>
__device__ __forceinline__ void ring_epilogue(const RingParams &prm, const RingTile<T> &tl, const f32x4 (&acc)[8][NY],
                                              const f32x4 (&bacc)[BIAS_GRAD ? 4 : 1], unsigned char *stg, int lane, int wm, int wn,
                                              int y0) {
#if defined(__HIP_DEVICE_COMPILE__)
    constexpr int CE = 8, MB = 16, TI = 8;
    constexpr uint32_t kOutOfRange = 0x80000000u;
    constexpr int kRsrcFlags = 0x00020000;   // raw buffer, 32-bit data format
    // (opaque per tile: its addresses would otherwise be kept in registers across the slab loop)
    int el = lane;
    asm volatile("" : "+v"(el));
    const int lb = el & 15, hq = el >> 4;
    T *Cb = (T *)prm.C + tl.c_off;
    T *aux = (T *)prm.aux + tl.c_off;
    const int io_r = hq, io_c = lb;
    const uint32_t col_off = wn * 128 + io_c * CE < tl.p_valid ? (uint32_t)((wn * 128 + io_c * CE) * 2) : kOutOfRange;
    // byte offset of this lane's 16 bytes in row i * 4 + io_r of block row y (past the end outside the tile)
    auto io_offset = [&](int y, int i) -> uint32_t {
        const int row = 64 * wm + (y0 + y) * MB + i * 4 + io_r;
        const uint32_t off = row < tl.q_valid ? (uint32_t)((int64_t)row * prm.ldc * 2) + col_off : kOutOfRange;
        return off | (col_off & kOutOfRange);
    };
    auto wave_sync = [&]() {
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
        __builtin_amdgcn_wave_barrier();
    };
    // product with the activation's derivative: the saved pre-activations come in as the results go out, whole row
    // pieces through the staging area, one block row ahead of the one that is worked on
    constexpr bool kDAct = EPI == kEpiDAct;
    const __amdgpu_buffer_rsrc_t aux_rs = __builtin_amdgcn_make_buffer_rsrc(aux, 0, (int)kOutOfRange, kRsrcFlags);
    u32x4 ahead[kDAct ? 4 : 1];
    auto request_aux = [&](int y) {
#pragma unroll
        for (int i = 0; i < 4; ++i) ahead[i] = __builtin_amdgcn_raw_buffer_load_b128(aux_rs, (int)io_offset(y, i), 0, 0);
    };
    if constexpr (kDAct) request_aux(0);
    constexpr int kKinds = EPI == kEpiBiasAct ? 2 : 1;
    // Weight gradients go out nontemporally: nothing of the launch reads them, and where they make up most of its traffic they
    // would push the operands out of L2.  64 experts of 8192 x 2048, 64 / 256 / 512 rows each: 395 / 692 / 1067 us through the
    // caches, 347 / 678 / 1036 like this.  (The other products' results are the next launch's input; nontemporal they gain nothing.)
    constexpr int kPolicy = BIAS_GRAD ? 2 : 0;
#pragma unroll
    for (int kind = kKinds - 1; kind >= 0; --kind) {   // 1: the pre-activation, 0: the result
        if (kind == 1 && !AUX) continue;
        const __amdgpu_buffer_rsrc_t rs =
            __builtin_amdgcn_make_buffer_rsrc(EPI == kEpiBiasAct && kind == 1 ? aux : Cb, 0, (int)kOutOfRange, kRsrcFlags);
#pragma unroll
        for (int y = 0; y < NY; ++y) {
            if constexpr (kDAct) {
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const int r = i * 4 + io_r;
                    *(u32x4 *)(stg + r * 256 + ((io_c ^ r) << 4)) = ahead[i];
                }
                if (y + 1 < NY) request_aux(y + 1);
                wave_sync();
            }
#pragma unroll
            for (int x = 0; x < TI; ++x) {
                unsigned char *at = stg + lb * 256 + (((2 * x + (hq >> 1)) ^ lb) << 4) + (hq & 1) * 8;
                alignas(8) T res[4], pre[4];
                if constexpr (kDAct) *(u32x2 *)pre = *(const u32x2 *)at;
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    float v = acc[x][y][i];
                    if (EPI == kEpiBiasAct && kind == 0) v = apply_act<true>(v, ACT);
                    if constexpr (kDAct) v *= act_grad<true>((float)pre[i], ACT);
                    res[i] = (T)v;
                }
                *(u32x2 *)at = *(const u32x2 *)res;
            }
            wave_sync();
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int r = i * 4 + io_r;
                const u32x4 v = *(const u32x4 *)(stg + r * 256 + ((io_c ^ r) << 4));
                __builtin_amdgcn_raw_buffer_store_b128(v, rs, (int)io_offset(y, i), 0, kPolicy);
            }
            wave_sync();
        }
    }
    if constexpr (BIAS_GRAD) {
        if (prm.bias_grad != nullptr && tl.n0 == 0 && wn == 0 && hq == 0) {
#pragma unroll
            for (int y = 0; y < NY; ++y) {
                const int row = 64 * wm + (y0 + y) * MB + lb;
                if (row < tl.q_valid) ((T *)prm.bias_grad)[(int64_t)tl.expert * prm.n_rows + tl.m0 + row] = (T)bacc[y][0];
            }
        }
    }
#endif
}

template <typename T, int PSHAPE, int QSHAPE, int RAGGED, int EPI, int ACT, bool AUX>
__global__ __launch_bounds__(kRingThreads) void grouped_gemm_ring_kernel(const RingParams prm) {
#if defined(__HIP_DEVICE_COMPILE__)  // the host pass only needs the launch stub
    static_assert(sizeof(T) == 2, "16-bit element types");
    static_assert(EPI != kEpiDAct || PSHAPE == kMC, "the data gradient alone multiplies by the activation's derivative");
    constexpr int CE = 8, BKE = 64, MB = 16;
    constexpr int TI = 8, TJ = 4;            // MFMA blocks per wave: 128 columns, 64 rows
    constexpr int PF = 4;                    // block columns per phase
    constexpr int NLOAD = 8;                 // 16-byte loads per loading thread, slab and operand
    constexpr uint32_t kOutOfRange = 0x80000000u;
    constexpr int kRsrcFlags = 0x00020000;   // raw buffer, 32-bit data format
    constexpr bool kForward = RAGGED == kRaggedRows && PSHAPE == kKC;
    // With both operands [contraction][row] a fragment is two transposing reads, and a phase issues its loads, reads and
    // products in four interleaved quarters (weight gradient, 256 rows per expert: 415 -> 370 us); otherwise a
    // phase's loads go out together ahead of its reads (forward, K = 14336: 1590 -> 1389 us).
    constexpr bool kQuarters = PSHAPE == kMC && QSHAPE == kMC;
    constexpr bool kWithBiasGrad = RAGGED == kRaggedK && QSHAPE == kMC;

    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    typedef ring_i32x4 i32x4;
    typedef const int32_t __attribute__((address_space(4))) *DevTab;    // read-only, uniform: scalar loads
    typedef const i32x4 __attribute__((address_space(4))) *DevTab4;
    const DevTab dtab = (DevTab)(uintptr_t)prm.dev_tab;

    const int t = threadIdx.x, lane = t & 63;
    const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int lb = lane & 15, hq = lane >> 4;        // row inside an MFMA block, contraction chunk inside a step
    const int wm = wave >> 1, wn = wave & 1;
    const uint32_t lds_base = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) void *)smem;

    // -- this workgroup's list of items -----------------------------------------------------
    const int xcd = blockIdx.x & 7, slot = blockIdx.x >> 3, per = gridDim.x >> 3;
    auto uniform = [](int v) { return __builtin_amdgcn_readfirstlane(v); };
    int n_items, tm_total;
    RingPlan plan{0, 0, 0};
    int run_lo = 0, run_hi = 0, k_slabs = 0;   // this workgroup's run of the tail's slabs
    RingDeal deal{INT32_MAX, 0, 0};
    int deal_w = xcd * per + slot;   // this workgroup's place in the dealing
    if (RAGGED == kRaggedRows) {
        tm_total = dtab[segtab::kTiles256];
        k_slabs = (prm.k_extent + BKE - 1) / BKE;
        plan = ring_plan(RingShare(tm_total, prm.tiles_n).tiles(xcd), per, k_slabs, prm.split_ws != nullptr);
        plan.full = uniform(plan.full);
        plan.tail = uniform(plan.tail);
        plan.split_wgs = uniform(plan.split_wgs);
        n_items = plan.full;
        if (plan.split_wgs == 0) {
            n_items += slot < plan.tail ? 1 : 0;
        } else if (slot < plan.split_wgs) {
            const int slabs = plan.tail * k_slabs;
            run_lo = uniform(slot * slabs / plan.split_wgs);
            run_hi = uniform((slot + 1) * slabs / plan.split_wgs);
            n_items += uniform((run_hi - 1) / k_slabs - run_lo / k_slabs + 1);
        }
    } else {
        tm_total = prm.tiles_m;
        const int grid = gridDim.x, n_live = uniform(ring_live(prm, grid));
        const int total = n_live * prm.tiles_m * prm.tiles_n;
        const int rounds = uniform(total / grid), rest = total - rounds * grid;
        n_items = rounds + (ring_zigzag(rounds, grid, deal_w) < total ? 1 : 0);
        if (rounds > 0 && rest + rounds > 1 && n_live <= kDealExperts && grid <= kDealGroups) {
            // rounds alone are level enough where the first one is: its first and last tile differ by less than a sixteenth of a list
            const int tpe = prm.tiles_m * prm.tiles_n;
            const int longest = ring_tile_cost(dtab[prm.dev_order_off + 2]);
            const int shortest = ring_tile_cost(dtab[prm.dev_order_off + 4 * uniform((grid - 1) / tpe) + 2]);
            const float list = ((float)dtab[segtab::kRows] / 64.f + (kDealTileCost + 0.5f) * (float)n_live) * (float)tpe / (float)grid;
            const int spread = uniform(longest) - uniform(shortest);
            if (spread >= kDealSpread && (float)spread * 16.f > list) {
                // (eight tiles in a row to an XCD, which share operands, then the next: as many long tiles as one expert has
                // would otherwise all be on one or two XCDs, the 64 experts of ring_deal's comment 150 us instead of 133)
                const int chunk = per % 8 == 0 ? 8 : 1;
                const int w = (slot / chunk) * (8 * chunk) + xcd * chunk + slot % chunk;
                const RingDeal planned = ring_deal(prm, n_live, tpe, total, grid, w, *(DealLds *)smem);
                if (uniform(planned.rounds) > 0) {
                    deal_w = uniform(w);
                    deal.rounds = uniform(planned.rounds);
                    deal.first = uniform(planned.first);
                    n_items = deal.rounds + uniform(planned.count);
                }
                __syncthreads();   // the plan is read; the slabs take its place
            }
        }
    }
    if (n_items == 0) {
        if constexpr (RAGGED == kRaggedK) ring_fill<T>(prm, xcd * per + slot);
        return;
    }

    typedef RingTile<T> Tile;
    auto decode = [&](int r) {
        Tile tl;
        int rem, ei = 0, mt, nt;
        ring_i32x4 entry;
        tl.partial = false;
        tl.first_slab = tl.ws_slot = 0;
        if (RAGGED == kRaggedRows) {
            tl.K = prm.k_extent;
            if (plan.split_wgs == 0 || r < plan.full) {
                rem = r * per + slot;
            } else {
                const int first_tile = uniform(run_lo / k_slabs), tail_tile = first_tile + (r - plan.full);
                const int lo = max(run_lo, tail_tile * k_slabs), hi = min(run_hi, (tail_tile + 1) * k_slabs);
                rem = plan.full * per + tail_tile;
                tl.partial = hi - lo < k_slabs;
                tl.first_slab = lo - tail_tile * k_slabs;
                tl.K = min(prm.k_extent - tl.first_slab * BKE, (hi - lo) * BKE);
                tl.ws_slot = ring_ws_slot(xcd, per, slot, tail_tile);
            }
        } else {
            const int grid = gridDim.x, tpe = prm.tiles_m * prm.tiles_n;
            const int q = r < deal.rounds ? ring_zigzag(r, grid, deal_w) : deal.first + (r - deal.rounds);
            ei = uniform(q / tpe);
            rem = q - ei * tpe;
            entry = *(DevTab4)(dtab + prm.dev_order_off + 4 * ei);
        }
        if (RAGGED == kRaggedRows) RingShare(tm_total, prm.tiles_n).coords(xcd, rem, tm_total, prm.tiles_n, mt, nt);
        else ring_tile_coords(rem, prm.tiles_n, tm_total, mt, nt);
        tl.n0 = nt * kRingTile;
        tl.p_valid = min(kRingTile, prm.n_cols - tl.n0);
        if (RAGGED == kRaggedRows) {
            entry = *(DevTab4)(dtab + prm.dev_map_off + 4 * mt);   // {expert, first row, rows}
            const int64_t k0 = (int64_t)tl.first_slab * BKE;
            tl.m0 = 0;
            tl.q_valid = entry[2];
            tl.Q = (const T *)prm.Q + (int64_t)entry[1] * prm.ldq + k0;   // (the row operand is [row][contraction])
            const T *Pe = (const T *)prm.P + (int64_t)entry[0] * prm.p_expert_stride;
            tl.P = (PSHAPE == kKC) ? Pe + (int64_t)tl.n0 * prm.ldp + k0 : Pe + tl.n0 + k0 * prm.ldp;
            tl.c_off = (int64_t)entry[1] * prm.ldc + tl.n0;
        } else {                                                   // {expert, first row, rows}, the whole expert
            tl.m0 = mt * kRingTile;
            tl.q_valid = min(kRingTile, prm.n_rows - tl.m0);
            tl.K = entry[2];
            tl.Q = (const T *)prm.Q + (int64_t)entry[1] * prm.ldq + tl.m0;
            tl.P = (const T *)prm.P + (int64_t)entry[1] * prm.ldp + tl.n0;
            tl.c_off = (int64_t)entry[0] * prm.c_expert_stride + (int64_t)tl.m0 * prm.ldc + tl.n0;
        }
        tl.expert = entry[0];
        return tl;
    };

    // -- global -> LDS ------------------------------------------------------------------------
    // As in gemm_kernel.hpp: loading thread t < 256 fetches, in pass it, the chunk that belongs in LDS slot
    // it * 256 + t.  A pass is 32 rows (KC) or 8 contraction rows (MC) below the one before, so a running offset
    // (MC: two, the swizzle alternates) gives all eight; rows outside the tile lie past the end of the buffer
    // resource and read as zero.  The resources move along the contraction from slab to slab.
    const uint32_t p_step = (uint32_t)((PSHAPE == kKC ? 32 : 16) * prm.ldp * 2);
    const uint32_t q_step = (uint32_t)((QSHAPE == kKC ? 32 : 16) * prm.ldq * 2);
    // contraction element of a KC chunk of this thread
    const int kc_elem = ((t & 7) ^ swz((t >> 3) & 31)) * CE;
    struct Operand {
        uint32_t lo, hi, bytes;      // buffer resource of the slab to be requested next
        uint32_t off0, off1;         // this thread's offsets at a slab's start (even, odd passes) ...
        uint32_t run0, run1;         // ... and of its next pass
    };
    Operand ldp_op, ldq_op;
    int ld_index = 0, ld_left = 0;   // the load cursor: tile of the list, contraction elements from the next slab on

    auto set_slab_bytes = [&](auto shape_tag, Operand &op, int64_t ld) {
        if (decltype(shape_tag)::value == kMC) op.bytes = (uint32_t)(max(0, min(ld_left, BKE)) * (int)(ld * 2));
    };
    auto set_operand = [&](auto shape_tag, Operand &op, const T *origin, int64_t ld, int valid, int k0) {
        const uint64_t a = (uint64_t)origin;
        op.lo = (uint32_t)a;
        op.hi = (uint32_t)(a >> 32) & 0xffffu;
        if (decltype(shape_tag)::value == kKC) {
            const int r = (t >> 3) & 31;
            op.off0 = op.off1 = (uint32_t)(r * (int)(ld * 2) + (((t & 7) ^ swz(r)) << 4));
            op.bytes = valid > 0 ? (uint32_t)(valid * (int)(ld * 2) - k0 * 2) : 0u;   // to the end of the last row
        } else {
            const int kk = (t >> 5) & 7;
            const int c0 = (t & 31) ^ ((kk & 3) << 2), c1 = c0 ^ 2;
            op.off0 = c0 * CE < valid ? (uint32_t)(kk * (int)(ld * 2) + c0 * 16) : kOutOfRange;
            op.off1 = c1 * CE < valid ? (uint32_t)((kk + 8) * (int)(ld * 2) + c1 * 16) : kOutOfRange;
        }
        set_slab_bytes(shape_tag, op, ld);
    };
    typedef std::integral_constant<int, PSHAPE> PTag;
    typedef std::integral_constant<int, QSHAPE> QTag;
    auto load_tile = [&](int r) {
        ld_index = r;
        const bool live = r < n_items;   // past the last tile everything reads as zero
        const Tile tl = decode(live ? r : 0);
        ld_left = live ? tl.K : 0;
        set_operand(PTag{}, ldp_op, tl.P, prm.ldp, live ? tl.p_valid : 0, tl.first_slab * BKE);
        set_operand(QTag{}, ldq_op, tl.Q, prm.ldq, live ? tl.q_valid : 0, tl.first_slab * BKE);
    };
    auto move_operand = [&](auto shape_tag, Operand &op, int64_t ld) {
        const uint32_t by = decltype(shape_tag)::value == kKC ? (uint32_t)kSlabBytes : (uint32_t)(BKE * (int)(ld * 2));
        const uint64_t a = (((uint64_t)op.hi << 32) | op.lo) + by;
        op.lo = (uint32_t)a;
        op.hi = (uint32_t)(a >> 32);
        if (decltype(shape_tag)::value == kKC) op.bytes -= kSlabBytes;
        else set_slab_bytes(shape_tag, op, ld);
    };
    auto advance = [&]() {
        ld_left -= BKE;
        if (ld_left <= 0) {
            load_tile(ld_index + 1);
        } else {
            move_operand(PTag{}, ldp_op, prm.ldp);
            move_operand(QTag{}, ldq_op, prm.ldq);
        }
    };
    // The pass `it` of the operand's slab into the 32 KiB at lds_off.  go (scalar, only where cond says so): skipped by
    // a branch the compiler does not see, so that the products around it stay one basic block.
    auto issue = [&](auto shape_tag, Operand &op, uint32_t step, uint32_t lds_off, auto it_tag, auto cond, bool go) {
        constexpr int SHAPE = decltype(shape_tag)::value, it = decltype(it_tag)::value;
        if (it == 0) {
            // sign bit set where a KC chunk starts past the end of the contraction
            const uint32_t past = SHAPE == kKC ? ((uint32_t)(ld_left - 1 - kc_elem) & kOutOfRange) : 0u;
            op.run0 = op.off0 | past;
            op.run1 = op.off1;
        }
        constexpr bool odd = SHAPE == kMC && (it & 1);
        const uint32_t voff = odd ? op.run1 : op.run0;
        i32x4 rs;
        rs[0] = __builtin_amdgcn_readfirstlane((int)op.lo);
        rs[1] = __builtin_amdgcn_readfirstlane((int)op.hi);
        rs[2] = __builtin_amdgcn_readfirstlane((int)op.bytes);
        rs[3] = kRsrcFlags;
        const uint32_t lds_addr = __builtin_amdgcn_readfirstlane(lds_base + lds_off + wave * 1024);
        if constexpr (decltype(cond)::value) {
            asm volatile("s_cmp_eq_u32 %3, 0\n\ts_cbranch_scc1 .Lring_skip%=\n\t"
                         "s_add_u32 m0, %0, %4\n\tbuffer_load_dwordx4 %1, %2, 0 offen lds\n.Lring_skip%=:"
                         :
                         : "s"(lds_addr), "v"(voff), "s"(rs), "s"(__builtin_amdgcn_readfirstlane((int)go)), "n"(it * 4096)
                         : "memory", "m0", "scc");
        } else {
            asm volatile("s_add_u32 m0, %0, %3\n\tbuffer_load_dwordx4 %1, %2, 0 offen lds"
                         :
                         : "s"(lds_addr), "v"(voff), "s"(rs), "n"(it * 4096)
                         : "memory", "m0", "scc");
        }
        if (odd) op.run1 += step; else op.run0 += step;
    };
    auto issue_p = [&](int buf, auto it_tag) {
        issue(PTag{}, ldp_op, p_step, (uint32_t)(buf * kRingSlab), it_tag, std::false_type{}, true);
    };
    auto issue_q = [&](int buf, auto it_tag, bool go) {
        issue(QTag{}, ldq_op, q_step, (uint32_t)(kRingQBase + buf * kRingSlab), it_tag, std::true_type{}, go);
    };
    auto issue_slab = [&](auto issue_one) {   // the eight passes of one operand
        issue_one(std::integral_constant<int, 0>{});
        issue_one(std::integral_constant<int, 1>{});
        issue_one(std::integral_constant<int, 2>{});
        issue_one(std::integral_constant<int, 3>{});
        issue_one(std::integral_constant<int, 4>{});
        issue_one(std::integral_constant<int, 5>{});
        issue_one(std::integral_constant<int, 6>{});
        issue_one(std::integral_constant<int, 7>{});
    };

    // -- fragments ------------------------------------------------------------------------------
    // KC: block j's fragment of step ks at (16 j + lb) * 128 + (((4 ks + hq) ^ swz(lb)) << 4);
    // MC: two transposing reads at A ^ (j << 5) + ks * 16384 (+ 2048), with A from the lane (see gemm_kernel.hpp).
    auto frag_base = [&](int shape, int first_block) -> uint32_t {
        if (shape == kKC) return (uint32_t)((first_block * 16 + lb) * kSlabBytes + ((hq ^ swz(lb)) << 4));
        const int s16 = lane & 15, kb = hq * 8 + (s16 >> 2);
        const int sw = ((s16 >> 2) << 2) | ((hq & 1) << 1);
        return (uint32_t)((((sw | ((s16 >> 1) & 1)) << 4) | ((s16 & 1) * 8) | (kb * 512)) ^ (first_block << 5));
    };
    const uint32_t p_frag = frag_base(PSHAPE, wn * TI), q_frag = frag_base(QSHAPE, wm * TJ);
    auto frag = [&](int shape, uint32_t base, uint32_t buf_off, int j, int ks) -> u32x4 {
        if (shape == kKC) return *(const u32x4 *)(smem + buf_off + (base ^ (ks << 6)) + j * 2048);
        typedef short s16x4 __attribute__((ext_vector_type(4)));
        typedef __attribute__((address_space(3))) s16x4 *lds_s16x4_ptr;
        const unsigned char *at = smem + buf_off + (base ^ (uint32_t)(j << 5)) + ks * 16384;
        const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4_ptr)(at));
        const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4_ptr)(at + 2048));
        const u32x2 l2 = __builtin_bit_cast(u32x2, lo), h2 = __builtin_bit_cast(u32x2, hi);
        return u32x4{l2[0], l2[1], h2[0], h2[1]};
    };

    f32x4 acc[TI][TJ];
    f32x4 bacc[kWithBiasGrad ? TJ : 1];
    u32x4 pf[2][PF], qf[2][TJ];
    constexpr int kPReads = PSHAPE == kMC ? 2 : 1, kQReads = QSHAPE == kMC ? 2 : 1;   // LDS reads per fragment
    // A quarter of the fragments of phase ph (the row operand's first: the phase's first product needs all of them)
    auto read_part = [&](int ph, int part, uint32_t p_buf, uint32_t q_buf) {
        if ((ph & 1) == 0) {
            if (part < 2) {
#pragma unroll
                for (int y = 2 * part; y < 2 * part + 2; ++y) qf[ph >> 1][y] = frag(QSHAPE, q_frag, q_buf, y, ph >> 1);
            } else {
#pragma unroll
                for (int x = 2 * part - 4; x < 2 * part - 2; ++x) pf[0][x] = frag(PSHAPE, p_frag, p_buf, x, ph >> 1);
            }
        } else {
            pf[1][part] = frag(PSHAPE, p_frag, p_buf, PF + part, ph >> 1);
        }
    };
    auto read_phase0 = [&](uint32_t p_buf, uint32_t q_buf) {
#pragma unroll
        for (int part = 0; part < 4; ++part) read_part(0, part, p_buf, q_buf);
    };
    // Phase ph in four steps of four products, each with a quarter of the next phase's fragment reads and,
    // in the loading waves, a quarter of the phase's loads: a loading wave is blocked some 35 ns per
    // direct-to-LDS load, which its own products then follow one load at a time.
    auto phase = [&](int ph, uint32_t p_buf, uint32_t q_buf, auto load_step) {
        const int next = (ph + 1) & 3;
        if constexpr (kQuarters) {
            auto quarter = [&](auto x_tag) {
                constexpr int x = decltype(x_tag)::value;
                load_step(x_tag);
                read_part(next, x, p_buf, q_buf);
#pragma unroll
                for (int y = 0; y < TJ; ++y) Elem<T>::mma(acc[(ph & 1) * PF + x][y], pf[ph & 1][x], qf[ph >> 1][y]);
                const int reads = (next & 1) ? kPReads : (x < 2 ? 2 * kQReads : 2 * kPReads);
#pragma unroll
                for (int i = 0; i < TJ; ++i) {
                    if (i < reads) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);   // LDS read
                    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);                 // MFMA
                }
                __builtin_amdgcn_sched_barrier(0);
            };
            quarter(std::integral_constant<int, 0>{});
            quarter(std::integral_constant<int, 1>{});
            quarter(std::integral_constant<int, 2>{});
            quarter(std::integral_constant<int, 3>{});
        } else {
            load_step(std::integral_constant<int, 0>{});
            load_step(std::integral_constant<int, 1>{});
            load_step(std::integral_constant<int, 2>{});
            load_step(std::integral_constant<int, 3>{});
#pragma unroll
            for (int x = 0; x < PF; ++x) read_part(next, x, p_buf, q_buf);
#pragma unroll
            for (int x = 0; x < PF; ++x)
#pragma unroll
                for (int y = 0; y < TJ; ++y) Elem<T>::mma(acc[(ph & 1) * PF + x][y], pf[ph & 1][x], qf[ph >> 1][y]);
            const int reads = PF * kPReads + ((next & 1) == 0 ? TJ * kQReads : 0);
#pragma unroll
            for (int i = 0; i < PF * TJ; ++i) {
                if (i < reads) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    // The accumulators start from the bias (forward product; columns past the tile and a missing bias read as zero).
    // It is requested before the epilogue of the tile before, so that nothing waits for it.
    u32x2 bias_raw[kForward ? TI : 1];
    auto request_bias = [&](const Tile &tl) {
        if constexpr (kForward) {
            const bool has = prm.bias != nullptr && tl.first_slab == 0;
            const T *bias = has ? (const T *)prm.bias + (int64_t)tl.expert * prm.bias_expert_stride + tl.n0 : nullptr;
            const __amdgpu_buffer_rsrc_t bias_rs =
                __builtin_amdgcn_make_buffer_rsrc(const_cast<T *>(bias), 0, has ? tl.p_valid * 2 : 0, kRsrcFlags);
#pragma unroll
            for (int x = 0; x < TI; ++x)
                bias_raw[x] = __builtin_amdgcn_raw_buffer_load_b64(bias_rs, (wn * 128 + x * MB + hq * 4) * 2, 0, 0);
        }
    };
    auto init_acc = [&]() {
#pragma unroll
        for (int x = 0; x < TI; ++x) {
            f32x4 start = {0.f, 0.f, 0.f, 0.f};
            if constexpr (kForward) {
                alignas(8) T bv[4];
                *(u32x2 *)bv = bias_raw[x];
#pragma unroll
                for (int i = 0; i < 4; ++i) start[i] = (float)bv[i];
            }
#pragma unroll
            for (int y = 0; y < TJ; ++y) acc[x][y] = start;
            // (kept here: sunk towards its uses, the conversion leaves the bias pending on the way into the slab
            // loop as far as the compiler can tell, and its wait there drains the slab loads too)
            if constexpr (kForward) {
#pragma unroll
                for (int y = 0; y < TJ; ++y) asm volatile("" : "+v"(acc[x][y]));
            }
        }
        if (kWithBiasGrad) {
#pragma unroll
            for (int y = 0; y < TJ; ++y) bacc[y] = f32x4{0.f, 0.f, 0.f, 0.f};
        }
    };
    const uint32_t one2 = std::is_same<T, __bf16>::value ? 0x3f803f80u : 0x3c003c00u;
    const u32x4 ones = {one2, one2, one2, one2};
    auto wait_loads = [&](auto n_tag) {   // at most n of this wave's memory operations outstanding, all LDS reads done
        constexpr int n = decltype(n_tag)::value;
        __builtin_amdgcn_s_waitcnt(0x0070 | (n & 15) | ((n >> 4) << 14));
    };
    auto slab_barrier = [&]() {
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
    };

    // -- the stream of slabs --------------------------------------------------------------------------
    auto run = [&](auto loads_tag) {
        constexpr bool kLoads = decltype(loads_tag)::value;
        constexpr int kNoWait = 63;
        if constexpr (kLoads) {
            load_tile(0);
            issue_slab([&](auto it) { issue_p(0, it); });
            issue_slab([&](auto it) { issue_q(0, it, true); });
            advance();
            issue_slab([&](auto it) { issue_p(1, it); });
            issue_slab([&](auto it) { issue_q(1, it, true); });
            advance();
        }
        __builtin_amdgcn_sched_barrier(0);
        wait_loads(std::integral_constant<int, kLoads ? 2 * NLOAD : kNoWait>{});
        slab_barrier();
        read_phase0(0, kRingQBase);
        __builtin_amdgcn_sched_barrier(0);

        int pc = 0, qc = 0;   // LDS buffers of the current slab
        Tile tile = decode(0);
        request_bias(tile);
        init_acc();
        for (int tile_index = 0;;) {
            const int n_slabs = tile.K > BKE ? (tile.K + BKE - 1) / BKE : 1;
            const bool active = 64 * wm < tile.q_valid;
            const bool want_bias = kWithBiasGrad && prm.bias_grad != nullptr && tile.n0 == 0 && wn == 0;
            const Tile next = decode(tile_index + 1 < n_items ? tile_index + 1 : tile_index);
            if (kLoads || active) {
                for (int left = n_slabs; left > 0; --left) {
                    const int pn = pc == kRingPBufs - 1 ? 0 : pc + 1;
                    const int pl = pn == kRingPBufs - 1 ? 0 : pn + 1;   // receives slab s + 2
                    const uint32_t sp = pc * kRingSlab, sq = kRingQBase + qc * kRingSlab;
                    auto bias_products = [&](int ks) {
                        if constexpr (kWithBiasGrad) {
                            if (want_bias) {
#pragma unroll
                                for (int y = 0; y < TJ; ++y) Elem<T>::mma(bacc[y], ones, qf[ks][y]);
                            }
                            __builtin_amdgcn_sched_barrier(0);
                        }
                    };
                    phase(0, sp, sq, [](auto) {});
                    bias_products(0);
                    phase(1, sp, sq, [&](auto x) { if constexpr (kLoads) issue_p(pl, x); });
                    phase(2, sp, sq, [&](auto x) { if constexpr (kLoads) issue_p(pl, std::integral_constant<int, 4 + x()>{}); });
                    bias_products(1);
                    wait_loads(std::integral_constant<int, kLoads ? NLOAD : kNoWait>{});   // all but the P loads of slab s + 2
                    slab_barrier();
                    // (the Q buffer of a tile's last slab stages its epilogue first)
                    const uint32_t np = pn * kRingSlab, nq = kRingQBase + (qc ^ 1) * kRingSlab;
                    phase(3, np, nq, [&](auto x) {
                        if constexpr (kLoads) {
                            issue_q(qc, std::integral_constant<int, 2 * x()>{}, left > 1);
                            issue_q(qc, std::integral_constant<int, 2 * x() + 1>{}, left > 1);
                        }
                    });
                    if constexpr (kLoads) {
                        if (left > 1) advance();
                    }
                    pc = pn;
                    qc ^= 1;
                }
                const uint32_t stage = kRingQBase + (qc ^ 1) * kRingSlab;
                request_bias(next);
                if (RAGGED == kRaggedRows && tile.partial) {
                    // part of a tile: the accumulators go to memory as [16 bytes of a lane][thread]
                    f32x4 *dst = (f32x4 *)prm.split_ws + (int64_t)tile.ws_slot * (kRingTile * kRingTile / 4) + t;
#pragma unroll
                    for (int x = 0; x < TI; ++x)
#pragma unroll
                        for (int y = 0; y < TJ; ++y) __builtin_nontemporal_store(acc[x][y], dst + (x * TJ + y) * kRingThreads);
                } else {
                    ring_epilogue<T, EPI, ACT, AUX, kWithBiasGrad, TJ>(prm, tile, acc, bacc, smem + stage + wave * 4096, lane, wm, wn, 0);
                }
            } else {
                for (int left = n_slabs; left > 0; --left) {
                    slab_barrier();
                    pc = pc == kRingPBufs - 1 ? 0 : pc + 1;
                    qc ^= 1;
                }
                read_phase0(pc * kRingSlab, kRingQBase + qc * kRingSlab);
                request_bias(next);
            }
            init_acc();   // (before the exit, so that no path into the slab loop has the bias still pending)
            if (++tile_index == n_items) break;
            tile = next;
            __builtin_amdgcn_s_waitcnt(0xc07f);   // lgkmcnt(0): this wave is done with its staging area
            slab_barrier();
            if constexpr (kLoads) {
                issue_slab([&](auto it) { issue_q(qc ^ 1, it, true); });
                advance();
            }
        }
        // loads requested past the last slab (they read zeros) land before the workgroup gives its LDS back
        wait_loads(std::integral_constant<int, 0>{});
    };
    if (wave < kLoadWaves) run(std::true_type{});
    else run(std::false_type{});
    if constexpr (RAGGED == kRaggedK) ring_fill<T>(prm, xcd * per + slot);
#endif  // __HIP_DEVICE_COMPILE__
}

// Second kernel of a launch with a shared tail: one wave per workgroup stands in for one block row (16 rows, 128 columns)
// of a wave of a tail tile, adds up the tile's parts in ascending order of their slabs (a fixed order) and runs the
// epilogue.  The parts of a tile are read by 32 waves with 32 loads each in flight (by 8 waves with 4 loads it took 47 us
// for 16 tiles of 8 parts).  Grid: 8 XCDs x the most tail tiles of an XCD x 32; a wave whose tile does not
// exist or was not shared leaves at once.
template <typename T, int EPI, int ACT, bool AUX>
__global__ __launch_bounds__(64) void ring_combine_kernel(const RingParams prm) {
#if defined(__HIP_DEVICE_COMPILE__)
    __shared__ __attribute__((aligned(16))) unsigned char stage[4096];
    typedef const int32_t __attribute__((address_space(4))) *DevTab;
    typedef const ring_i32x4 __attribute__((address_space(4))) *DevTab4;
    const DevTab dtab = (DevTab)(uintptr_t)prm.dev_tab;
    const int per = prm.ws_wgs >> 3;
    const int y = blockIdx.x & 3, wave = (blockIdx.x >> 2) & 7, unit = blockIdx.x >> 5, xcd = unit & 7, tail_tile = unit >> 3;
    const int tm_total = dtab[segtab::kTiles256];
    const RingShare share(tm_total, prm.tiles_n);
    const int k_slabs = (prm.k_extent + 63) / 64;
    const RingPlan plan = ring_plan(share.tiles(xcd), per, k_slabs, true);
    if (plan.split_wgs == 0 || tail_tile >= plan.tail) return;
    const int slabs = plan.tail * k_slabs, wgs = plan.split_wgs;
    const int first = ring_run_of(tail_tile * k_slabs, slabs, wgs), last = ring_run_of((tail_tile + 1) * k_slabs - 1, slabs, wgs);
    if (first == last) return;   // one workgroup had all of it and has stored it
    RingTile<T> tl{};
    int mt, nt;
    share.coords(xcd, plan.full * per + tail_tile, tm_total, prm.tiles_n, mt, nt);
    const ring_i32x4 entry = *(DevTab4)(dtab + prm.dev_map_off + 4 * mt);
    tl.n0 = nt * kRingTile;
    tl.p_valid = min(kRingTile, prm.n_cols - tl.n0);
    tl.q_valid = entry[2];
    tl.expert = entry[0];
    tl.c_off = (int64_t)entry[1] * prm.ldc + tl.n0;
    if (64 * (wave >> 1) + 16 * y >= tl.q_valid) return;
    constexpr int kBatch = 4;   // parts read at a time
    f32x4 acc[8][1];
    for (int j0 = first; j0 <= last; j0 += kBatch) {
        f32x4 v[kBatch][8];
#pragma unroll
        for (int b = 0; b < kBatch; ++b) {
            // (the same for the workgroup; with the last part read again in a missing one's place the launch took 21.4 us instead of
            // 14.8 on 64 tail tiles of 4 columns of tiles, K = 4096)
            if (j0 + b > last) continue;
            const f32x4 *src = (const f32x4 *)prm.split_ws + (int64_t)ring_ws_slot(xcd, per, j0 + b, tail_tile) * (kRingTile * kRingTile / 4) +
                               wave * 64 + threadIdx.x;
#pragma unroll
            for (int x = 0; x < 8; ++x) v[b][x] = __builtin_nontemporal_load(src + (x * 4 + y) * kRingThreads);
        }
#pragma unroll
        for (int b = 0; b < kBatch; ++b)
#pragma unroll
            for (int x = 0; x < 8; ++x) {
                if (b == 0) acc[x][0] = j0 == first ? v[0][x] : acc[x][0] + v[0][x];
                else if (j0 + b <= last) acc[x][0] += v[b][x];
            }
    }
    const f32x4 none[1] = {};
    ring_epilogue<T, EPI, ACT, AUX, false, 1>(prm, tl, acc, none, stage, threadIdx.x, wave >> 1, wave & 1, y);
#endif
}

// one workgroup per compute unit, the same number for each of the eight XCDs
inline int ring_workgroups() { return std::max(8, device_compute_units() / 8 * 8); }

template <typename T, int PS, int QS, int RG, int EPI, int ACT = FMOE_ACT_NONE, bool AUX = false>
int launch_ring(RingParams prm, hipStream_t stream) {
    static std::atomic<int> configured[16];
    auto kern = grouped_gemm_ring_kernel<T, PS, QS, RG, EPI, ACT, AUX>;
    int dev = 0;
    FMOE_HIP_CHECK(hipGetDevice(&dev));
    FMOE_REQUIRE(dev >= 0 && dev < 16, "device index %d out of range", dev);
    if (configured[dev].load(std::memory_order_acquire) != 1) {
        const hipError_t err = hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, kRingLds);
        configured[dev].store(err == hipSuccess ? 1 : 2, std::memory_order_release);
        FMOE_HIP_CHECK(err);
    }
    const int grid = ring_workgroups();
    prm.ws_wgs = grid;
    if (RG != kRaggedRows || !ring_split_possible((prm.k_extent + 63) / 64)) prm.split_ws = nullptr;
    kern<<<grid, kRingThreads, kRingLds, stream>>>(prm);
    FMOE_LAUNCH_CHECK();
    if constexpr (RG == kRaggedRows) {
        if (prm.split_ws != nullptr) {
            // (a tail that is cut has at most half as many tiles as an XCD has workgroups)
            ring_combine_kernel<T, EPI, ACT, AUX><<<grid / 16 * 256, 64, 0, stream>>>(prm);
            FMOE_LAUNCH_CHECK();
        }
    }
    return FMOE_OK;
}

}  // namespace gemm

// Defined in gemm_ring_inst.hip, once per element type and product.
#define FMOE_DECLARE_RING(NAME) int NAME(const gemm::RingParams &prm, int epilogue, int activation, hipStream_t stream)
FMOE_DECLARE_RING(launch_ring_bf16_fwd);
FMOE_DECLARE_RING(launch_ring_bf16_dgrad);
FMOE_DECLARE_RING(launch_ring_bf16_wgrad);
FMOE_DECLARE_RING(launch_ring_f16_fwd);
FMOE_DECLARE_RING(launch_ring_f16_dgrad);
FMOE_DECLARE_RING(launch_ring_f16_wgrad);

}  // namespace fmoe
