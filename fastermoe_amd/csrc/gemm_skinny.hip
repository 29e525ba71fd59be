// Grouped forward product Y[seg_e] = act(X[seg_e] . W_e^T + b_e) for few rows per expert, 16- and 32-bit types over a device
// segment table (gfx950): decoding steps, where every weight is read once and meets a handful of rows.
//
// Bound by the weights' way from memory, so nothing is staged: weights and rows go from memory (the rows: L2, where they stay) straight
// into the registers of 16 x 16 x 32 MFMAs (float32: 16 x 16 x 4).  A workgroup of four waves has up to 64 columns of up to 32 rows of one expert; the
// waves take the contraction in turns of one unit, with the next unit's loads under way before the products of the current one, and add
// up their accumulators through LDS in a fixed order.  What it takes to come near the 6.9 TB/s that such loads alone reach here
// (8 experts of 4096 x 14336, 8 rows each: 189 us before, 137 now; of 14336 x 4096: 187 and 142):
//   * a load takes whole lines, 128 bytes of eight rows, and leaves no trace in the caches (6.2 TB/s through them; 64 bytes of
//     sixteen rows, the operands' own shape, read nontemporally: 5.5, as the halves of a line are fetched apart), unless the weights are read
//     again soon and fit there (weights_cached);
//   * the rows' loads, which take as many places in a unit's queue of loads as the weights' do, serve two or four blocks of 16 columns
//     (one block: 362 us for that layer's pass, without the rows' loads 300);
//   * each workgroup of an expert begins its contraction one unit further on than the one before, so that they don't all ask the same
//     channels for the same columns at once (162 -> 142 us for 14336 x 4096); where it begins is its expert's and its columns' own, so that a row's
//     sum, in the order of the units from there on, does not depend on how many rows other experts have;
//   * the compiler may not move a unit's loads behind the products of the one before, which left none in flight at their end.
// Where it is used, and what it measured: use_skinny() in grouped_gemm.hip.
#include "gemm_skinny.hpp"
#include "segment_table.hpp"

namespace fmoe {
namespace gemm {
namespace {

constexpr int kSkWaves = 4, kSkThreads = 64 * kSkWaves;
constexpr int kSkRows = 32;   // rows of a pass

// one 16 x 16 block over 64 bytes of contraction; acc as for the 16 x 16 x 32 form
template <typename T> __device__ __forceinline__ void mma_step(f32x4 &acc, const u32x4 &w, const u32x4 &x) { Elem<T>::mma(acc, w, x); }
template <> __device__ __forceinline__ void mma_step<float>(f32x4 &acc, const u32x4 &w, const u32x4 &x) {
    // product j takes element j of every lane's four: contraction elements j, 4 + j, 8 + j and 12 + j of the step
#pragma unroll
    for (int j = 0; j < 4; ++j)
        acc = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(w[j]), __uint_as_float(x[j]), acc, 0, 0, 0);
}

// Two loads of 128 bytes of rows 0 to 7 and 8 to 15 (lane: row lane % 8, bit 3: half of the line) become the operands of two
// steps (lane: row lane % 16, chunk lane / 16 of the step's 64 bytes): the lanes with bit 3 set give the first load's second chunks
// for the second load's first.
__device__ __forceinline__ void pair_to_steps(u32x4 &a, u32x4 &b) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const uint32_t lo = a[i], hi = b[i];   // (row_ror 8 within 16 lanes, written to the upper or to the lower eight)
        a[i] = __builtin_amdgcn_update_dpp(lo, hi, 0x128, 0xf, 0xc, false);
        b[i] = __builtin_amdgcn_update_dpp(hi, lo, 0x128, 0xf, 0x3, false);
    }
}

// COL_BLOCKS: blocks of 16 columns of a workgroup.  APART: an expert's groups of rows have workgroups of their own (see launch)
template <typename T, int COL_BLOCKS, bool APART>
__global__ __launch_bounds__(kSkThreads, COL_BLOCKS == 4 ? 3 : 4) void grouped_gemm_skinny_kernel(const SkinnyParams prm) {
#if defined(__HIP_DEVICE_COMPILE__)  // the host pass only needs the launch stub
    constexpr int EB = (int)sizeof(T), CE = 16 / EB, kLine = 128 / EB;    // elements per lane's load and per line
    typedef std::conditional_t<sizeof(T) == 2, u32x2, u32x4> Vec4;        // four elements
    constexpr uint32_t kOutOfRange = 0x80000000u;
    constexpr int kRsrcFlags = 0x00020000;   // raw buffer, 32-bit data format
    typedef const int32_t __attribute__((address_space(4))) *DevTab;    // read-only, uniform: scalar loads
    typedef int i32x4 __attribute__((ext_vector_type(4)));
    typedef const i32x4 __attribute__((address_space(4))) *DevTab4;
    __shared__ f32x4 part[kSkWaves - 1][COL_BLOCKS * 2][64];

    const DevTab dtab = (DevTab)(uintptr_t)prm.dev_tab;
    int place = __builtin_amdgcn_readfirstlane(blockIdx.x / prm.tiles_n);
    const int tile_n = blockIdx.x - place * prm.tiles_n, n0 = tile_n * (COL_BLOCKS * 16), K = prm.k_extent;
    const DevTab4 order = (DevTab4)(dtab + prm.order_off);   // {expert, first row, rows}: of an expert, or (not APART) of a tile of at most 128 rows
    const int live = dtab[APART ? segtab::kLive : segtab::kTiles128];
    int r0 = 0;   // first row
    i32x4 entry;
    if (APART && place < prm.extra_groups) {
        // A further group of an expert with more rows than one pass takes; the experts come in descending order of their rows
        int i = 0, skip = place;
        for (;; ++i) {
            entry = order[i];   // (there is an expert 0; the ones before have more than kSkRows rows, so `i` is not past the last live one)
            const int groups = (entry[2] - 1) / kSkRows;   // (without rows: 0)
            if (groups == 0) return;
            if (skip < groups) break;
            skip -= groups;
            if (i + 1 >= live) return;
        }
        r0 = (skip + 1) * kSkRows;
    } else {
        place -= prm.extra_groups;
        entry = order[place];   // (asked for together with their number; the launch has as many places as experts can have rows, or as there can be tiles)
        asm volatile("" : "+s"(entry));
        if (place >= live) return;
    }
    const int expert = entry[0], first = entry[1], rows = entry[2];
    if (rows == 0) return;
    // where its contraction begins, by expert and columns alone: a row's sum does not depend on the rows that other experts have
    const uint32_t start = __builtin_amdgcn_readfirstlane((uint32_t)expert * (uint32_t)prm.tiles_n + (uint32_t)tile_n);
    const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int lb = lane & 15, hq = lane >> 4;
    // A load takes 128 bytes of eight rows, this lane 16 bytes of row lane % 8 (see pair_to_steps)
    const int chunk = hq | ((lane & 8) >> 1), row8 = lane & 7;

    // weights: rows past the last column lie past the end of the resource and read as zero
    const T *W = (const T *)prm.w + ((int64_t)expert * prm.n_cols + n0) * K;
    const int w_bytes = min(COL_BLOCKS * 16, prm.n_cols - n0) * K * EB;
    const __amdgpu_buffer_rsrc_t w_rs = __builtin_amdgcn_make_buffer_rsrc(const_cast<T *>(W), 0, w_bytes, kRsrcFlags);
    const uint32_t w_off = (uint32_t)(row8 * K * EB + chunk * 16), eight_rows = (uint32_t)(8 * K * EB);
    const bool gather = prm.row_index != nullptr;

    // NB blocks of 16 columns from column c0 of the workgroup on times RB blocks of 16 rows from the expert's row r0 on; a unit is LINES times
    // 128 bytes of contraction.  POLICY: of the weights' loads
    auto pass = [&](auto nb_tag, auto rb_tag, auto lines_tag, auto policy_tag, int c0, int r0) {
        constexpr int NB = decltype(nb_tag)::value, RB = decltype(rb_tag)::value, LINES = decltype(lines_tag)::value;
        constexpr int POLICY = decltype(policy_tag)::value;
        static_assert(NB * RB <= 2 * COL_BLOCKS && NB <= kSkWaves, "the waves' sums");
        struct Unit { u32x4 w[LINES][NB][2], x[LINES][RB][2]; };
        // The rows, in a resource that begins at the pass's first or at the tile's: all of an expert can be more than the 2 GiB that offsets reach (bit
        // 31 marks one as out of range), these are at most 32 or 128 of 4 MiB.  A gathered matrix is less than 2 GiB as a whole.
        const int base = APART ? r0 : 0, base_rows = APART ? min(rows - r0, 16 * RB) : rows;
        const int64_t base_at = (int64_t)first + base;
        const __amdgpu_buffer_rsrc_t x_rs = __builtin_amdgcn_make_buffer_rsrc(
            const_cast<T *>((const T *)prm.x + (gather ? (int64_t)0 : base_at * K)), 0, (int)(gather ? prm.x_total_rows : (int64_t)base_rows) * K * EB, kRsrcFlags);
        const __amdgpu_buffer_rsrc_t index_rs = __builtin_amdgcn_make_buffer_rsrc(
            const_cast<int64_t *>(gather ? prm.row_index + base_at : nullptr), 0, gather ? base_rows * 8 : 0, kRsrcFlags);
        const uint32_t w_base = w_off + (uint32_t)c0 * (uint32_t)(K * EB);
        const int n_units = (K + kLine * LINES - 1) / (kLine * LINES);
        const int turn = __builtin_amdgcn_readfirstlane((int)(start % (uint32_t)n_units));   // the unit it begins with
        // (offsets past the contraction, as of every unit past it, have the sign bit set)
        auto line_offset = [&](int unit, int l) -> uint32_t {
            const int at = unit + turn < n_units ? unit + turn : unit + turn - n_units;
            const int k = unit < n_units ? (at * LINES + l) * kLine : K;
            return (uint32_t)(k * EB) | ((uint32_t)(K - 1 - k - chunk * CE) & kOutOfRange);
        };
        auto load_w = [&](Unit &u, int unit) {
#pragma unroll
            for (int l = 0; l < LINES; ++l) {
                const uint32_t at = w_base + line_offset(unit, l);
#pragma unroll
                for (int n = 0; n < NB; ++n) {
                    u.w[l][n][0] = __builtin_amdgcn_raw_buffer_load_b128(w_rs, (int)(at + 2 * n * eight_rows), 0, POLICY);
                    u.w[l][n][1] = __builtin_amdgcn_raw_buffer_load_b128(w_rs, (int)(at + (2 * n + 1) * eight_rows), 0, POLICY);
                }
            }
        };
        Unit a, b;
        int unit = wave;
        // (asked for ahead of the first weights and waited for behind them)
        u32x2 index[RB][2];
#pragma unroll
        for (int y = 0; y < RB; ++y)
#pragma unroll
            for (int h = 0; h < 2; ++h) index[y][h] = __builtin_amdgcn_raw_buffer_load_b64(index_rs, (r0 - base + 16 * y + 8 * h + row8) * 8, 0, 0);
        load_w(a, unit);
        __builtin_amdgcn_sched_barrier(0);
        uint32_t x_off[RB][2];
#pragma unroll
        for (int y = 0; y < RB; ++y)
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const int row = r0 - base + 16 * y + 8 * h + row8;
                uint32_t src = row;
                bool valid = row < base_rows;
                if (gather) {
                    const uint32_t idx = index[y][h][0];
                    src = prm.div_shift < 0 ? idx : __umulhi(idx, prm.div_mul) >> prm.div_shift;
                    valid = valid && index[y][h][1] == 0 && idx <= (uint32_t)INT32_MAX && (int64_t)src < prm.x_total_rows;
                }
                x_off[y][h] = valid ? src * (uint32_t)(K * EB) + chunk * 16 : kOutOfRange;
            }
        f32x4 acc[NB][RB];
#pragma unroll
        for (int n = 0; n < NB; ++n)
#pragma unroll
            for (int y = 0; y < RB; ++y) acc[n][y] = f32x4{0.f, 0.f, 0.f, 0.f};
        auto load_x = [&](Unit &u, int unit) {
#pragma unroll
            for (int l = 0; l < LINES; ++l) {
                const uint32_t at = line_offset(unit, l);
#pragma unroll
                for (int y = 0; y < RB; ++y) {
#pragma unroll
                    for (int h = 0; h < 2; ++h)   // (both offsets may have the sign bit)
                        u.x[l][y][h] = __builtin_amdgcn_raw_buffer_load_b128(x_rs, (int)((x_off[y][h] + (at & ~kOutOfRange)) | (at & kOutOfRange)), 0, 0);
                }
            }
        };
        auto multiply = [&](Unit &u) {
#pragma unroll
            for (int l = 0; l < LINES; ++l) {
#pragma unroll
                for (int y = 0; y < RB; ++y) pair_to_steps(u.x[l][y][0], u.x[l][y][1]);
#pragma unroll
                for (int n = 0; n < NB; ++n) {
                    pair_to_steps(u.w[l][n][0], u.w[l][n][1]);
#pragma unroll
                    for (int s = 0; s < 2; ++s)
#pragma unroll
                        for (int y = 0; y < RB; ++y) mma_step<T>(acc[n][y], u.w[l][n][s], u.x[l][y][s]);
                }
            }
        };
        load_x(a, unit);
        while (unit < n_units) {
            load_w(b, unit + kSkWaves);
            load_x(b, unit + kSkWaves);
            __builtin_amdgcn_sched_barrier(0);   // (or the compiler moves the loads behind the products, and none are in flight at their end)
            multiply(a);
            __builtin_amdgcn_sched_barrier(0);
            unit += kSkWaves;
            if (unit >= n_units) break;
            load_w(a, unit + kSkWaves);
            load_x(a, unit + kSkWaves);
            __builtin_amdgcn_sched_barrier(0);
            multiply(b);
            __builtin_amdgcn_sched_barrier(0);
            unit += kSkWaves;
        }
        // the waves' sums in ascending order of the wave; wave n adds column block n's
        __syncthreads();   // (the pass before has read its sums)
#pragma unroll
        for (int n = 0; n < NB; ++n) {
            if (wave == n) continue;
#pragma unroll
            for (int y = 0; y < RB; ++y) part[wave - (wave > n ? 1 : 0)][n * RB + y][lane] = acc[n][y];
        }
        __syncthreads();
#pragma unroll
        for (int n = 0; n < NB; ++n) {
            if (wave != n) continue;
            // acc[n][y][i] is C(row 16 y + lb, column 16 n + 4 hq + i)
            const int col = n0 + c0 + 16 * n + 4 * hq;
            alignas(16) T b4[4] = {};
            if (prm.bias != nullptr && col < prm.n_cols)
                *(Vec4 *)b4 = *(const Vec4 *)((const T *)prm.bias + (int64_t)expert * prm.n_cols + col);
#pragma unroll
            for (int y = 0; y < RB; ++y) {
                f32x4 v = n == 0 ? acc[n][y] : part[0][n * RB + y][lane];
#pragma unroll
                for (int w = 1; w < kSkWaves; ++w) v += w == n ? acc[n][y] : part[w - (w > n ? 1 : 0)][n * RB + y][lane];
                const int row = r0 + 16 * y + lb;
                if (row >= rows || col >= prm.n_cols) continue;
                alignas(16) T pre[4], res[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const float p = v[i] + (float)b4[i];
                    pre[i] = (T)p;
                    res[i] = (T)apply_act<sizeof(T) == 2>(p, prm.activation);
                }
                const int64_t at = (int64_t)(first + row) * prm.n_cols + col;
                if (prm.aux != nullptr) *(Vec4 *)((T *)prm.aux + at) = *(const Vec4 *)pre;
                *(Vec4 *)((T *)prm.y + at) = *(const Vec4 *)res;
            }
        }
    };
    typedef std::integral_constant<int, 0> Cached;
    typedef std::integral_constant<int, 2> Nontemporal;
    typedef std::integral_constant<int, 1> One;
    typedef std::integral_constant<int, 2> Two;
    typedef std::integral_constant<int, COL_BLOCKS> All;
    typedef std::integral_constant<int, (COL_BLOCKS < 2 ? COL_BLOCKS : 2)> UpToTwo;
    // (Two units have to fit 168 registers: scratch memory costs launches that never touch it a tenth of their time.  The weights of an
    // expert with several groups are read again, from the caches.)
    if (rows <= 16) {
        const std::integral_constant<int, COL_BLOCKS == 1 ? 2 : 1> lines;
        if (prm.weights_cached) pass(All{}, One{}, lines, Cached{}, 0, 0);
        else pass(All{}, One{}, lines, Nontemporal{}, 0, 0);
        return;
    }
    auto up_to_two = [&](int c0) {
        if (rows <= kSkRows && !prm.weights_cached) {
            pass(UpToTwo{}, Two{}, One{}, Nontemporal{}, c0, 0);
        } else if constexpr (APART) {
            pass(UpToTwo{}, Two{}, One{}, Cached{}, c0, r0);
        } else {
            for (int row = 0; row < rows; row += kSkRows) pass(UpToTwo{}, Two{}, One{}, Cached{}, c0, row);
        }
    };
    up_to_two(0);
    if (COL_BLOCKS > 2 && prm.n_cols - n0 > 32) up_to_two(32);
#endif
}

// Column blocks of a workgroup.  More of them share a row's loads; fewer spread a launch, and the long contractions of an expert with
// more than 16 rows, over more workgroups.  us with 1 / 2 / 4 blocks, 16-bit types, equal counts unless said otherwise: 2 experts of 4096
// x 1024, one row each: 9.5 / 13.0 / 19.2; 8 of 1024 x 4096, 8 rows in all: 16.9 / 14.8 / 14.2; 256 of 2048 x 1024, 512: 187 / 163 / 168;
// 8 of 4096 x 14336, 64: 178 / 152 / 137, shares 1 / rank^1.2: 179 / 157 / 146; 64 of 8192 x 2048, 512, such shares: 445 / 400 / 515.  So
// one where two would make fewer workgroups than there are compute units, and four where one expert makes half as many.
// (float32 with 4 loses on skewed counts everywhere: 8 of 2048 x 8192, 192 rows: 183 / 144 / 161.)
template <typename T> int skinny_blocks(const SkinnyParams &prm, int64_t experts) {
    const int64_t cus = device_compute_units();
    if (experts * ceil_div(prm.n_cols, 32) < cus) return 1;
    // (a workgroup's weights in one buffer resource)
    return sizeof(T) == 2 && ceil_div(prm.n_cols, 64) * 2 >= cus && (int64_t)prm.k_extent * 2 * 64 < ((int64_t)1 << 31) ? 4 : 2;
}

template <typename T> int launch(const SkinnyParams &params, int64_t rows_cap, int64_t n_expert, hipStream_t stream) {
    SkinnyParams prm = params;
    // An expert's groups of rows go to workgroups of their own, where the experts come in order of their rows: the further groups first,
    // which leave at once where there are none.  128 experts of 1280 x 1280, 448 rows, 144 of them one expert's: 37 us in turn, 29 apart; 64 of 1280 x
    // 1280 in float32, 900 and 274: 116 and 82.
    // More experts are in no order, and those with rows are found through the map of row tiles, at most as many as there are rows: 8192 experts of 64 x
    // 1024, 8 slots: 9 us on 256 workgroups, where a place for each expert makes 262144 and 71; 2048 of 512 x 512, 64 slots: 9 and 17.
    const bool apart = n_expert <= segtab::kSmallExperts;
    prm.order_off = (int32_t)(apart ? segtab::order_off(rows_cap, n_expert) : segtab::map128_off(rows_cap, n_expert));
    prm.extra_groups = apart ? (int32_t)(rows_cap / kSkRows) : 0;
    const int64_t experts = apart ? std::min(rows_cap, n_expert) : segtab::cap_tiles(rows_cap, n_expert, 128);
    const int blocks = apart ? skinny_blocks<T>(prm, experts) : 2;
    prm.tiles_n = (int)ceil_div(prm.n_cols, 16 * blocks);
    const int64_t grid = (experts + prm.extra_groups) * prm.tiles_n;
    if (grid > (int64_t)INT32_MAX) return fail(FMOE_ELIMIT, "grouped GEMM: grid of %lld workgroups", (long long)grid);
    if (!apart) grouped_gemm_skinny_kernel<T, 2, false><<<(unsigned)grid, kSkThreads, 0, stream>>>(prm);
    else if (blocks == 1) grouped_gemm_skinny_kernel<T, 1, true><<<(unsigned)grid, kSkThreads, 0, stream>>>(prm);
    else if (blocks == 2) grouped_gemm_skinny_kernel<T, 2, true><<<(unsigned)grid, kSkThreads, 0, stream>>>(prm);
    else if constexpr (sizeof(T) == 2) grouped_gemm_skinny_kernel<T, 4, true><<<(unsigned)grid, kSkThreads, 0, stream>>>(prm);
    FMOE_LAUNCH_CHECK();
    return FMOE_OK;
}

}  // namespace

int launch_skinny(const SkinnyParams &prm, int dtype, int64_t rows_cap, int64_t n_expert, hipStream_t stream) {
    FMOE_REQUIRE(dtype == FMOE_BF16 || dtype == FMOE_F16 || dtype == FMOE_F32, "grouped GEMM: dtype %d is not a 16- or 32-bit float type", dtype);
    if (dtype == FMOE_F32) return launch<float>(prm, rows_cap, n_expert, stream);
    return dtype == FMOE_BF16 ? launch<__bf16>(prm, rows_cap, n_expert, stream) : launch<_Float16>(prm, rows_cap, n_expert, stream);
}

}  // namespace gemm
}  // namespace fmoe
